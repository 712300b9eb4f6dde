"""The resident launches of few items (k_dft_share: four waves share 64 rows
and add their sums) at its edges: rows around 64, component counts that leave
waves without components or with part of a tile, channel counts off a chunk,
all model types without a matrix-core route, every operation, and the graph
and no-allocation calls.  Against the FP64 oracle within 1e-5 of the peak (the
split DFT's bound), and graph replays bit-equal to the launch."""
import numpy as np
import pytest

from obit_amd import synth

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _case(kind, nif, nchan, rows, ncomp):
    base, _, _ = synth.workload(1, rows=rows)
    rng = np.random.default_rng(ncomp)
    uv = synth.make_uv(base.buffer[:, :5], nif, nchan, 2, base.freq, synth.freq_table(base.freq, nif, nchan, 1e6), rng)
    l, m = rng.uniform(-0.5, 0.5, (2, ncomp)) * synth.DG2RAD
    flux = rng.exponential(0.01, ncomp)
    flux[0] = 0.5
    cols = [synth.point_row(flux, l, m)]
    if "gauss" in kind:
        maj = rng.uniform(2.0, 30.0, ncomp) / 3600.0
        gp = np.stack(synth.gauss_coeffs(maj, maj * rng.uniform(0.3, 1.0, ncomp), rng.uniform(0, 180, ncomp)), -1)
        gp[rng.uniform(size=ncomp) < (1.0 if kind == "gauss0" else 0.6)] = 0.0
        cols.append(gp)
    kw = {}
    if "spec" in kind:
        cols.append(rng.normal(-0.7, 0.3, (ncomp, 1)))
        kw = dict(nSpecTerm=1, imgRefFreq=float(uv.freqArr[0]))
    code = {"gauss": 1, "gauss0": 1, "spec": 10, "gaussspec": 11}[kind]
    return uv, synth.SkyModel(comps=np.concatenate(cols, axis=1).astype(np.float32), modType=code, **kw)


CASES = [
    ("gauss", 1, 64, 1, 1), ("gauss", 1, 64, 63, 2), ("gauss", 1, 37, 64, 3), ("gauss", 2, 33, 65, 5),
    ("gauss0", 1, 64, 130, 255), ("gauss", 1, 64, 351, 257), ("gauss", 1, 100, 351, 1000),
    ("spec", 1, 64, 65, 4), ("spec", 1, 48, 351, 300), ("gaussspec", 1, 64, 64, 63), ("gaussspec", 2, 17, 200, 515),
]


@pytest.mark.parametrize("kind,nif,nchan,rows,ncomp", CASES)
def test_shared_rows(oracle, kind, nif, nchan, rows, ncomp):
    from obit_amd.skymodel import SkyModelDFT
    uv, sky = _case(kind, nif, nchan, rows, ncomp)
    ref = oracle.dft_model_fp64(uv, sky, nthreads=8)
    peak = np.abs(ref).max()
    d0 = uv.data_view()

    def run(op, path):
        with SkyModelDFT(uv, sky, op=op) as sm:
            sm.set_vis(uv.buffer)
            (sm.graph_launch if path == "graph" else sm.calc_resident)()
            return sm.get_vis()
    out = run("repl", "resident")
    assert np.array_equal(run("repl", "graph"), out)
    d1 = out[:, 5:].reshape(d0.shape)
    for s in range(2):
        assert np.abs((d1[..., s, 0] + 1j * d1[..., s, 1]) - ref).max() <= TOL * peak
    assert np.array_equal(d1[..., 2], d0[..., 2]) and np.array_equal(out[:, :5], uv.buffer[:, :5])
    sub = run("sub", "resident")[:, 5:].reshape(d0.shape)
    got = (d0[..., 0, 0] + 1j * d0[..., 0, 1]) - (sub[..., 0, 0] + 1j * sub[..., 0, 1])
    assert np.abs(got - ref).max() <= TOL * peak + 4e-7 * np.abs(d0[..., :2]).max()
    div = run("div", "resident")[:, 5:].reshape(d0.shape)
    assert np.abs(div[..., 2] - d0[..., 2] * np.abs(ref)[..., None]).max() <= 2 * TOL * peak


@pytest.mark.parametrize("kind,nif,nchan,rows,ncomp", [
    ("point", 1, 64, 1, 1), ("point", 1, 64, 351, 100), ("point", 1, 37, 65, 255), ("point", 2, 16, 700, 257),
    ("gauss0", 1, 64, 351, 100), ("gauss", 2, 33, 64, 63), ("gaussspec", 1, 48, 129, 5),
])
def test_shared_rows_buffer(oracle, kind, nif, nchan, rows, ncomp):
    """Host buffers of less than a round of workgroups, every operation."""
    from obit_amd.skymodel import SkyModelDFT
    uv, sky = _case("gauss0" if kind == "point" else kind, nif, nchan, rows, ncomp)
    if kind == "point":
        sky = synth.SkyModel(comps=np.ascontiguousarray(sky.comps[:, :4]), modType=0)
    ref = oracle.dft_model_fp64(uv, sky, nthreads=8)
    peak = np.abs(ref).max()
    d0 = uv.data_view()
    out = {}
    for op in ("repl", "sub"):
        with SkyModelDFT(uv, sky, op=op) as sm:
            out[op] = sm.calc(uv.buffer.copy())[:, 5:].reshape(d0.shape)
    for st in range(2):
        got = out["repl"][..., st, 0] + 1j * out["repl"][..., st, 1]
        assert np.abs(got - ref).max() <= TOL * peak
        left = d0[..., st, 0] + 1j * d0[..., st, 1] - (out["sub"][..., st, 0] + 1j * out["sub"][..., st, 1])
        assert np.abs(left - ref).max() <= TOL * peak + 4e-7 * np.abs(d0[..., :2]).max()
    assert np.array_equal(out["sub"][..., 2], d0[..., 2])
