"""The matrix-core kernel for spectral point models (k_dft_spec) at its
edges: component counts around a 32-component tile, rows off the 4 rows of a
workgroup, channel runs that are whole 16-channel blocks or ragged, more than
one pass of 16 blocks, coarse bins off a block's grid, channel selections,
every operation, the resident, graph and per-buffer paths; and tables that it
cannot factor, which stay on the VALU kernel.  Against the FP64 oracle within
1e-5 of the model's peak (the split DFT's bound); the resident launch on both
kernels differs bit for bit exactly where the matrix-core kernel is taken."""
import numpy as np
import pytest

from obit_amd import synth

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _uv(nif, nchan, rows):
    base, _, _ = synth.workload(1, rows=rows)
    rng = np.random.default_rng(rows)
    return synth.make_uv(base.buffer[:, :5], nif, nchan, 2, base.freq,
                         synth.freq_table(base.freq, nif, nchan, 1e6), rng)


def _sky(kind, uv, ncomp, bins=None):
    rng = np.random.default_rng(ncomp)
    l, m = rng.uniform(-0.5, 0.5, (2, ncomp)) * synth.DG2RAD
    flux = rng.exponential(0.01, ncomp) * np.where(rng.uniform(size=ncomp) < 0.2, -1.0, 1.0)
    flux[0] = 0.5
    row = synth.point_row(flux, l, m)
    if kind == "tab":
        idx = np.searchsorted(np.asarray(bins), np.arange(uv.nif * uv.nchan), side="right").astype(np.int32)
        n = int(idx.max()) + 1
        S = flux[:, None] * rng.uniform(0.5, 1.5, (ncomp, n))
        comps = np.concatenate([row, rng.normal(-0.7, 0.3, (ncomp, 1)), S], axis=1)
        sf = np.array([uv.freqArr[idx == i].mean() for i in range(n)])
        return synth.SkyModel(comps=comps.astype(np.float32), modType=20, specFreq=sf, specIndex=idx)
    nt = 1 if kind == "power" else 2
    c = [rng.normal(-0.7, 0.3, (ncomp, 1))] + ([rng.normal(0.0, 2.0, (ncomp, 1))] if nt == 2 else [])
    return synth.SkyModel(comps=np.concatenate([row] + c, axis=1).astype(np.float32), modType=10, nSpecTerm=nt,
                          imgRefFreq=float(uv.freqArr[0]))


def _run(uv, sky, op, path="resident", variant=None, **kw):
    from obit_amd.skymodel import SkyModelDFT
    with SkyModelDFT(uv, sky, op=op, **kw) as sm:
        if path == "buffer":
            return sm.calc(uv.buffer.copy())
        if variant:
            sm.set_variant(*variant)
        sm.set_vis(uv.buffer)
        for _ in range(2 if path == "graph" else 1):
            (sm.graph_launch if path == "graph" else sm.calc_resident)()
        return sm.get_vis()


# nif, nchan, rows, ncomp, kind, bins, selection, on the matrix units
CASES = [
    (4, 64, 61, 1, "power", None, {}, True),
    (4, 64, 62, 31, "power", None, {}, True),
    (1, 256, 63, 32, "power", None, {}, True),
    (1, 256, 64, 33, "tab", [64, 128, 192], {}, True),
    (4, 256, 3, 129, "power", None, {}, True),                     # four passes
    (2, 96, 65, 100, "tab", [48, 96, 144], {}, True),
    (4, 60, 61, 200, "tab", [30, 60, 90, 120, 150, 180, 210], {}, True),   # last blocks moved back
    (3, 60, 62, 96, "tab", [50], {}, True),                        # a run shorter than a block
    (4, 60, 61, 200, "tab", [37, 100, 180], {}, False),            # 18 blocks: the second pass nearly empty
    (4, 64, 62, 64, "power", None, dict(startChannel=3, numberChannel=58, startIF=2, numberIF=3), True),
    (1, 64, 61, 100, "power", None, {}, False),                    # too few channels
    (4, 64, 61, 100, "curved", None, {}, False),                   # a curvature the factors miss
]


@pytest.mark.parametrize("nif,nchan,rows,ncomp,kind,bins,sel,mm", CASES)
def test_spectral_matrix_core(oracle, nif, nchan, rows, ncomp, kind, bins, sel, mm):
    uv = _uv(nif, nchan, rows)
    sky = _sky(kind, uv, ncomp, bins)
    ref = oracle.dft_model_fp64(uv, sky, nthreads=8)
    peak = np.abs(ref).max()
    b0, nb = sel.get("startIF", 1) - 1, sel.get("numberIF", nif)
    c0, nc = sel.get("startChannel", 1) - 1, sel.get("numberChannel", nchan)
    pick = np.zeros((nif, nchan), bool)
    pick[b0:b0 + nb, c0:c0 + nc] = True
    d0 = uv.data_view()
    outs = {}
    for path, variant in (("resident", (64, 64, 2)), ("resident", (32, 64, 2)), ("graph", (64, 64, 2)),
                          ("buffer", None)):
        out = _run(uv, sky, "repl", path, variant, **sel)
        outs[path, variant] = out
        d1 = out[:, 5:].reshape(d0.shape)
        for s in range(2):
            err = np.abs((d1[..., s, 0] + 1j * d1[..., s, 1]) - ref)[:, pick].max()
            assert err <= TOL * peak, (path, variant, err / peak)
        assert np.array_equal(d1[:, ~pick], d0[:, ~pick])
        assert np.array_equal(d1[..., 2], d0[..., 2])
    valu, mat = outs["resident", (32, 64, 2)], outs["resident", (64, 64, 2)]
    assert np.array_equal(valu, mat) != mm
    assert np.array_equal(mat, outs["graph", (64, 64, 2)])
    sub = _run(uv, sky, "sub", "resident", (64, 64, 2), **sel)[:, 5:].reshape(d0.shape)
    want = (d0[..., 0, 0] + 1j * d0[..., 0, 1]) - np.where(pick, ref, 0)
    assert np.abs((sub[..., 0, 0] + 1j * sub[..., 0, 1]) - want).max() <= TOL * peak + 4e-7 * np.abs(d0[..., :2]).max()
    div = _run(uv, sky, "div", "resident", (64, 64, 2), **sel)[:, 5:].reshape(d0.shape)
    wt = d0[..., 2] * np.where(pick, np.abs(ref), 1.0)[..., None]
    assert np.abs(div[..., 2] - wt).max() <= 2 * TOL * peak + 1e-6 * np.abs(wt).max()
