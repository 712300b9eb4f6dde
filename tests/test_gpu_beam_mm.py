"""The matrix-core beam DFT (k_beam_mm) at its edges, against the FP64 oracle:
component counts around a 32-component tile and a 128-component fold, row
counts off the 4 rows of a workgroup, channel runs of one beam channel that
are whole 16-channel blocks, ragged, or shorter than a block, more than one
pass of 16 blocks, 2 and 4 correlations, every operation, channel selections,
and smooth per-channel amplitudes.  Tolerance: the model within 1e-5 of its
peak (the split DFT's bound); the rest of a row bit-identical."""
import numpy as np
import pytest

from obit_amd import synth
from obit_amd.beam import BeamDFT
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

NANT = 27


def _uv(ncorr, rows, nif, nchan, seed):
    rng = np.random.default_rng(seed)
    base, _, _ = synth.workload(1, rows=rows)
    buf = np.zeros((rows, 5 + nif * nchan * 3 * ncorr), np.float32)
    buf[:, :5] = base.buffer[:, :5]
    vis = buf[:, 5:].reshape(rows, nif, nchan, ncorr, 3)
    vis[..., :2] = rng.normal(size=vis.shape[:-1] + (2,))
    vis[..., 2] = np.where(rng.uniform(size=vis.shape[:-1]) < 0.08, -1.0, 1.0)
    vis[rng.uniform(size=(rows, nif, nchan)) < 0.02, :, 2] = 0.0
    buf[1::37, 3] = 256 * 3 + 31                         # an antenna outside the table
    fr = (base.freq * (1.0 + 0.05 * np.arange(nif))[:, None] + 1e6 * np.arange(nchan)[None, :]).ravel()
    return synth.UVData(buffer=buf, nchan=nchan, nif=nif, nstok=ncorr, freq=base.freq, freqArr=fr, crval_stokes=-5.0)


# ncorr, rows, nif, nchan, beam-channel run, ncomp, types, op, spectral index, selection
CASES = [
    (2, 61, 4, 64, 32, 1, 1, "sub", None, None),
    (2, 62, 4, 64, 64, 31, 2, "repl", None, None),
    (4, 63, 2, 64, 16, 32, 2, "sub", None, None),
    (4, 64, 1, 100, 100, 33, 1, "div", None, None),
    (2, 3, 5, 64, 37, 128, 1, "sub", None, None),       # ragged runs, two passes
    (4, 1, 3, 100, 50, 129, 3, "repl", None, None),
    (2, 65, 2, 96, 11, 200, 1, "sub", None, None),      # runs shorter than a block
    (2, 61, 4, 64, 32, 300, 1, "sub", -0.7, None),
    (4, 62, 2, 128, 128, 161, 2, "repl", 1.3, None),
    (2, 63, 1, 256, 100, 96, 1, "div", -0.7, None),
    (2, 64, 4, 64, 64, 64, 1, "sub", None, ((5, 60), (1, 3))),
    (4, 61, 4, 64, 32, 64, 1, "sub", -0.7, ((0, 55), (0, 2))),
    (2, 61, 1, 64, 32, 100, 2, "sub", None, None),      # 8 blocks or fewer: a correlation a half-wave
    (4, 66, 1, 128, 64, 95, 1, "repl", -0.7, None),
    (2, 61, 1, 128, 128, 70, 1, "div", None, None),
]


@pytest.mark.parametrize("ncorr,rows,nif,nchan,run,ncomp,ntype,op,alpha,sel", CASES)
def test_beam_matrix_core(ncorr, rows, nif, nchan, run, ncomp, ntype, op, alpha, sel):
    uv = _uv(ncorr, rows, nif, nchan, seed=ncomp)
    rng = np.random.default_rng(ncomp + 1)
    _, sky, _ = synth.workload(1, rows=8)
    comps = sky.comps[:ncomp].copy()
    comps[0, 0] = 1.0
    nf = nif * nchan
    jmap = (np.arange(nf) // nchan) * -(-nchan // run) + (np.arange(nf) % nchan) // run
    njchan = int(jmap.max()) + 1
    jones = np.zeros((ntype, ncomp, njchan, 2, 2), np.complex128)
    jones[..., 0, 0] = jones[..., 1, 1] = 1.0
    jones += 0.15 * (rng.normal(size=jones.shape) + 1j * rng.normal(size=jones.shape))
    jones = jones.astype(np.complex64).astype(np.complex128)
    ant_type = rng.integers(0, ntype, NANT)
    sf, chi, stok = (1.0, 0.9, 0.8, 1.1), 0.41, 1 + ncomp % 4
    if op == "div":
        stok = 1                                        # a model that is not zero where its leakage is
    kw = {} if sel is None else dict(chan_sel=sel[0], if_sel=sel[1])
    amps = None
    if alpha is not None:
        amps = (comps[:, :1].astype(np.float64) *
                (uv.freqArr / uv.freq)[None, :] ** (alpha + 0.2 * rng.normal(size=(ncomp, 1)))).astype(np.float32)
    with BeamDFT(uv, comps, ant_type, jmap, njchan, ntype=ntype, stok_type=stok, op=op, stok_fact=sf, **kw) as bm:
        bm.set_jones(jones)
        if amps is not None:
            bm.set_amps(amps)
        got = bm.calc(uv.buffer, par_ang=chi)
    model, live = orc.beam_model_fp64(uv.buffer, comps, uv.freqArr / uv.freq, ant_type, jmap, jones, stok, chi,
                                      ilocb=uv.ilocb, stok_fact=sf, amps=amps)
    a = (uv.buffer, model, live, uv.nrparm, nif, nchan, uv.incf, uv.incif, ncorr, op)
    want = orc.beam_apply(*a, **kw)
    moved = np.isnan(orc.beam_apply(a[0], np.full_like(model, complex(np.nan, np.nan)), *a[2:], **kw))
    assert moved.any() and np.array_equal(got[~moved], uv.buffer[~moved])
    err = np.abs(got[moved].astype(np.float64) - want[moved]).max()
    scale = 2.0 * np.abs(want[moved]).max() if op == "div" else np.abs(model[live]).max()
    assert err < 1e-5 * scale, (err, scale)
