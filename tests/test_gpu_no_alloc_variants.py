"""ObitHIPSkyModelDFTCalcNoAlloc on handles set to any kernel shape, the
matrix-core kernel among them: every selected channel written, against the FP64
oracle."""
import ctypes as C

import numpy as np
import pytest

from obit_amd import _lib, synth

pytestmark = pytest.mark.gpu

TOL = 1e-5  # of the model's peak: the split DFT's bound


@pytest.mark.parametrize("nchan", [64, 100])
@pytest.mark.parametrize("gauss", [False, True])
@pytest.mark.parametrize("cpt", [None, 16, 32, 64])
def test_variants(oracle, cpt, gauss, nchan):
    from obit_amd.skymodel import SkyModelDFT
    lib = _lib.load()
    rows, ncomp = 300, 200
    base, _, _ = synth.workload(1, rows=rows)
    rng = np.random.default_rng(ncomp)
    uv = synth.make_uv(base.buffer[:, :5], 2, nchan, 2, base.freq, synth.freq_table(base.freq, 2, nchan, 1e6), rng)
    l, m = rng.uniform(-0.5, 0.5, (2, ncomp)) * synth.DG2RAD
    cols = [synth.point_row(rng.exponential(0.01, ncomp), l, m)]
    if gauss:
        maj = rng.uniform(2.0, 30.0, ncomp) / 3600.0
        gp = np.stack(synth.gauss_coeffs(maj, 0.5 * maj, rng.uniform(0, 180, ncomp)), -1)
        gp[::3] = 0.0
        cols.append(gp)
    sky = synth.SkyModel(comps=np.concatenate(cols, axis=1).astype(np.float32), modType=int(gauss))
    ref = oracle.dft_model_fp64(uv, sky)
    dv, dm = C.c_void_p(), C.c_void_p()
    _lib.check(lib.ObitHIPMalloc(C.byref(dv), uv.buffer.nbytes))
    _lib.check(lib.ObitHIPMalloc(C.byref(dm), sky.comps.nbytes))
    try:
        _lib.check(lib.ObitHIPMemcpyH2D(dv, _lib.ptr(uv.buffer), uv.buffer.nbytes))
        _lib.check(lib.ObitHIPMemcpyH2D(dm, _lib.ptr(sky.comps), sky.comps.nbytes))
        with SkyModelDFT(uv, sky, op="repl") as sm:
            if cpt:
                sm.set_variant(cpt, 64, 2)
            _lib.check(lib.ObitHIPSkyModelDFTCalcNoAlloc(sm.g, dm, ncomp, dv, rows), "NoAlloc")
            _lib.check(lib.ObitHIPDeviceSynchronize())
        out = np.empty_like(uv.buffer)
        _lib.check(lib.ObitHIPMemcpyD2H(_lib.ptr(out), dv, out.nbytes))
    finally:
        lib.ObitHIPFree(dv)
        lib.ObitHIPFree(dm)
    d = out[:, uv.nrparm:].reshape(uv.nrow, uv.nif, uv.nchan, uv.nstok, 3)
    for s in range(2):
        err = np.abs(d[..., s, 0] + 1j * d[..., s, 1] - ref).max()
        assert err <= TOL * np.abs(ref).max()
