"""Models that are small in some channels or correlations: those are as exact,
against their own size, as the bright ones (the matrix-core kernels' FP16 parts
hold 22 bits below their scale)."""
import numpy as np
import pytest

from obit_amd import synth
from obit_amd.beam import BeamDFT
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# of the channels' own peak: the kernels' error is 2..5e-7 of the model's norm, its
# worst value some four times that
TOL = 2e-6
LEVELS = [1e-2, 1e-4, 1e-6, 1e-9]


def _uv(rows, nif, nchan, ncorr):
    base, sky, _ = synth.workload(1, rows=rows)
    nf = nif * nchan
    buf = np.zeros((rows, 5 + nf * 3 * ncorr), np.float32)
    buf[:, :5] = base.buffer[:, :5]
    buf[:, 5:].reshape(rows, nf * ncorr, 3)[..., 2] = 1.0
    fr = (base.freq * (1.0 + 0.05 * np.arange(nif))[:, None] + 1e6 * np.arange(nchan)[None, :]).ravel()
    return synth.UVData(buffer=buf, nchan=nchan, nif=nif, nstok=ncorr, freq=base.freq, freqArr=fr,
                        crval_stokes=-5.0), sky


def _beam(uv, comps, jones, amps):
    nant, nf = 27, uv.nif * uv.nchan
    jmap = np.zeros(nf, np.int32)
    with BeamDFT(uv, comps, np.zeros(nant, np.int32), jmap, 1, stok_type=1, op="repl") as bm:
        bm.set_jones(jones)
        if amps is not None:
            bm.set_amps(amps)
        got = bm.calc(uv.buffer, par_ang=0.2)
    model, live = orc.beam_model_fp64(uv.buffer, comps, uv.freqArr / uv.freq, np.zeros(nant, int), jmap, jones, 1, 0.2,
                                      ilocb=uv.ilocb, stok_fact=(1.0,) * 4, amps=amps)
    want = orc.beam_apply(uv.buffer, model, live, uv.nrparm, uv.nif, uv.nchan, uv.incf, uv.incif, uv.nstok, "repl")
    d = np.abs(got.astype(np.float64) - want)[:, 5:].reshape(uv.nrow, nf, uv.nstok, 3)[..., :2]
    return d, np.abs(want)[:, 5:].reshape(uv.nrow, nf, uv.nstok, 3)[..., :2]


@pytest.mark.parametrize("level", LEVELS)
@pytest.mark.parametrize("shape", ["ripple", "smooth"])
def test_beam_channels(shape, level):
    uv, sky = _uv(61, 4, 64, 2)
    comps = sky.comps[:100].copy()
    x = (uv.freqArr / uv.freq) ** -0.7
    x[-32:] *= level * (1.0 + 0.3 * np.cos(1.3 * np.arange(32)) if shape == "ripple" else 1.0)
    amps = (comps[:, :1].astype(np.float64) * x[None, :]).astype(np.float32)
    jones = np.zeros((1, 100, 1, 2, 2), np.complex128)
    jones[..., 0, 0] = jones[..., 1, 1] = 1.0
    d, w = _beam(uv, comps, jones, amps)
    for c in (slice(0, 224), slice(224, 256)):
        e = d[:, c].max() / w[:, c].max()
        print(f"{shape} {level:g}, channels {c.start}..{c.stop - 1}: {e:.2e} of their peak", flush=True)
        assert e < TOL


@pytest.mark.parametrize("level", LEVELS)
@pytest.mark.parametrize("nif", [4, 1])
def test_beam_cross_hands(nif, level):
    """Leakages of the given level: the cross hands against their own peak."""
    uv, sky = _uv(61, nif, 64, 4)
    comps = sky.comps[:100].copy()
    rng = np.random.default_rng(3)
    jones = np.zeros((1, 100, 1, 2, 2), np.complex128)
    jones[..., 0, 0] = jones[..., 1, 1] = 1.0
    jones[..., 0, 1], jones[..., 1, 0] = level * (rng.normal(size=(2, 1, 100, 1)) + 1j * rng.normal(size=(2, 1, 100, 1)))
    d, w = _beam(uv, comps, jones.astype(np.complex64).astype(np.complex128), None)
    for s in ([0, 1], [2, 3]):
        e = d[:, :, s].max() / w[:, :, s].max()
        print(f"{level:g}, correlations {s}: {e:.2e} of their peak", flush=True)
        assert e < TOL


@pytest.mark.parametrize("level", LEVELS)
def test_tabulated_bin(oracle, level):
    from obit_amd.skymodel import SkyModelDFT
    uv, _ = _uv(61, 1, 256, 2)
    ncomp = 100
    rng = np.random.default_rng(4)
    l, m = rng.uniform(-0.5, 0.5, (2, ncomp)) * synth.DG2RAD
    flux = rng.exponential(0.01, ncomp)
    idx = (np.arange(256) // 64).astype(np.int32)
    S = flux[:, None] * np.array([1.0, 0.9, 0.8, level])
    comps = np.concatenate([synth.point_row(flux, l, m), rng.normal(-0.7, 0.3, (ncomp, 1)), S], axis=1)
    sky = synth.SkyModel(comps=comps.astype(np.float32), modType=20, specIndex=idx,
                         specFreq=np.array([uv.freqArr[idx == i].mean() for i in range(4)]))
    with SkyModelDFT(uv, sky, op="repl") as sm:
        sm.set_variant(64, 64, 2)
        sm.set_vis(uv.buffer)
        sm.calc_resident()
        out = sm.get_vis()[:, 5:].reshape(uv.nrow, 256, 2, 3)
    ref = oracle.dft_model_fp64(uv, sky)[:, 0]
    for c in (slice(0, 192), slice(192, 256)):
        e = np.abs(out[:, c, 0, 0] + 1j * out[:, c, 0, 1] - ref[:, c]).max() / np.abs(ref[:, c]).max()
        print(f"{level:g}, channels {c.start}..{c.stop - 1}: {e:.2e} of their peak", flush=True)
        assert e < TOL
