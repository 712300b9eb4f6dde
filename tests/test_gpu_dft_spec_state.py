"""The spectral matrix-core kernel (k_dft_spec) after what its tables were made
from has changed: frequencies uploaded again, other reference frequencies under
a captured graph, the sin/cos policy.  Each against a handle made for the new
state, bit for bit, and against the FP64 oracle."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from obit_amd import synth

pytestmark = pytest.mark.gpu

TOL = 1e-5  # of the model's peak: the split DFT's bound


class _Head(C.Structure):
    """The first fields of a GPUInfo."""
    _fields_ = [("ints", C.c_int * 10), ("nmodel", C.c_int * 4), ("d_model", C.c_void_p * 4), ("d_freq", C.c_void_p)]


def _uv(nif, nchan, rows, step=1e6, scale=1.0):
    base, _, _ = synth.workload(1, rows=rows)
    uv = synth.make_uv(base.buffer[:, :5], nif, nchan, 2, base.freq,
                       synth.freq_table(base.freq, nif, nchan, step), np.random.default_rng(rows))
    return dataclasses.replace(uv, freqArr=uv.freqArr * scale)


def _sky(uv, ncomp, ref):
    rng = np.random.default_rng(ncomp)
    l, m = rng.uniform(-0.5, 0.5, (2, ncomp)) * synth.DG2RAD
    flux = rng.exponential(0.01, ncomp)
    flux[0] = 0.5
    c = np.concatenate([synth.point_row(flux, l, m), rng.normal(-0.7, 0.3, (ncomp, 1))], axis=1)
    return synth.SkyModel(comps=c.astype(np.float32), modType=10, nSpecTerm=1, imgRefFreq=float(ref))


def _model(uv, rows):
    d = rows[:, uv.nrparm:].reshape(uv.nrow, uv.nif, uv.nchan, uv.nstok, 3)
    return d[..., 0, 0] + 1j * d[..., 0, 1]


@pytest.mark.parametrize("path", ["resident", "buffer"])
@pytest.mark.parametrize("step,scale", [(1e6, 1.01), (1.3e6, 1.0), (1e6, 0.9)])
def test_frequencies_uploaded_again(oracle, path, step, scale):
    from obit_amd import _lib
    from obit_amd.skymodel import SkyModelDFT
    rows = 100
    a, b = _uv(1, 256, rows), _uv(1, 256, rows, step, scale)
    sky = _sky(a, 200, a.freq)

    def apply(sm):
        if path == "buffer":
            return sm.calc(a.buffer.copy())
        sm.set_vis(a.buffer)
        sm.set_variant(64, 64, 2)
        sm.calc_resident()
        return sm.get_vis()

    with SkyModelDFT(a, sky, op="repl", useFreq64=False) as sm:
        first = apply(sm)
        fs = np.ascontiguousarray(b.fscale, dtype=np.float32)
        h = C.cast(sm.g, C.POINTER(_Head)).contents
        _lib.load().ObitCUDAUtilHost2GPU(h.d_freq, _lib.ptr(fs), fs.nbytes, None)
        got = apply(sm)
    with SkyModelDFT(b, sky, op="repl", useFreq64=False) as sm:
        want = apply(sm)
    c = np.arange(256.0)
    fit = np.polyval(np.polyfit(c, b.fscale.astype(np.float64), 1), c)
    ref = oracle.dft_model_fp64(b, sky, freq_ratio=fit)
    peak = np.abs(ref).max()
    e = [np.abs(_model(b, x) - ref).max() / peak for x in (first, got, want)]
    print(f"of the peak: first table {e[0]:.2e}, uploaded again {e[1]:.2e}, a new handle {e[2]:.2e}", flush=True)
    assert e[0] > 1e-3 and e[2] <= TOL
    assert e[1] <= TOL and np.array_equal(got, want)


@pytest.mark.parametrize("between", [True, False])
@pytest.mark.parametrize("factor", [4.0, 0.1])
def test_graph_after_new_reference(oracle, factor, between):
    """A launch captured before the reference frequency changed is captured
    again, whether or not another launch has made the table in between."""
    from obit_amd import _lib
    from obit_amd.skymodel import SkyModelDFT
    uv = _uv(4, 64, 61)
    sky = _sky(uv, 100, uv.freq)
    new = dataclasses.replace(sky, imgRefFreq=sky.imgRefFreq * factor)
    with SkyModelDFT(uv, new, op="repl") as sm:
        sm.set_variant(64, 64, 2)
        sm.set_vis(uv.buffer)
        sm.calc_resident()
        want = sm.get_vis()
    with SkyModelDFT(uv, sky, op="repl") as sm:
        sm.set_variant(64, 64, 2)
        sm.set_vis(uv.buffer)
        for _ in range(2):
            sm.graph_launch()
        sm.get_vis()
        f = np.array([new.imgRefFreq])
        _lib.check(sm.lib.ObitHIPSkyModelDFTSetSpecRef(sm.g, f.ctypes.data_as(C.POINTER(C.c_double)), 1))
        if between:
            sm.calc_resident()
        for _ in range(2):
            sm.graph_launch()
            assert np.array_equal(sm.get_vis(), want)
    ref = oracle.dft_model_fp64(uv, new)
    assert np.abs(_model(uv, want) - ref).max() <= TOL * np.abs(ref).max()


@pytest.mark.parametrize("path", ["resident", "buffer"])
def test_precision_policies(oracle, path):
    """Hardware sin/cos for the centre phasors and the steps (0), for the centre
    phasors (1), for neither (2): each result its own."""
    from obit_amd.skymodel import SkyModelDFT
    uv = _uv(4, 64, 61)
    sky = _sky(uv, 100, uv.freq)
    ref = oracle.dft_model_fp64(uv, sky)
    out = []
    for prec in (0, 1, 2):
        with SkyModelDFT(uv, sky, op="repl") as sm:
            sm.set_precision(prec)
            if path == "buffer":
                out.append(sm.calc(uv.buffer.copy()))
            else:
                sm.set_variant(64, 64, 2)
                sm.set_vis(uv.buffer)
                sm.calc_resident()
                out.append(sm.get_vis())
        assert np.abs(_model(uv, out[-1]) - ref).max() <= TOL * np.abs(ref).max()
    assert not np.array_equal(out[1], out[2]) and not np.array_equal(out[0], out[1])
