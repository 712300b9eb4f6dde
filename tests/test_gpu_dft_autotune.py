"""Autotune against the choice that an untuned launch makes: a handle whose
launch an untuned one runs on k_dft_share several times faster than on any shape
that a caller can set keeps that kernel."""
import numpy as np
import pytest

from obit_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,ncomp", [(351, 3000), (2000, 1000)])
def test_few_items_stay_shared(rows, ncomp):
    from obit_amd.skymodel import SkyModelDFT
    base, _, _ = synth.workload(1, rows=rows)
    rng = np.random.default_rng(ncomp)
    uv = synth.make_uv(base.buffer[:, :5], 1, 64, 2, base.freq, synth.freq_table(base.freq, 1, 64, 1e6), rng)
    l, m = rng.uniform(-0.5, 0.5, (2, ncomp)) * synth.DG2RAD
    maj = rng.uniform(2.0, 30.0, ncomp) / 3600.0
    gp = np.stack(synth.gauss_coeffs(maj, 0.5 * maj, rng.uniform(0, 180, ncomp)), -1)
    comps = np.concatenate([synth.point_row(rng.exponential(0.01, ncomp), l, m), gp], axis=1).astype(np.float32)
    sky = synth.SkyModel(comps=comps, modType=1)
    out = {}
    for name in ("untuned", "tuned", "set"):
        with SkyModelDFT(uv, sky, op="repl") as sm:
            sm.set_vis(uv.buffer)
            if name == "tuned":
                shape = sm.autotune(sample_rows=1024, reps=3)
            if name == "set":
                sm.set_variant(32, 64, 2)
            sm.calc_resident()
            out[name] = sm.get_vis()
    # the sums of component quarters differ from k_dft_split's in some bits
    assert not np.array_equal(out["untuned"], out["set"])
    assert np.array_equal(out["tuned"], out["untuned"]) and shape == (32, 64, 2)
