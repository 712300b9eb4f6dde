"""The gridder's rounding (one conversion instruction for the CPU's lround and
its half-up columns) at and around every kind of tie: samples whose scaled u, v
or tap offset lies within a few ulps of half an integer, positive and negative,
small and beyond the grid, against the CPU gridder's own arithmetic."""
import numpy as np
import pytest

from obit_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [0.5, 0.005, 0.0])
def test_ties(oracle, half):
    """half: 0.5 for ties of the cells, 0.005 (and 0) for those of the 100 taps a
    cell."""
    from obit_amd.gridder import GPUGrid
    uv, _, _ = synth.workload(4, rows=4096)
    f = synth.make_facets(1, 1024, 0.4 / 3600.0, 0.0)
    f[0].rot = np.eye(3, dtype=np.float32).reshape(9)
    f[0].shift = np.zeros(3, np.float32)
    rng = np.random.default_rng(1)
    cell = 1024 * 0.4 / 3600.0 * np.pi / 180.0          # cells a wavelength
    n = uv.nrow
    chan = rng.integers(0, 256, n)
    fs = uv.freqArr[chan] / uv.freq
    for col in (0, 1):
        cells = np.where(rng.random(n) < 0.9, rng.integers(-500, 500, n), rng.integers(-60000, 60000, n)) + half
        taps = rng.integers(0, 100, n) * 0.01 if half < 0.5 else 0.0
        u = ((cells + taps) / (cell * fs)).astype(np.float32)
        # a few ulps to either side
        uv.buffer[:, col] = (u.view(np.int32) + rng.integers(-3, 4, n).astype(np.int32)).view(np.float32)
    uv.buffer[:, 2] = 0.0
    with GPUGrid(uv, f) as gg:
        iu, iv, itu, itv, vis = gg.prep_debug(0, uv.buffer)
    oiu, oiv, oitu, oitv, ovis = oracle.grid_prep(uv, f[0])
    ok = ovis.reshape(-1, 2).any(axis=1)
    # the samples this is about: the scaled coordinate of each row's channel
    at = np.arange(n) * 256 + chan
    print(f"{ok.sum()} valid samples, {ok[at].sum()} of them at the ties", flush=True)
    assert ok[at].sum() > 1000
    for a, b in ((iu, oiu), (iv, oiv), (itu, oitu), (itv, oitv)):
        assert np.array_equal(a[ok], b[ok])
