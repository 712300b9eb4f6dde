"""Gridding passes with few entries: work items of fewer tracks than 128 and
binning threads that take a part of the planes, against the FP64 oracle."""
import numpy as np
import pytest

from obit_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,nx,nplane,nfacet,beam", [
    (1, 512, 1, 1, False),       # one track
    (65, 256, 3, 2, False),      # planes divided one a thread, 256 channels in 3
    (351, 1000, 7, 1, False),    # planes that divide the channels unevenly
    (2000, 512, 1, 1, False),    # lists of up to about 8 items of 16 tracks
    (2000, 512, 1, 1, True),     # a beam: items of 128 tracks
    (9001, 512, 8, 1, False),    # 81,000 entries: 32 tracks
    (9001, 2048, 8, 3, False),   # 330,000: 64 tracks
])
def test_small_pass(oracle, rows, nx, nplane, nfacet, beam):
    from obit_amd.gridder import GPUGrid, plane_of_channel
    uv, _, _ = synth.workload(4, rows=rows)
    facets = synth.make_facets(nfacet, nx, 0.4 / 3600.0, 0.3 * np.pi / 180.0)
    b, e = synth.coarse_bins(256, nplane)
    poc = plane_of_channel(256, b, e, cpu_parity=False)
    with GPUGrid(uv, facets, nplane=nplane, plane_of_chan=poc, beam=beam, nVisPIO=rows) as gg:
        gg.grid(uv.buffer)
        gg.flip()
        got = [gg.to_host(i) for i in range(nfacet)]
    i = nfacet - 1
    worst = cpu = 0.0
    for p in range(nplane):
        kw = dict(bChan=int(b[p]), eChan=int(e[p]) + 1, isBeam=beam)
        ref = oracle.trim_centre(oracle.grid_fp64(uv, facets[i], **kw), facets[i])
        peak = np.abs(ref).max()
        worst = max(worst, np.abs(got[i][p] - ref).max() / peak)
        obit = oracle.trim_centre(oracle.grid_obit(uv, facets[i], **kw), facets[i])
        cpu = max(cpu, np.abs(obit - ref).max() / peak)
    print(f"max |dG|/peak {worst:.3e} (Obit's CPU gridder {cpu:.3e})", flush=True)
    # FP32 sums of up to 10^4 samples a cell: no worse than Obit's own, which
    # adds them one by one (a lost sample is 1e-4 of the peak or more)
    assert worst < max(2e-6, 1.5 * cpu)


@pytest.mark.parametrize("order", ["up", "down", "mixed"])
@pytest.mark.parametrize("nx", [64, 200, 512])
def test_channel_orders(oracle, order, nx):
    """Tracks through tiles along ascending, descending and unordered channel
    frequencies, most of them leaving the smaller grids or outside them."""
    from obit_amd.gridder import GPUGrid, plane_of_channel
    uv, _, _ = synth.workload(4, rows=700)
    if order != "up":
        f = uv.freqArr[::-1] if order == "down" else np.random.default_rng(5).permutation(uv.freqArr)
        uv.freqArr = np.ascontiguousarray(f)
    facets = synth.make_facets(2, nx, 0.4 / 3600.0, 0.3 * np.pi / 180.0)
    b, e = synth.coarse_bins(256, 3)
    poc = plane_of_channel(256, b, e, cpu_parity=False)
    with GPUGrid(uv, facets, nplane=3, plane_of_chan=poc) as gg:
        gg.grid(uv.buffer)
        gg.flip()
        got = gg.to_host(1)
    for p in range(3):
        kw = dict(bChan=int(b[p]), eChan=int(e[p]) + 1)
        ref = oracle.trim_centre(oracle.grid_fp64(uv, facets[1], **kw), facets[1])
        peak = np.abs(ref).max()
        assert peak > 0
        # FP32 sums of up to some 10^3 samples a cell (a lost one is 1e-3 of the peak)
        assert np.abs(got[p] - ref).max() < 4e-6 * peak
