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


@pytest.mark.parametrize("nx", [1024, 2048])
@pytest.mark.parametrize("scale", [0.0, 1e-3, 1.0])
def test_image_of_few_columns(oracle, nx, scale):
    """Transforms of planes whose column blocks are almost all empty (one row at
    the origin or near it, or three somewhere), and of a plane without channels."""
    import ctypes as C
    from obit_amd import _lib
    from obit_amd.gridder import GPUGrid
    uv, _, _ = synth.workload(4, rows=3 if scale == 1.0 else 1)
    uv.buffer[:, :3] *= np.float32(scale)
    f = synth.make_facets(1, nx, 0.4 / 3600.0, 0.0)
    cf = oracle.convfunc()[0]
    corr = np.zeros(nx, np.float32)
    _lib.load().ObitHostGridCorrFn(nx, nx // 2 + 1, cf.ctypes.data_as(C.POINTER(C.c_float)), 7, 100,
                                   corr.ctypes.data_as(C.POINTER(C.c_float)))
    poc = np.zeros(256, np.int32)
    poc[1::2] = 2  # the even channels in plane 0, none in 1, the odd ones in 2
    norm = np.ones(3, np.float32)
    with GPUGrid(uv, f, nplane=3, plane_of_chan=poc) as gg:
        gg.grid(uv.buffer)
        gg.flip()
        planes = gg.to_host(0)
        img, _ = gg.fft_image(0, False, norm)
    assert np.abs(planes[0]).max() > 0 and not planes[1].any() and not img[1].any()
    ref, _ = oracle.fft2image(planes, cf, False, norm, corr=(corr, corr))
    taper = (corr[:, None] * corr[None, :]).astype(np.float64)
    for p in (0, 2):
        peak = np.abs(ref[p] / taper).max()
        # FP32 transform of 2^22 points: 22 butterflies of 6e-8, on the uncorrected scale
        assert np.abs((img[p] - ref[p]) / taper).max() < 1e-6 * peak


@pytest.mark.parametrize("nx,nplane", [(128, 32), (128, 33), (1024, 32), (1024, 33)])
def test_image_norms(oracle, nx, nplane):
    """Images of as many planes as take their norms in the kernel's arguments,
    and of one more, each plane by its own norm."""
    import ctypes as C
    from obit_amd import _lib
    from obit_amd.gridder import GPUGrid
    uv, _, _ = synth.workload(4, rows=5)
    f = synth.make_facets(1, nx, 0.4 / 3600.0 * 1024 / nx, 0.0)
    cf = oracle.convfunc()[0]
    corr = np.zeros(nx, np.float32)
    _lib.load().ObitHostGridCorrFn(nx, nx // 2 + 1, cf.ctypes.data_as(C.POINTER(C.c_float)), 7, 100,
                                   corr.ctypes.data_as(C.POINTER(C.c_float)))
    norm = np.linspace(0.5, 9.0, nplane).astype(np.float32)
    with GPUGrid(uv, f, nplane=nplane, plane_of_chan=(np.arange(256) % nplane).astype(np.int32)) as gg:
        gg.grid(uv.buffer)
        gg.flip()
        planes = gg.to_host(0)
        img, _ = gg.fft_image(0, False, norm)
    look = [0, 1, nplane - 1]
    ref, _ = oracle.fft2image(planes[look], cf, False, norm[look], corr=(corr, corr))
    taper = (corr[:, None] * corr[None, :]).astype(np.float64)
    for k, p in enumerate(look):
        assert np.abs((img[p] - ref[k]) / taper).max() < 1e-6 * np.abs(ref[k] / taper).max()
