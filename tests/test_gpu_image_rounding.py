"""Images at the scale of their gridding correction, which magnifies FP32
rounding by up to 5e4 in the corners, against recorded pixels of the same
images: regrouped sums of samples or another order of a transform's radices
move corner pixels by 1e-3 to 1e-2 of the images' rms while every test on the
uncorrected scale passes.  The pixels are those of one pass on an MI355X in
128-track items dealt out in turn, with transforms of 4, 16, 16 and 8, 8, 8
points a row; _own is the most that five more passes differed from it."""
import os

import numpy as np
import pytest

from obit_amd import synth

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "image_rounding.npz")
# (side, rows, planes, facets, beam): few rows, whose planes differ between two
# passes in a few cells at most, and passes of lists of up to 183 tracks
CASES = {
    "few_1024": (1024, 29, 3, 1, False),
    "few_2048": (2048, 29, 3, 1, False),
    "few_2048_beam": (2048, 29, 3, 1, True),
    "lists_1200": (1200, 3000, 1, 2, False),
    "lists_512": (512, 1000, 1, 1, False),
}


def pixels(name):
    """Sampled pixels of the case's last image."""
    from obit_amd.gridder import GPUGrid, plane_of_channel
    nx, rows, nplane, nfacet, beam = CASES[name]
    uv, _, _ = synth.workload(4, rows=rows)
    facets = synth.make_facets(nfacet, nx, 0.4 / 3600.0, 0.3 * np.pi / 180.0)
    b, e = synth.coarse_bins(256, nplane)
    with GPUGrid(uv, facets, nplane=nplane, plane_of_chan=plane_of_channel(256, b, e, cpu_parity=False), beam=beam,
                 nVisPIO=rows) as gg:
        gg.grid(uv.buffer)
        gg.flip()
        img, _ = gg.fft_image(nfacet - 1, beam, np.full(nplane, 100.0, np.float32))
    img = img.reshape(nplane, nx, nx)
    at = np.random.default_rng(nx).integers(0, img.size, 3072)
    c = 8
    corners = [img[-1][y, x] for y in (slice(0, c), slice(nx - c, nx)) for x in (slice(0, c), slice(nx - c, nx))]
    return np.concatenate([img.reshape(-1)[at]] + [x.reshape(-1) for x in corners])


@pytest.mark.parametrize("name", list(CASES))
def test_recorded_pixels(name):
    got = pixels(name)
    g = np.load(GOLDEN)
    want, rms = g[name].astype(np.float64), float(g[name + "_rms"])
    d = np.abs(got - want) / np.maximum(rms, np.abs(want))
    print(f"{name}: max |d| / max(rms, pixel) {d.max():.2e}", flush=True)
    # four times what two passes differed by, in the order of their device
    # atomics, and at least 4e-4
    assert d.max() <= 4 * float(g[name + "_own"])


@pytest.mark.parametrize("rows", [27, 351, 1000])
def test_items_of_128_tracks(rows):
    """A list of up to 128 tracks is one work item, whose sums have one order."""
    import ctypes as C
    from obit_amd import _lib
    from obit_amd.gridder import GPUGrid
    uv, _, _ = synth.workload(4, rows=rows)
    with GPUGrid(uv, synth.make_facets(1, 1024, 0.4 / 3600.0, 0.0), nVisPIO=rows) as gg:
        gg.grid(uv.buffer)
        st = (C.c_longlong * 8)()
        _lib.check(gg.lib.ObitHIPGridListStats(gg.c, 0, st))
    print(f"lists {st[1]}, entries {st[2]}, items {st[3]}, longest {st[4]}, split {st[5]}", flush=True)
    assert st[4] <= 128
    assert st[5] == 0 and st[3] == st[1]
