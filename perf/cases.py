"""Performance cases: what users of this library have it do, with seeded inputs.

Four kinds of call, each through the package's own drivers:

  dft     a CLEAN-component model applied to visibilities (SkyModelDFT): host
          buffers in pieces of nVisPIO rows ("buffer", Obit's SubUV loop) or
          rows resident in device memory ("resident", one call per major cycle)
  beam    the same with antenna Jones matrices per component (BeamDFT)
  grid    visibilities to images: clear the facet grids, grid, flip, transform
          (GPUGrid); or to the gridded planes in host memory
  stokes  Stokes I records of a resident data set (stokes_i_device)

Row layouts, arrays, source counts and image sizes are those of the synthetic
workloads (obit_amd/synth.py), and odd sizes around them.
"""
import ctypes
import math

import numpy as np
import torch

from obit_amd import _lib, synth
from obit_amd.beam import BeamDFT, tspec_amps
from obit_amd.gridder import GPUGrid, plane_of_channel
from obit_amd.skymodel import SkyModelDFT
from obit_amd.stokes import stokes_i_device

TWOPI = 2.0 * math.pi
DEG = math.pi / 180.0
NSPEC = 4            # subbands of a tabulated spectrum
PAR_ANG = 0.3        # parallactic angle (rad)
STOK_FACT = (1.0, 0.95, 0.9, 1.05)
BEAM_N = 65          # side of a beam image (pixels)
BEAM_CELL = 0.05     # its cell (deg)
REF_SIZE = 25.0 * 1.1 * DEG / 299792458.0   # antenna size x fudge x deg->rad / c


def listed():
    return [
        # one integration of a 27-antenna array in a host buffer, a short
        # component list: an interactive call, where latency counts
        dict(name="buffer_one_integration", kind="dft", path="buffer", model="point", op="sub", nant=27,
             rows=351, nif=1, nchan=64, nstok=2, ncomp=100, piece=10000),
        # two of Obit's 10,000-row uv buffers and a ragged rest, subtracted
        # while the caller reads and writes the data on the host
        dict(name="buffer_points", kind="dft", path="buffer", model="point", op="sub", nant=64,
             rows=22345, nif=4, nchan=64, nstok=2, ncomp=4000, piece=10000),
        # the subtract of a CLEAN major cycle on resident data: many points
        dict(name="resident_points", kind="dft", path="resident", model="point", op="sub", nant=64,
             rows=60000, nif=4, nchan=64, nstok=2, ncomp=10000, piece=1024),
        # the same with extended components among the points, one IF
        dict(name="resident_gauss", kind="dft", path="resident", model="gauss", op="sub", nant=27,
             rows=70201, nif=1, nchan=64, nstok=2, ncomp=6000, piece=1024),
        # wideband data and components with a spectral index (calibration:
        # the model replaces the data)
        dict(name="resident_spectra", kind="dft", path="resident", model="pspec", op="repl", nant=64,
             rows=12101, nif=4, nchan=256, nstok=2, ncomp=3001, piece=1024),
        # the data divided by a model with a tabulated spectrum, odd channels
        dict(name="resident_tabulated", kind="dft", path="resident", model="tspec", op="div", nant=27,
             rows=20011, nif=2, nchan=96, nstok=4, ncomp=1000, piece=1024),
        # beam-corrected subtract, parallel hands, Jones matrices handed in
        dict(name="beam_parallel_hands", kind="beam", model="point", op="sub", nant=64, rows=20160, nif=4,
             nchan=64, ncorr=2, ncomp=2000, ntype=1, njchan=8, stokes=1, images=False),
        # full polarisation, two antenna types, tabulated spectra, the Jones
        # matrices formed from beam images at each parallactic angle
        dict(name="beam_full_polarisation", kind="beam", model="tspec", op="sub", nant=27, rows=7020, nif=2,
             nchan=64, ncorr=4, ncomp=700, ntype=2, njchan=4, stokes=2, images=True),
        # a small field gridded from host buffers, the planes read back
        dict(name="grid_host_planes", kind="grid", path="host", out="planes", nant=27, rows=10530, nchan=64,
             nfacet=1, nplane=1, nx=512, beam=False),
        # dirty beam of an odd-sized field
        dict(name="grid_beam_odd_size", kind="grid", path="device", out="image", nant=27, rows=35100, nchan=96,
             nfacet=2, nplane=3, nx=1200, beam=True),
        # the regrid and transform of a wideband many-facet major cycle
        dict(name="grid_facets", kind="grid", path="device", out="image", nant=27, rows=105300, nchan=256,
             nfacet=20, nplane=8, nx=2048, beam=False),
        # the records the gridder reads, formed from a resident data set
        dict(name="stokes_records", kind="stokes", nant=64, rows=302400, nif=4, nchan=64, nstok=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dft", "dft", "dft", "beam", "grid", "stokes"])
    nant = rng.choice([27, 64])
    if kind == "stokes":
        return dict(kind=kind, nant=nant, rows=_log(rng, 351, 150000), nif=rng.choice([1, 2, 4]),
                    nchan=rng.choice([37, 64, 96, 128]), nstok=rng.choice([1, 2, 4]))
    if kind == "grid":
        dev = rng.random() < 0.6
        nx = rng.choice([512, 640, 1000, 1024, 1200, 2048])
        nplane = rng.choice([1, 2, 3, 8])
        nchan = rng.choice([48, 64, 96, 128, 256])
        nfacet = rng.randint(1, 6) if nx < 2048 else rng.randint(1, 3)
        return dict(kind=kind, path="device" if dev else "host",
                    out=rng.choice(["image", "image", "planes"]) if dev else "planes", nant=nant,
                    rows=_log(rng, 500, 60000 if dev else 20000), nchan=nchan, nfacet=nfacet if dev else 1,
                    nplane=nplane if dev else min(nplane, 2), nx=nx, beam=rng.random() < 0.3)
    if kind == "beam":
        nif, nchan = rng.choice([(1, 64), (2, 40), (2, 64), (4, 64), (1, 128)])
        ncorr = rng.choice([2, 4])
        ncomp = _log(rng, 20, 2000)
        most = 1.0e10 if ncorr == 2 else 3.0e9
        rows = _log(rng, 351, max(352, min(40000, int(most / (nif * nchan * ncomp)))))
        return dict(kind=kind, model=rng.choice(["point", "gauss", "tspec"]),
                    op=rng.choice(["sub", "sub", "repl", "div"]), nant=nant, rows=rows, nif=nif, nchan=nchan,
                    ncorr=ncorr, ncomp=ncomp, ntype=rng.choice([1, 1, 2, 3]), njchan=rng.choice([1, 2, 4, 8]),
                    stokes=rng.choice([1, 1, 2, 3, 4]), images=rng.random() < 0.4)
    path = rng.choice(["buffer", "resident", "resident"])
    nif, nchan = rng.choice([(1, 64), (2, 64), (4, 64), (1, 256), (4, 256), (1, 100), (2, 96), (3, 37), (4, 48)])
    ncomp = _log(rng, 10, 10000)
    most = 2.0e10 if path == "resident" else 5.0e9
    cap = 80000 if path == "resident" else 25000
    rows = _log(rng, 100, max(101, min(cap, int(most / (nif * nchan * ncomp)), int(1.2e8 / (6 * nif * nchan)))))
    return dict(kind="dft", path=path, model=rng.choice(["point", "point", "gauss", "pspec", "tspec", "gspec"]),
                op=rng.choice(["sub", "sub", "repl", "div"]), nant=nant, rows=rows, nif=nif, nchan=nchan,
                nstok=rng.choice([1, 2, 2, 4]), ncomp=ncomp, piece=10000 if path == "buffer" else 1024)


# ------------------------------------------------------------------ inputs

def _hdr(case, rng, f0):
    """uvw tracks, baselines and times of the first rows of an observation."""
    if case["nant"] == 27:
        enu, dt = synth.y_array(rng), 10.0
    else:
        enu, dt = synth.core_arm_array(rng), 8.0
    nb = len(enu) * (len(enu) - 1) // 2
    nt = -(-case["rows"] // nb)
    # a few integrations are spread over the observation, many follow it
    return synth.uvw_tracks(enu, 34.08, 30.0, nt, max(dt, 1200.0 / nt), f0)[:case["rows"]].astype(np.float32)


def _uv(case, seed):
    """(UVData over a virtual buffer, device rows): random parameters, N(0,1)
    correlations and weights, a few of them flagged."""
    rng = np.random.default_rng([seed, 1])
    nif, nchan = case.get("nif", 1), case["nchan"]
    nstok = case.get("nstok", case.get("ncorr", 1))
    f0 = 1.4e9 if case["nant"] == 27 else 1.28e9
    hdr = _hdr(case, rng, f0)
    ncor = nif * nchan * nstok
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    rows = torch.empty((case["rows"], 5 + 3 * ncor), dtype=torch.float32, device="cuda")
    rows[:, :5] = torch.from_numpy(hdr).cuda()
    vis = rows[:, 5:].view(case["rows"], ncor, 3)
    vis.copy_(torch.randn((case["rows"], ncor, 3), device="cuda", generator=g))
    wt = 0.5 + 1.5 * torch.rand((case["rows"], ncor), device="cuda", generator=g)
    vis[:, :, 2] = torch.where(torch.rand((case["rows"], ncor), device="cuda", generator=g) < 0.02, -wt, wt)
    buf = np.broadcast_to(np.float32(0.0), tuple(rows.shape))
    first = 1.0 if nstok == 1 else (-5.0 if "ncorr" in case else -1.0)
    uv = synth.UVData(buffer=buf, nchan=nchan, nif=nif, nstok=nstok, freq=f0,
                      freqArr=synth.freq_table(f0, nif, nchan, 1e6), crval_stokes=first)
    return uv, rows


def _sky(case, uv, seed):
    """Component table of one field: positions within half a degree, fluxes
    in Jy, a fifth of an extended model's components Gaussians of 2..30"."""
    rng = np.random.default_rng([seed, 2])
    n, model = case["ncomp"], case["model"]
    l, m = rng.uniform(-0.5, 0.5, (2, n)) * DEG
    flux = synth.powerlaw_fluxes(rng, n, smin=1e-4)
    flux[0] = 2.0 + 0.5 * np.sqrt(n)          # the calibrator or the field's bright source
    rows = [synth.point_row(flux, l, m)]
    if model in ("gauss", "gspec"):
        maj = rng.uniform(2.0, 30.0, n) / 3600.0
        gp = np.stack(synth.gauss_coeffs(maj, maj * rng.uniform(0.3, 1.0, n), rng.uniform(0, 180.0, n)), axis=-1)
        gp[rng.uniform(size=n) >= 0.2] = 0.0
        gp[0] = 0.0
        rows.append(gp)
    if model in ("pspec", "gspec"):
        rows.append(rng.normal(-0.7, 0.3, (n, 1)))
    if model == "tspec":
        rows += [rng.normal(-0.7, 0.3, (n, 1)), flux[:, None] * rng.uniform(0.8, 1.2, (n, NSPEC))]
    comps = np.concatenate(rows, axis=1).astype(np.float32)
    kw = {}
    if model in ("pspec", "gspec"):
        kw = dict(nSpecTerm=1, imgRefFreq=uv.freq)
    if model == "tspec":
        b, e = synth.coarse_bins(uv.nif * uv.nchan, NSPEC)
        idx = np.zeros(uv.nif * uv.nchan, np.int32)
        for i in range(NSPEC):
            idx[b[i]:e[i] + 1] = i
        kw = dict(specFreq=np.array([uv.freqArr[(b[i] + e[i]) // 2] for i in range(NSPEC)]), specIndex=idx)
    code = dict(point=0, gauss=1, pspec=10, gspec=11, tspec=20)[model]
    return synth.SkyModel(comps=comps, modType=code, **kw)


def _spectrum(sky, case, uv):
    """Amplitude of every component in every channel, FP64 [ncomp, nif*nchan]."""
    c, model = sky.comps.astype(np.float64), case["model"]
    nf = uv.nif * uv.nchan
    if model in ("point", "gauss"):
        return np.repeat(c[:, :1], nf, axis=1)
    if model in ("pspec", "gspec"):
        alpha = c[:, 4] if model == "pspec" else c[:, 7]
        return c[:, :1] * np.exp(alpha[:, None] * np.log(uv.freqArr / sky.imgRefFreq)[None, :])
    s = sky.specIndex
    return c[:, 5:][:, s] * np.exp(c[:, 4:5] * np.log(uv.freqArr / sky.specFreq[s])[None, :])


def _beam_tables(case, uv, seed):
    rng = np.random.default_rng([seed, 3])
    n, nf = case["ncomp"], uv.nif * uv.nchan
    t = dict(ant_type=rng.permutation(np.arange(case["nant"]) % case["ntype"]).astype(np.int32),
             jmap=((np.arange(nf) * case["njchan"]) // nf).astype(np.int32))
    l, m = rng.uniform(-0.5, 0.5, (2, n)) * DEG
    flux = synth.powerlaw_fluxes(rng, n, smin=1e-4)
    flux[0] = 2.0 + 0.5 * np.sqrt(n)
    comps = [synth.point_row(flux, l, m)]
    if case["model"] == "gauss":
        maj = rng.uniform(2.0, 30.0, n) / 3600.0
        gp = np.stack(synth.gauss_coeffs(maj, maj * rng.uniform(0.3, 1.0, n), rng.uniform(0, 180.0, n)), axis=-1)
        gp[rng.uniform(size=n) >= 0.2] = 0.0
        comps.append(gp)
    t["comps"] = np.concatenate(comps, axis=1).astype(np.float32)
    t["amps"] = None
    if case["model"] == "tspec":
        b, e = synth.coarse_bins(nf, NSPEC)
        idx = np.minimum(np.arange(nf) // (nf // NSPEC), NSPEC - 1)
        sf = np.array([uv.freqArr[(b[i] + e[i]) // 2] for i in range(NSPEC)])
        t["amps"] = tspec_amps(flux[:, None] * rng.uniform(0.8, 1.2, (n, NSPEC)),
                               np.repeat(rng.normal(-0.7, 0.3, (n, 1)), NSPEC, axis=1), idx,
                               uv.freqArr / uv.freq, uv.freq / sf)
    if case["images"]:
        # eight planes a type: voltage patterns falling off the centre,
        # leakages at the per cent level
        x = (np.arange(BEAM_N) - BEAM_N // 2) * BEAM_CELL
        r2 = x[None, :] ** 2 + x[:, None] ** 2
        img = np.zeros((case["ntype"], 8, case["njchan"], BEAM_N, BEAM_N), np.float32)
        for a in range(case["ntype"]):
            for j in range(case["njchan"]):
                w = 0.55 * (1.0 + 0.05 * rng.uniform(-1, 1)) * (1.0 + 0.02 * j)
                g = np.exp(-r2 / (2 * w * w))
                img[a, 0, j], img[a, 2, j] = g, g * (1.0 + 0.03 * rng.uniform(-1, 1))
                img[a, 1, j] = 0.05 * g * x[None, :]
                img[a, 3, j] = 0.05 * g * x[:, None]
                for k in range(4, 8):
                    img[a, k, j] = 0.03 * rng.uniform(-1, 1) * g * x[None, :] * x[:, None]
        t["img"] = img
        t["pos"] = np.stack([l / DEG, m / DEG], axis=-1).astype(np.float32)
        t["bfreq"] = np.linspace(uv.freqArr[0], uv.freqArr[-1], case["njchan"]).astype(np.float32)
    else:
        j = np.zeros((case["ntype"], n, case["njchan"], 2, 2), np.complex64)
        j[..., 0, 0] = j[..., 1, 1] = 1.0
        t["jones"] = j + (0.1 * (rng.normal(size=j.shape) + 1j * rng.normal(size=j.shape))).astype(np.complex64)
    return t


def _facets(case):
    # the wide fields' facets tile the sky at the workloads' cell size
    return synth.make_facets(case["nfacet"], case["nx"], 0.4 / 3600.0, 0.3 * DEG)


def _norm(case):
    """Plane normalisation of an image (what its beam gave)."""
    return np.full(case["nplane"], 0.8 * case["rows"] * case["nchan"] / case["nplane"], np.float32)


def prepare(case, seed):
    uv, rows = _uv(case, seed)
    st = dict(case=case, uv=uv, rows=rows)
    if case["kind"] == "dft":
        st["dft"] = SkyModelDFT(uv, _sky(case, uv, seed), op=case["op"], numberPoln=min(2, uv.nstok),
                                nVisPIO=case["piece"])
        if case["path"] == "buffer":
            st["host"] = rows.cpu().numpy()
        else:
            st["dft"].attach_vis(rows.data_ptr(), case["rows"])
    elif case["kind"] == "beam":
        t = _beam_tables(case, uv, seed)
        b = BeamDFT(uv, t["comps"], t["ant_type"], t["jmap"], case["njchan"], ntype=case["ntype"],
                    stok_type=case["stokes"], op=case["op"], stok_fact=STOK_FACT)
        if t["amps"] is not None:
            b.set_amps(t["amps"])
        if case["images"]:
            d = dict(nx=BEAM_N, ny=BEAM_N, proj=0, hwidth=2, crval=(0.0, 0.0),
                     crpix=(BEAM_N // 2 + 1.0, BEAM_N // 2 + 1.0), cdelt=(BEAM_CELL, BEAM_CELL))
            b.set_beams([d] * case["ntype"], list(t["img"]), t["bfreq"], REF_SIZE, -1.0e20)
        else:
            b.set_jones(t["jones"])
        st.update(beam=b, pos=t.get("pos"))
    elif case["kind"] == "grid":
        nci = case["nchan"]
        b, e = synth.coarse_bins(nci, case["nplane"])
        st["grid"] = GPUGrid(uv, _facets(case), nplane=case["nplane"],
                             plane_of_chan=plane_of_channel(nci, b, e, cpu_parity=False), beam=case["beam"])
        st["norm"] = _norm(case)
        if case["path"] == "host":
            st["host"] = rows.cpu().numpy()
        elif case["out"] == "image":
            st["img"] = torch.empty((case["nfacet"], case["nplane"], case["nx"], case["nx"]), device="cuda")
        else:
            st["img"] = torch.empty((case["nfacet"], case["nplane"], case["nx"], case["nx"] // 2 + 1, 2),
                                    device="cuda")
    else:
        st["lib"] = _lib.load()
        st["out"] = torch.empty((case["rows"], 5 + 3 * uv.nif * uv.nchan), device="cuda")
    return st


# ------------------------------------------------------------------ one pass

def _parts(rows):
    """A record's random parameters and its correlations."""
    return [rows[:, :5], rows[:, 5:]]


def run(st):
    case = st["case"]
    if case["kind"] == "dft":
        if case["path"] == "buffer":
            return _parts(st["dft"].calc(st["host"]))
        st["dft"].calc_resident()
        return _parts(st["rows"])
    if case["kind"] == "beam":
        if case["images"]:
            st["beam"].jones_from_beams(st["pos"], PAR_ANG)
        st["beam"].calc_device(st["rows"].data_ptr(), case["rows"], PAR_ANG)
        return _parts(st["rows"])
    if case["kind"] == "stokes":
        stokes_i_device(st["lib"], st["rows"].data_ptr(), st["out"].data_ptr(), st["uv"])
        return _parts(st["out"])
    g = st["grid"]
    g.lib.ObitCUDAGridInit(g.c, 0)     # a new image: the facet grids cleared
    if case["path"] == "host":
        g.grid(st["host"])
        g.flip()
        return [g.to_host(i) for i in range(case["nfacet"])]
    g.grid_device(st["rows"].data_ptr(), case["rows"])
    g.flip()
    if case["out"] == "planes":
        for i in range(case["nfacet"]):
            _lib.check(g.lib.ObitHIPGrid2Device(g.c, i, ctypes.c_void_p(st["img"][i].data_ptr())), "Grid2Device")
        return st["img"]
    norms = []
    for i in range(case["nfacet"]):
        norm = st["norm"].copy()
        _lib.check(g.lib.ObitHIPGridFFT2Image(g.c, i, int(case["beam"]),
                                              norm.ctypes.data_as(ctypes.POINTER(ctypes.c_float)),
                                              ctypes.c_void_p(st["img"][i].data_ptr())), "FFT2Image")
        norms.append(norm)
    return [st["img"], np.stack(norms)]


def work(case):
    rows, nf = case["rows"], case.get("nif", 1) * case["nchan"]
    if case["kind"] == "dft":
        # u, v, w and the selected correlations read and written, the table
        # read; one complex multiply-add per (row, channel, component)
        lrec = 5 + 3 * nf * case["nstok"]
        moved = 2 * lrec if case["path"] == "buffer" else 3 + 5 * nf * min(2, case["nstok"])
        return dict(bytes=4.0 * (rows * moved + 7 * case["ncomp"]), flops=8.0 * rows * nf * case["ncomp"])
    if case["kind"] == "beam":
        return dict(bytes=4.0 * (rows * (4 + 5 * nf * case["ncorr"]) +
                                 8.0 * case["ntype"] * case["ncomp"] * case["njchan"]),
                    flops=8.0 * rows * nf * case["ncomp"] * case["ncorr"])
    if case["kind"] == "stokes":
        return dict(bytes=4.0 * rows * (10 + 3 * nf * (1 + min(2, case["nstok"]))), flops=8.0 * rows * nf)
    planes = case["nfacet"] * case["nplane"]
    half = 8.0 * case["nx"] * (case["nx"] // 2 + 1) * planes
    out = 4.0 * case["nx"] ** 2 * planes if case["out"] == "image" else half
    fft = 2.5 * case["nx"] ** 2 * 2 * math.log2(case["nx"]) * planes if case["out"] == "image" else 0.0
    return dict(bytes=4.0 * rows * (5 + 3 * nf) + half + out, flops=200.0 * rows * nf * case["nfacet"] + fft)


# ------------------------------------------------------------------ 64 bits

def _apply(rows, model, op, weights_rule, sel):
    """Obit's rules for one correlation: data [row, chan, 3] and model."""
    d = sel.double()
    wt = d[..., 2]
    z = torch.complex(d[..., 0], d[..., 1])
    ok = (wt > 0) | (op == "repl")
    if weights_rule is not None:
        ok = ok & weights_rule
    if op == "div":
        new, w = z / model, wt * model.abs()
    else:
        new, w = (z - model if op == "sub" else model), wt
    d[..., 0] = torch.where(ok, new.real, d[..., 0])
    d[..., 1] = torch.where(ok, new.imag, d[..., 1])
    d[..., 2] = torch.where(ok, w, wt)
    return d


def _phasors(uvw, xyz, f):
    """exp(2 pi i (u x + v y + w z) f) [row, comp] for one channel."""
    t = (uvw @ xyz.T) * f
    t = (t - torch.round(t)) * TWOPI
    return torch.complex(torch.cos(t), torch.sin(t))


def _taper(uvw, gp, f):
    u, v = uvw[:, :1] * f, uvw[:, 1:2] * f
    return torch.exp(gp[:, 0] * u * u + gp[:, 1] * v * v + gp[:, 2] * u * v)


def _chunks(n, ncomp):
    step = max(1, int(6.0e7 / max(ncomp, 1)))
    return range(0, n, step), step


def _exact_dft(case, seed):
    uv, rows = _uv(case, seed)
    sky = _sky(case, uv, seed)
    nf, nst = uv.nif * uv.nchan, uv.nstok
    amp = torch.from_numpy(_spectrum(sky, case, uv)).cuda().to(torch.complex128)
    c = torch.from_numpy(sky.comps.astype(np.float64)).cuda()
    xyz, gp = c[:, 1:4] / TWOPI, c[:, 4:7] if case["model"] in ("gauss", "gspec") else None
    out = rows.double()
    fr = uv.freqArr / uv.freq
    todo, step = _chunks(case["rows"], case["ncomp"])
    for r in todo:
        uvw = rows[r:r + step, :3].double()
        vis = out[r:r + step, 5:].view(-1, nf, nst, 3)
        for ch in range(nf):
            e = _phasors(uvw, xyz, float(fr[ch]))
            if gp is not None:
                e = e * _taper(uvw, gp, float(fr[ch]))
            mod = e @ amp[:, ch]
            for s in range(min(2, nst)):
                vis[:, ch, s] = _apply(rows, mod, case["op"], None, vis[:, ch, s])
    return _parts(out.cpu().numpy() if case["path"] == "buffer" else out)


def _lagrange(p, n):
    cen = np.clip(np.floor(p + 0.5).astype(int) - 2, 1, n - 4) - 1
    x = p - cen
    k = np.ones((p.size, 5))
    for j in range(5):
        for i in range(5):
            if i != j:
                k[:, j] *= (x - (i + 1)) / (j - i)
    return cen, k


def _exact_jones(case, t):
    """Jones matrices from the beam images (Lagrange interpolation, the
    reference gain divided out), complex128 [ntype, ncomp, njchan, 2, 2]."""
    pos = t["pos"].astype(np.float64)
    d0, d1 = -pos[:, 0], pos[:, 1]
    ang = np.float32(PAR_ANG)
    cr, sr = math.cos(ang), math.sin(ang)
    cell = float(np.float32(BEAM_CELL))
    px = (d0 * cr + d1 * sr) / cell + BEAM_N // 2 + 1
    py = (d1 * cr - d0 * sr) / cell + BEAM_N // 2 + 1
    xs, xk = _lagrange(px, BEAM_N)
    ys, yk = _lagrange(py, BEAM_N)
    off = np.hypot(d0, d1)
    out = np.zeros((case["ntype"], case["ncomp"], case["njchan"], 4), np.complex128)
    iy, ix = ys[:, None] + np.arange(5), xs[:, None] + np.arange(5)
    for a in range(case["ntype"]):
        for j in range(case["njchan"]):
            arg = float(np.float32(REF_SIZE)) * float(t["bfreq"][j]) * off
            ipb = np.where(arg > 1.02, 100.0, (1.0 - 4.0 * arg * arg) / np.cos(math.pi * arg))
            v = [ipb * np.einsum("nyx,ny,nx->n", t["img"][a, k, j].astype(np.float64)[iy[:, :, None], ix[:, None, :]],
                                 yk, xk) for k in range(8)]
            ok = (ipb < 10.0) & (np.abs(v[0]) <= 1.3)
            for q, (re, im) in enumerate(((0, 1), (4, 5), (6, 7), (2, 3))):
                out[a, :, j, q] = np.where(ok, v[re] + 1j * v[im], 1.0 if q in (0, 3) else 0.0)
    return out.reshape(out.shape[:3] + (2, 2))


def _exact_beam(case, seed):
    uv, rows = _uv(case, seed)
    t = _beam_tables(case, uv, seed)
    nf, nc = uv.nif * uv.nchan, case["ncorr"]
    J = torch.from_numpy(_exact_jones(case, t) if case["images"] else t["jones"].astype(np.complex128)).cuda()
    ang = 2.0 * float(np.float32(PAR_ANG))
    c2, s2 = math.cos(ang), math.sin(ang)
    P = {1: [[1, 0], [0, 1]], 2: [[c2, -s2], [-s2, -c2]], 3: [[s2, c2], [c2, -s2]], 4: [[0, 1j], [-1j, 0]]}
    P = torch.tensor(P[case["stokes"]], dtype=torch.complex128, device="cuda")
    c = torch.from_numpy(t["comps"].astype(np.float64)).cuda()
    xyz, gp = c[:, 1:4] / TWOPI, c[:, 4:7] if case["model"] == "gauss" else None
    amp = c[:, :1].repeat(1, nf) if t["amps"] is None else torch.from_numpy(t["amps"].astype(np.float64)).cuda()
    out = rows.double()
    bl = rows[:, 3].round().long()
    types = torch.from_numpy(t["ant_type"].astype(np.int64)).cuda()
    t1, t2 = types[bl // 256 - 1], types[bl % 256 - 1]
    fr, op = uv.freqArr / uv.freq, case["op"]
    for a in range(case["ntype"]):
        for b in range(case["ntype"]):
            pick = torch.nonzero((t1 == a) & (t2 == b)).flatten()
            todo, step = _chunks(pick.numel(), case["ncomp"])
            C = [J[a, :, j] @ P @ J[b, :, j].conj().transpose(1, 2) for j in range(case["njchan"])]
            for r in todo:
                at = pick[r:r + step]
                uvw = rows[at, :3].double()
                vis = out[at, 5:].view(-1, nf, nc, 3)
                for ch in range(nf):
                    e = _phasors(uvw, xyz, float(fr[ch]))
                    if gp is not None:
                        e = e * _taper(uvw, gp, float(fr[ch]))
                    m = e @ (amp[:, ch, None] * C[int(t["jmap"][ch])].reshape(-1, 4))
                    alive = (vis[:, ch, :, 2] > 0).any(dim=1) | (op == "repl")
                    for s, (prod, f) in enumerate(((0, 0), (3, 3), (1, 1), (2, 2))[:nc]):
                        if op == "div" and s > 1:
                            continue
                        mod = m[:, prod] * float(np.float32(STOK_FACT[f]))
                        vis[:, ch, s] = _apply(rows, mod, op, alive, vis[:, ch, s])
                out[at, 5:] = vis.reshape(at.numel(), -1)
    return _parts(out)


def _gcf():
    """The 101 x 7 gridding table: Schwab's spheroidal function (support 6,
    alpha 1), tabulated as single precision numbers."""
    f4 = np.float32
    lo = ([8.203343e-2, -3.644705e-1, 6.278660e-1, -5.335581e-1, 2.312756e-1], [8.212018e-1, 2.078043e-1], 0.5625)
    hi = ([4.028559e-3, -3.697768e-2, 1.021332e-1, -1.201436e-1, 6.412774e-2], [9.599102e-1, 2.918724e-1], 1.0)
    eta = np.arange(300, dtype=f4) / f4(299)
    e2 = eta * eta
    val = []
    for p, q, x0 in (lo, hi):
        x = e2 - f4(x0)
        num = np.zeros_like(x)
        for k in p[::-1]:
            num = f4(k) + x * num
        val.append((num.astype(np.float64) / (1.0 + (x * (f4(q[0]) + x * f4(q[1]))).astype(np.float64))).astype(f4))
    psi = np.where(eta <= f4(0.75), val[0], val[1])
    psi = np.where(eta == 0, psi, ((1.0 - e2.astype(np.float64)) * psi).astype(f4))
    psi[-1] = 0.0
    fn = np.zeros(708, f4)
    fn[350:650] = psi
    fn[1:350] = fn[699:350:-1]
    fn[700:] = 0.0
    return fn, np.stack([fn[np.arange(7) * 100 + it] for it in range(101)])


def _grid_corr(n, fn):
    """Gridding correction of one axis: defined by a single-precision phase
    ramp over the table (its rounding is part of the definition)."""
    f4 = np.float32
    size, bias, icent = 701, 351, n // 2 + 1
    p4 = f4(TWOPI / (100 * float(n)))
    p1 = f4(float(p4) * (1.0 - icent) * (1.0 - bias))
    p2 = f4(float(p4) * (1.0 - icent))
    p3 = f4(float(p4) * (1.0 - bias))
    i = np.arange(size, dtype=f4)
    ph, pr = p1 + i * p2, p3 + i * p4
    t = fn[:size].astype(np.float64)
    re, im = (t * np.cos(ph.astype(np.float64))).astype(f4), (t * np.sin(ph.astype(np.float64))).astype(f4)
    rr, ri = np.cos(pr.astype(np.float64)).astype(f4), np.sin(pr.astype(np.float64)).astype(f4)
    out = np.zeros(n, f4)
    for k in range(n):
        out[k] = np.cumsum(re, dtype=f4)[-1]
        re, im = re * rr - im * ri, re * ri + im * rr
    out = out * f4(1.0 / float(out[n // 2]))
    return (f4(1.0) / out).astype(np.float64)


def _round_half_away(x):
    d = x.double()
    return torch.where(x >= 0, d + 0.5, d - 0.5).trunc().long()


def _exact_grid(case, seed):
    uv, rows = _uv(case, seed)
    nx, npl, nch = case["nx"], case["nplane"], case["nchan"]
    fn, table = _gcf()
    gcf = torch.from_numpy(table.astype(np.float64)).cuda()
    f4 = np.float32
    cell = abs(f4(DEG * float(f4(0.4 / 3600.0))))
    us, vs = f4(nx * float(cell)), f4(-nx * float(cell))
    guard_u, guard_v = abs(f4(0.4) * f4(nx) / us), abs(f4(0.4) * f4(nx) / vs)
    b, e = synth.coarse_bins(nch, npl)
    fr = uv.fscale
    ncol = nx // 2 + 4
    res, norms = [], []
    for fac in _facets(case):
        shift = [0.0] * 3 if case["beam"] else [float(s) / TWOPI for s in fac.shift]
        u, v, w = (rows[:, i] for i in range(3))
        rot = [float(x) for x in fac.rot]
        uu, vv, ww = (u * rot[3 * i] + v * rot[3 * i + 1] + w * rot[3 * i + 2] for i in range(3))
        sign = torch.where(uu <= 0, -1.0, 1.0)
        grid = torch.zeros(npl * nx * ncol * 2, dtype=torch.float64, device="cuda")
        for p in range(npl):
            for ch in range(int(b[p]), int(e[p]) + 1):
                ff = sign * float(fr[ch])
                cu, cv, cw = uu * ff, vv * ff, ww * ff
                dat = rows[:, 5 + 3 * ch:8 + 3 * ch]
                bl2 = cu * cu + cv * cv
                ok = (dat[:, 2] > 0) & (cu < float(guard_u)) & (cv.abs() < float(guard_v)) & (bl2 < float(f4(1e12) * f4(1e12)))
                ok = torch.nonzero(ok).flatten()
                t = cu.double() * shift[0] + cv.double() * shift[1] + cw.double() * shift[2]
                t = ((t - torch.round(t)) * TWOPI)[ok]
                if case["beam"]:
                    z = torch.ones_like(t).to(torch.complex128)
                else:
                    z = torch.complex(dat[:, 0].double(), dat[:, 1].double() * sign.double())[ok]
                    z = z * torch.complex(torch.cos(t), torch.sin(t))
                z = z * dat[ok, 2].double()
                gu, gv = (cu * float(us))[ok], (cv * float(vs))[ok]
                iu, iv = (gu.double() + 0.5).trunc().long(), _round_half_away(gv)
                tu = 100 + _round_half_away((100.0 * ((iu.float() - gu).double() - 0.5)).float())
                tv = 100 + _round_half_away((100.0 * ((iv.float() - gv).double() - 0.5)).float())
                row0 = iv - 3 + nx // 2
                at = ((p * nx + row0[:, None, None] + torch.arange(7, device="cuda")[None, :, None]) * ncol +
                      iu[:, None, None] + torch.arange(7, device="cuda")[None, None, :]).reshape(-1)
                wt = gcf[tv][:, :, None] * gcf[tu][:, None, :]
                grid.index_add_(0, 2 * at, (wt * z.real[:, None, None]).reshape(-1))
                grid.index_add_(0, 2 * at + 1, (wt * z.imag[:, None, None]).reshape(-1))
        g = torch.view_as_complex(grid.view(npl, nx, ncol, 2))
        # fold the columns left of u = 0 onto their conjugates
        old = g[:, :, :7].clone()
        r1, r2 = torch.arange(1, nx // 2 + 1, device="cuda"), nx - torch.arange(1, nx // 2 + 1, device="cuda")
        for k in range(4):
            g[:, r1, 3 + k] = old[:, r1, 3 + k] + old[:, r2, 3 - k].conj()
            g[:, r2, 3 + k] = old[:, r2, 3 + k] + old[:, r1, 3 - k].conj()
        half = torch.roll(g[:, :, 3:], nx // 2, dims=1)
        if case["out"] == "planes":
            res.append(half.cpu().numpy() if case["path"] == "host" else torch.view_as_real(half.resolve_conj()).clone())
            continue
        img = torch.roll(torch.fft.irfft2(half, s=(nx, nx), norm="forward"), (nx // 2, nx // 2), dims=(1, 2))
        c = torch.from_numpy(_grid_corr(nx, fn)).cuda()
        img = img * c[None, :, None] * c[None, None, :]
        norm = img[:, nx // 2, nx // 2].cpu().numpy().copy() if case["beam"] else _norm(case).astype(np.float64)
        res.append(img / torch.from_numpy(norm).cuda()[:, None, None])
        norms.append(norm)
    if case["path"] == "host":
        return res
    if case["out"] == "planes":
        return torch.stack(res)
    return [torch.stack(res), np.stack(norms)]


def _exact_stokes(case, seed):
    uv, rows = _uv(case, seed)
    nf, nst = uv.nif * uv.nchan, uv.nstok
    vis = rows[:, 5:].view(-1, nf, nst, 3).double()
    out = torch.empty((case["rows"], 5 + 3 * nf), dtype=torch.float64, device="cuda")
    out[:, :5] = rows[:, :5].double()
    o = out[:, 5:].view(-1, nf, 3)
    if nst == 1:
        # true Stokes I: the record's own correlation; half its weight is kept
        w = vis[:, :, 0, 2].clamp(min=0.0) * 0.5
        o[:, :, 2] = 2.0 * w
        o[:, :, :2] = torch.where((w > 0)[..., None], vis[:, :, 0, :2], 0.0)
        return _parts(out)
    w = vis[:, :, :2, 2].clamp(min=0.0) * 0.5
    wt = w.sum(dim=2)
    half = torch.where((w > 0)[..., None], 0.5 * vis[:, :, :2, :2], 0.0).sum(dim=2)
    half = torch.where(((w <= 0).any(dim=2))[..., None], 2.0 * half, half)
    o[:, :, :2] = torch.where((wt > 0)[..., None], half, 0.0)
    o[:, :, 2] = wt
    return _parts(out)


def exact(case, seed):
    nf = case.get("nif", 1) * case["nchan"]
    if case["kind"] == "stokes":
        return _exact_stokes(case, seed)
    if case["kind"] == "grid":
        if case["rows"] * nf * case["nfacet"] > 6.0e7:
            return None
        return _exact_grid(case, seed)
    if case["rows"] * nf * case["ncomp"] > 3.0e11:
        return None
    return _exact_dft(case, seed) if case["kind"] == "dft" else _exact_beam(case, seed)
