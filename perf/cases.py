"""The workloads whose speed counts, through the package's public entry points.

Each case is a dict of plain values; its "kind" names the entry point:

  pair       torch_ops.beam_convolve of one detector pair, and the gradients
             that the case asks for through autograd
  host       pypisco.GPUConvolver on host arrays (update_scan, then
             exec_convolution), as a program written for the reference calls it
  batch      batched.DetectorBatch: many pairs on one boresight pointing, the
             TOD of all of them and the sky gradient
  focalplane pointing.focal_plane_to_sky, then the TOD of a DetectorBatch with
             a pointing of its own for each pair
  map        mapmaker.DeviceSkyMap: one binned map of many detectors

Inputs: pixel-noise skies (uK), Gaussian beams with or without a cross-polar
part, constant-elevation or raster scans with seeded start times and centres.
exact() evaluates the same quantities in float64 torch from their formulas.
"""
import math

import numpy as np
import torch

from pisco4cmb_amd import batched, mapmaker, pointing, pypisco, torch_ops

DEG = math.pi / 180.0
TWO_PI = 2.0 * math.pi
MAX_VISITS = 2.2e9          # (sample, disc pixel) pairs of the largest drawn case


def listed():
    return [
        # the smallest useful call: a short pointing list on a coarse sky, where
        # launches and host work count (interactive checks, unit-sized jobs)
        dict(name="tod_512_samples", kind="pair", nside=64, nside_beam=512, cap=3.0, fwhm=1.0,
             samples=512, scan="ces", cross=False, vterm=False, sky_grad=False, beam_grad=False),
        # a raster over a small patch, with every gradient: one step of fitting
        # a sky and a beam to a calibration scan
        dict(name="fit_raster_2p5deg", kind="pair", nside=128, nside_beam=1024, cap=2.5, fwhm=1.0,
             samples=10000, scan="raster", cross=True, vterm=False, sky_grad=True,
             beam_grad=True),
        # the plain drop-in simulation: a whole-sky scan, small discs
        dict(name="tod_1p5deg", kind="pair", nside=256, nside_beam=2048, cap=1.5, fwhm=0.5,
             samples=1000000, scan="ces", cross=False, vterm=False, sky_grad=False,
             beam_grad=False),
        # the same through the reference's host interface, copies included
        dict(name="host_tod_1p5deg", kind="host", nside=256, nside_beam=2048, cap=1.5, fwhm=0.5,
             samples=1000000, scan="ces", cross=False, flag="p"),
        # sky gradient with small discs (map-making by optimisation), ragged length
        dict(name="step_1p5deg", kind="pair", nside=256, nside_beam=2048, cap=1.5, fwhm=0.5,
             samples=300007, scan="ces", cross=False, vterm=False, sky_grad=True,
             beam_grad=False),
        # middle-sized discs, cross-polar beams and a sky with V
        dict(name="tod_v_2p5deg", kind="pair", nside=512, nside_beam=4096, cap=2.5, fwhm=0.5,
             samples=250000, scan="ces", cross=True, vterm=True, sky_grad=False,
             beam_grad=False),
        # the headline shape, forward and sky gradient (a stretch of its scan)
        dict(name="step_5deg", kind="pair", nside=512, nside_beam=4096, cap=5.0, fwhm=0.33,
             samples=360000, scan="ces", cross=False, vterm=False, sky_grad=True,
             beam_grad=False),
        # beam gradient at the headline shape: beam characterisation
        dict(name="beam_step_5deg", kind="pair", nside=512, nside_beam=4096, cap=5.0, fwhm=0.5,
             samples=150001, scan="ces", cross=True, vterm=False, sky_grad=False,
             beam_grad=True),
        # 64 detectors on one boresight pointing, forward and sky gradient
        dict(name="batch_64det", kind="batch", nside=512, npairs=32, fwhm_lo=0.2, fwhm_hi=1.0,
             nside_beam_lo=2048, nside_beam_hi=2048, samples=60000),
        # a fine sky with beams from 0.1 to 1 degree
        dict(name="batch_fine_sky", kind="batch", nside=2048, npairs=16, fwhm_lo=0.1, fwhm_hi=1.0,
             nside_beam_lo=2048, nside_beam_hi=8192, samples=12000),
        # detectors across a focal plane: their pointing, then their TOD
        dict(name="focalplane_16", kind="focalplane", nside=512, nside_beam=2048, npairs=16,
             fwhm=0.5, cap=1.5, radius=4.0, samples=25000),
        # one binned map of 64 detectors
        dict(name="map_64det", kind="map", nside=512, ndet=64, samples=250000),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["pair", "pair", "pair", "host", "batch", "focalplane", "map"])
    if kind in ("pair", "host"):
        nside = rng.choice([64, 96, 128, 200, 256, 384, 512])
        nside_beam = min(4096, nside * rng.choice([4, 8, 8, 12]))
        cap = round(_log(rng, 1.0, 5.0), 3)
        disc = 12.0 * nside * nside * math.sin(0.5 * cap * DEG) ** 2
        samples = int(_log(rng, 100, min(1.0e6, 0.5 * MAX_VISITS / disc)))
        case = dict(kind=kind, nside=nside, nside_beam=nside_beam, cap=cap,
                    fwhm=round(cap / rng.uniform(2.5, 12.0), 3), samples=samples,
                    scan=rng.choice(["ces", "ces", "raster"]), cross=rng.random() < 0.5)
        if kind == "host":
            case["flag"] = rng.choice(["p", "a", "b"])
        else:
            case["vterm"] = rng.random() < 0.25
            case["sky_grad"] = rng.random() < 0.5
            case["beam_grad"] = rng.random() < 0.3
        return case
    if kind == "batch":
        nside = rng.choice([256, 512, 768, 1024, 2048])
        npairs = rng.randint(2, 33)
        lo = round(_log(rng, 0.15, 0.5), 3)
        hi = round(lo * rng.uniform(1.0, 3.0), 3)
        disc = 12.0 * nside * nside * math.sin(1.5 * hi * DEG) ** 2
        samples = int(_log(rng, 500, min(6.0e4, MAX_VISITS / (npairs * disc))))
        return dict(kind=kind, nside=nside, npairs=npairs, fwhm_lo=lo, fwhm_hi=hi,
                    nside_beam_lo=2048, nside_beam_hi=rng.choice([2048, 4096]), samples=samples)
    if kind == "focalplane":
        return dict(kind=kind, nside=rng.choice([128, 256, 512]), nside_beam=2048,
                    npairs=rng.randint(3, 24), fwhm=0.5, cap=round(rng.uniform(1.0, 2.0), 3),
                    radius=round(rng.uniform(1.0, 8.0), 3), samples=int(_log(rng, 500, 3.0e4)))
    return dict(kind=kind, nside=rng.choice([64, 128, 200, 256, 512]), ndet=rng.randint(6, 80),
                samples=int(_log(rng, 1.0e3, 2.0e5)))


# ---- inputs ------------------------------------------------------------------

def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * int(seed) + what)
    return g


def _normal(shape, seed, what, sigma=1.0):
    return sigma * torch.randn(shape, generator=_gen(seed, what), device="cuda")


def _sky(nside, seed):
    """I, Q, U, V: pixel noise of 100 uK (I) and 10 uK (Q, U), V of 1 uK."""
    n = 12 * nside * nside
    return tuple(_normal(n, seed, 1 + k, s) for k, s in enumerate((100.0, 10.0, 10.0, 1.0)))


def _scan(kind, n, seed):
    """ra, dec, pa (float32, radians): a constant-elevation scan (latitude -23
    deg, elevation 45 deg, 1 rpm, 100 Hz) or a raster over a 20 degree patch
    with pa cycling through 0, 45, 90, 135 deg."""
    r = np.random.default_rng([int(seed), 11])
    k = torch.arange(n, dtype=torch.float64, device="cuda")
    if kind == "raster":
        ncol = max(1, math.ceil(math.sqrt(n)))
        row, col = torch.div(k, ncol, rounding_mode="floor"), k % ncol
        col = torch.where(row % 2 == 0, col, ncol - 1 - col)
        step = 20.0 * DEG / max(ncol - 1, 1)
        ra = r.uniform(0.5, 5.5) + step * col - 10.0 * DEG
        dec = r.uniform(-0.9, 0.9) + step * row - 10.0 * DEG
        pa = (k % 4) * 45.0 * DEG
    else:
        t = r.uniform(0.0, 80000.0) + k / 100.0
        az, el, lat = TWO_PI / 60.0 * t, 45.0 * DEG, -23.0 * DEG
        sd = math.sin(el) * math.sin(lat) + math.cos(el) * math.cos(lat) * torch.cos(az)
        dec = torch.arcsin(sd)
        ha = torch.atan2(-torch.sin(az) * math.cos(el), math.sin(el) * math.cos(lat)
                         - math.cos(el) * math.sin(lat) * torch.cos(az))
        ra = torch.remainder(TWO_PI / 86164.0905 * t - ha, TWO_PI)
        pa = torch.atan2(torch.sin(ha),
                         math.tan(lat) * torch.cos(dec) - torch.sin(dec) * torch.cos(ha))
    return ra.float(), dec.float(), pa.float()


def _rings(nside):
    """theta, z, first pixel, pixels and shift (0 or 1/2) of rings 1..4N-1 at
    their own index (entry 0 unused), float64 / int64."""
    n = nside
    r = torch.arange(4 * n, dtype=torch.int64, device="cuda")
    north, south = r < n, r > 3 * n
    rp = torch.where(north, r, torch.where(south, 4 * n - r, torch.full_like(r, n)))
    t = (rp * rp).double() / (3.0 * n * n)
    z = torch.where(north, 1.0 - t, torch.where(south, t - 1.0,
                                                (2 * n - r).double() * 2.0 / (3.0 * n)))
    s = torch.sqrt(torch.where(north | south, t * (2.0 - t), (1.0 - z * z).clamp_min(0.0)))
    theta = torch.atan2(s, z)
    nr = 4 * rp
    start = torch.where(north, 2 * r * (r - 1),
                        torch.where(south, 12 * n * n - 2 * rp * (rp + 1),
                                    2 * n * (n - 1) + (r - n) * 4 * n))
    shift = torch.where(north | south | ((r - n) % 2 == 0), 0.5, 0.0).double()
    return theta, z, start, nr, shift


def _cap_pixels(nside, radius):
    """Pixels of the north-pole cap that a beam of this radius (rad) takes:
    the first pixel of the first ring at or beyond it."""
    theta, _, start, _, _ = _rings(nside)
    ring = int(torch.searchsorted(theta[1:].contiguous(), torch.tensor(radius, device="cuda",
                                                          dtype=torch.float64))) + 1
    return int(start[ring])


def _beam(case_nside, nside_beam, cap, fwhm, cross, seed, what):
    """Beams a and b, float32 [4, npix]: elliptical Gaussians, each with a
    cross-polar field of its own phase when `cross`; unit solid angle on the
    sky's pixels."""
    r = np.random.default_rng([int(seed), 12, what])
    npix = _cap_pixels(nside_beam, cap * DEG)
    theta_r, _, start, nr, shift = _rings(nside_beam)
    nring = int(torch.searchsorted(start[1:].contiguous(), npix)) + 1
    ring = torch.repeat_interleave(torch.arange(1, nring, device="cuda"), nr[1:nring])[:npix]
    p = torch.arange(npix, device="cuda")
    th = theta_r[ring]
    ph = TWO_PI * ((p - start[ring]).double() + shift[ring]) / nr[ring].double()
    out = []
    for _ in range(2):
        sx = fwhm * DEG / math.sqrt(8.0 * math.log(2.0))
        sy = sx * (1.0 - r.uniform(0.0, 0.1))
        p0 = r.uniform(0.0, math.pi)
        x, y = th * torch.cos(ph - p0) / sx, th * torch.sin(ph - p0) / sy
        co = torch.polar(torch.exp(-0.25 * (x * x + y * y)), 0.3 * x * x * float(cross))
        xp = r.uniform(0.2, 0.35) if cross else 0.0
        cx = torch.polar(xp * co.abs() * (0.4 + 0.6 * torch.cos(ph - r.uniform(0.0, 1.5)) ** 2),
                         r.uniform(-1.0, 1.0) + 0.5 * torch.sin(ph))
        i, q = co.abs() ** 2 + cx.abs() ** 2, co.abs() ** 2 - cx.abs() ** 2
        uv = 2.0 * co * cx.conj()
        norm = i.sum() * (case_nside / nside_beam) ** 2
        out.append((torch.stack([i, q, uv.real, -uv.imag]) / norm).float())
    return out


def _batch_specs(case, seed):
    """Pairs of a batch: FWHM spread evenly in logarithm, cap 3 x FWHM, finer
    beam maps for the narrower beams, an angle offset for each."""
    r = np.random.default_rng([int(seed), 13])
    n = case["npairs"]
    specs = []
    for k in range(n):
        u = (k + r.uniform(0.0, 1.0)) / n
        fwhm = case["fwhm_lo"] * (case["fwhm_hi"] / case["fwhm_lo"]) ** u
        nb = case["nside_beam_hi"] if fwhm < 0.35 else case["nside_beam_lo"]
        a, b = _beam(case["nside"], nb, 3.0 * fwhm, fwhm, k % 2 == 1, seed, 100 + k)
        specs.append((a, b, nb, float(r.uniform(-math.pi, math.pi))))
    return specs


def _focal_plane(case, seed):
    """Detector offsets (dx, dy), angles, and the array centre's ra, dec, pa."""
    r = np.random.default_rng([int(seed), 14])
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    n = case["npairs"]
    rad = case["radius"] * DEG * np.sqrt(r.uniform(0.0, 1.0, n))
    ang = r.uniform(0.0, TWO_PI, n)
    ra, dec, pa = _scan("ces", case["samples"], seed)
    return (t(rad * np.cos(ang)), t(rad * np.sin(ang)), t(r.uniform(-math.pi, math.pi, n)),
            ra.double(), dec.double(), pa.double())


# ---- the calls ---------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    n = case["samples"]
    s = dict(case=case)
    if kind in ("pair", "host"):
        sky = _sky(case["nside"], seed)
        ba, bb = _beam(case["nside"], case["nside_beam"], case["cap"], case["fwhm"],
                       case["cross"], seed, 0)
        scan = _scan(case["scan"], n, seed)
    if kind == "pair":
        s["sky"] = [x.requires_grad_(case["sky_grad"]) for x in sky]
        s["beams"] = [b.requires_grad_(case["beam_grad"]) for b in (ba, bb)]
        s["scan"] = scan
        s["g"] = [_normal(n, seed, 21), _normal(n, seed, 22)]
    elif kind == "host":
        conv = pypisco.GPUConvolver(pypisco.default_run_config())
        conv.configure_execution()
        conv.update_sky(pypisco.Sky(case["nside"], *[x.cpu().numpy() for x in sky]))
        beam = pypisco.PolBeam(case["nside_beam"], ba.shape[1], 0.0, "p")
        for k in range(4):
            beam.aBeams[k][:] = ba[k].cpu().numpy()
            beam.bBeams[k][:] = bb[k].cpu().numpy()
        conv.update_beam(beam)
        s["conv"] = conv
        s["scan"] = pypisco.Scan(n, *[x.cpu().numpy() for x in scan])
        s["tod"] = [np.zeros(n, np.float32) if d in _dets(case) else None for d in "ab"]
    elif kind == "batch":
        s["sky"] = _sky(case["nside"], seed)[:3]
        s["batch"] = batched.DetectorBatch(_batch_specs(case, seed))
        s["scan"] = _scan("ces", n, seed)
        s["g"] = _normal((case["npairs"], 2, n), seed, 21)
    elif kind == "focalplane":
        s["sky"] = _sky(case["nside"], seed)[:3]
        specs = []
        for k in range(case["npairs"]):
            a, b = _beam(case["nside"], case["nside_beam"], case["cap"], case["fwhm"],
                         k % 2 == 1, seed, 100 + k)
            specs.append((a, b, case["nside_beam"], 0.0))
        s["batch"] = batched.DetectorBatch(specs)
        s["plane"] = _focal_plane(case, seed)
    else:
        s["map"] = mapmaker.DeviceSkyMap(case["nside"])
        s["scan"] = _scan("ces", n, seed)
        s["pol"], s["data"] = _map_data(case, seed)
    return s


def _dets(case):
    return "ab" if case["flag"] == "p" else case["flag"]


def _map_data(case, seed):
    r = np.random.default_rng([int(seed), 15])
    pol = torch.from_numpy(r.uniform(-math.pi, math.pi, case["ndet"]).astype(np.float32)).cuda()
    return pol, _normal((case["ndet"], case["samples"]), seed, 23, 30.0)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "pair":
        I, Q, U, V = state["sky"]
        V = V if case["vterm"] else None
        ba, bb = state["beams"]
        tod = torch_ops.beam_convolve(I, Q, U, ba, bb, *state["scan"], case["nside"],
                                      case["nside_beam"], V=V)
        wrt = ([I, Q, U] + ([V] if case["vterm"] else []) if case["sky_grad"] else []) + (
            [ba, bb] if case["beam_grad"] else [])
        grads = torch.autograd.grad(tod, wrt, state["g"]) if wrt else ()
        return [t.detach() for t in tod] + list(grads)
    if kind == "host":
        conv = state["conv"]
        conv.update_scan(state["scan"])
        a, b = state["tod"]
        conv.exec_convolution(a, b, case["flag"])
        return [x for x in (a, b) if x is not None]
    if kind == "batch":
        batch, sky, scan = state["batch"], state["sky"], state["scan"]
        tod = batch.forward(*sky, *scan, case["nside"])
        return [tod] + list(batch.adjoint_map(state["g"], *scan, case["nside"]))
    if kind == "focalplane":
        ptg = pointing.focal_plane_to_sky(*state["plane"])
        return list(ptg) + [state["batch"].forward(*state["sky"], *ptg, case["nside"])]
    m = state["map"]
    m.reset()
    m.accumulate(*state["scan"], state["pol"], state["data"], shared_pointing=True)
    return list(m.solve())


def work(case):
    """Inputs read once, outputs written once; operations of the visits: 70 for
    the mapping into the beam frame, 14 for the polarised sum or for one of
    its adjoints."""
    n, kind = case["samples"], case["kind"]
    npix = 12 * case["nside"] ** 2
    disc = lambda cap: npix * math.sin(0.5 * cap * DEG) ** 2
    rows = lambda nb, cap: 12 * nb * nb * math.sin(0.5 * cap * DEG) ** 2
    if kind in ("pair", "host"):
        v = n * disc(case["cap"])
        beam = 32 * rows(case["nside_beam"], case["cap"])
        passes = 1
        nbytes = 12 * npix + beam + 20 * n
        if kind == "pair":
            if case["vterm"]:
                nbytes += 4 * npix
            if case["sky_grad"]:
                passes += 1
                nbytes += 12 * npix + beam + 20 * n
            if case["beam_grad"]:
                passes += 1
                nbytes += 12 * npix + beam + 20 * n
        return dict(bytes=nbytes, flops=84 * v * passes)
    if kind == "batch":
        v = beam = 0.0
        for k in range(case["npairs"]):
            fwhm = case["fwhm_lo"] * (case["fwhm_hi"] / case["fwhm_lo"]) ** (
                (k + 0.5) / case["npairs"])
            v += n * disc(3.0 * fwhm)
            nb = case["nside_beam_hi"] if fwhm < 0.35 else case["nside_beam_lo"]
            beam += 32 * rows(nb, 3.0 * fwhm)
        return dict(bytes=24 * npix + 2 * beam + 24 * n + 16 * n * case["npairs"],
                    flops=2 * 84 * v)
    if kind == "focalplane":
        np_ = case["npairs"]
        return dict(bytes=12 * npix + np_ * 32 * rows(case["nside_beam"], case["cap"]) + 24 * n
                    + 32 * np_ * n,
                    flops=np_ * n * (84 * disc(case["cap"]) + 300))
    return dict(bytes=12 * n + 4 * n * case["ndet"] + 16 * npix,
                flops=n * case["ndet"] * (15 + 60) + 100 * npix)


# ---- the same in float64 -----------------------------------------------------

class _Pair:
    """The convolution of one pair in float64: discs, mapping and sums from
    their formulas, over chunks of samples."""

    def __init__(self, nside, nside_beam, npix_beam):
        self.ns, self.nb, self.npb = nside, nside_beam, npix_beam
        self.theta, self.z, self.start, self.nr, self.shift = _rings(nside)
        self.dec = math.pi / 2.0 - self.theta
        th_b, _, start_b, _, _ = _rings(nside_beam)
        ring = int(torch.searchsorted(start_b[1:].contiguous(), npix_beam, right=True))
        self.rho_max = float(th_b[ring])

    def visits(self, ra, dec, pa):
        """sample, sky pixel, beam pixel and cos/sin 2 chi of the visits of a
        chunk that lie inside the beam."""
        n = self.ns
        th = (math.pi / 2.0 - dec)[:, None]
        lo = torch.searchsorted(self.theta[1:].contiguous(), (th - self.rho_max)).clamp_min(0) + 1
        hi = torch.searchsorted(self.theta[1:].contiguous(), (th + self.rho_max), right=True)
        width = int((hi - lo).max()) + 1
        if width <= 0:
            return None
        ring = lo + torch.arange(width, device="cuda")
        ok = ring <= hi
        ring = torch.where(ok, ring, 1)
        z, z0 = self.z[ring], torch.cos(th)
        xa = 1.0 / torch.sqrt((1.0 - z0) * (1.0 + z0))
        x = (math.cos(self.rho_max) - z * z0) * xa
        ysq = 1.0 - z * z - x * x
        dphi = torch.atan2(torch.sqrt(ysq.clamp_min(0.0)), x)
        whole = (th + self.theta[ring] <= self.rho_max) | (
            th + self.theta[ring] >= TWO_PI - self.rho_max)
        nr = self.nr[ring]
        sh = self.shift[ring]
        phi = torch.remainder(ra, TWO_PI)[:, None]
        k = nr.double() / TWO_PI
        ip0 = torch.floor(k * (phi - dphi) - sh).long() + 1
        ip1 = torch.floor(k * (phi + dphi) - sh).long()
        ip0 = torch.where(whole, torch.zeros_like(ip0), ip0)
        ip1 = torch.where(whole, nr - 1, ip1)
        cnt = torch.where(ok & (whole | (ysq > 0.0)), (ip1 - ip0 + 1).clamp_min(0), 0).flatten()
        first = torch.cumsum(cnt, 0) - cnt
        row = torch.repeat_interleave(torch.arange(cnt.numel(), device="cuda"), cnt)
        ip = ip0.flatten()[row] + torch.arange(row.numel(), device="cuda") - first[row]
        smp = torch.div(row, width, rounding_mode="floor")
        rg = ring.flatten()[row]
        nrv = self.nr[rg]
        pix = self.start[rg] + torch.remainder(ip, nrv)
        dra = (ip.double() + self.shift[rg]) * (TWO_PI / nrv.double()) - torch.remainder(
            ra, TWO_PI)[smp]
        dp, dc = self.dec[rg], dec[smp]
        cdp, sdp, cdc, sdc = torch.cos(dp), torch.sin(dp), torch.cos(dc), torch.sin(dc)
        sd, h2 = torch.sin(dra), 2.0 * torch.sin(0.5 * dra) ** 2
        s_d = torch.sin(dp - dc)
        omc = 2.0 * torch.sin(0.5 * (dp - dc)) ** 2 + cdc * cdp * h2    # 1 - cos rho
        alpha = torch.atan2(sd * cdp, s_d + cdp * sdc * h2)
        beta = torch.atan2(sd * cdc, cdc * sdp * h2 - s_d)
        psi = -pa[smp]
        sigma = math.pi - alpha - psi
        chi2 = 2.0 * (beta - sigma)
        # ang2pix of (rho, sigma), polar cap
        tt = torch.remainder(sigma * (2.0 / math.pi), 4.0)
        tp = tt - torch.floor(tt)
        tmp = self.nb * torch.sqrt(3.0 * omc)
        ir = torch.floor(tp * tmp) + torch.floor((1.0 - tp) * tmp) + 1.0
        bp = (2.0 * ir * (ir - 1.0) + torch.floor(tt * ir)).long()
        keep = bp < self.npb
        return smp[keep], pix[keep], bp[keep], torch.cos(chi2)[keep], torch.sin(chi2)[keep]

    def chunks(self, ra, dec, pa, budget=1.2e7):
        disc = 12.0 * self.ns ** 2 * math.sin(0.5 * self.rho_max) ** 2 + 16.0
        m = max(1, int(budget / disc))
        for s in range(0, ra.numel(), m):
            e = min(ra.numel(), s + m)
            v = self.visits(ra[s:e].double(), dec[s:e].double(), pa[s:e].double())
            if v is not None:
                yield s, e, v


def _exact_pair(ns, nb, sky, ba, bb, scan, g=None, vterm=False, sky_grad=False, beam_grad=False,
                fwd=True):
    """TOD a, b; gradients of the sky (I, Q, U, V) and of the beams, or None."""
    P = _Pair(ns, nb, ba.shape[1])
    I, Q, U, V = (x.detach().double() for x in (*sky[:3], sky[3] if vterm else sky[0]))
    A, B = ba.detach().double(), bb.detach().double()
    n = scan[0].numel()
    tod = torch.zeros((2, n), dtype=torch.float64, device="cuda")
    gs = torch.zeros((4, I.numel()), dtype=torch.float64, device="cuda") if sky_grad else None
    gb = torch.zeros((2, 4, A.shape[1]), dtype=torch.float64, device="cuda") if beam_grad else None
    for s, e, (smp, pix, bp, c, w) in P.chunks(*scan):
        q, u = Q[pix], U[pix]
        x, y = q * c + u * w, u * c - q * w
        for k, (T, sg) in enumerate(((A, 1.0), (B, -1.0))):
            t0, t1, t2 = T[0][bp], T[1][bp], T[2][bp]
            if fwd:
                v = I[pix] * t0 + sg * (t1 * x + t2 * y)
                if vterm:
                    v = v + V[pix] * T[3][bp]
                tod[k, s:e].index_add_(0, smp, v)
            if g is None or not (sky_grad or beam_grad):
                continue
            gk = g[k][s:e].double()[smp]
            if sky_grad:
                gs[0].index_add_(0, pix, gk * t0)
                gs[1].index_add_(0, pix, sg * gk * (t1 * c - t2 * w))
                gs[2].index_add_(0, pix, sg * gk * (t2 * c + t1 * w))
                if vterm:
                    gs[3].index_add_(0, pix, gk * T[3][bp])
            if beam_grad:
                gb[k, 0].index_add_(0, bp, gk * I[pix])
                gb[k, 1].index_add_(0, bp, sg * gk * x)
                gb[k, 2].index_add_(0, bp, sg * gk * y)
                if vterm:
                    gb[k, 3].index_add_(0, bp, gk * V[pix])
    return tod, gs, gb


def _exact_focal_plane(dx, dy, pol, ra, dec, rot):
    """Right ascension, declination and position angle of every detector: the
    great-circle offset (dx, dy) turned by the array's angle."""
    dx, dy, pol = dx[:, None], dy[:, None], pol[:, None]
    cr = torch.cos(dx) * torch.cos(dy)
    sr = torch.sqrt((1.0 - cr) * (1.0 + cr))
    alpha = torch.atan2(torch.sin(dy), torch.sin(dx) * torch.cos(dy))
    gamma = math.pi / 2.0 - alpha - rot
    sy, cy = torch.sin(dec), torch.cos(dec)
    d = torch.asin(cr * sy + sr * cy * torch.cos(gamma))
    a = ra - torch.atan2(sr * torch.sin(gamma), cr * cy - sr * sy * torch.cos(gamma))
    se = cy * torch.sin(rot) * torch.cos(dx) - sy * torch.sin(dx)
    ce = sy * torch.cos(dx) + cy * torch.sin(rot) * torch.sin(dx)
    p = torch.atan2(se, cy * torch.cos(rot) * torch.cos(dy) - ce * torch.sin(dy)) + pol
    return a, d, p


def _map_pixels(ns, ra, dec):
    """RING pixel of each pointing."""
    th, phi = math.pi / 2.0 - dec.double(), torch.remainder(ra.double(), TWO_PI)
    z = torch.cos(th)
    za = z.abs()
    tt = torch.remainder(phi * (2.0 / math.pi), 4.0)
    t1, t2 = ns * (0.5 + tt), ns * z * 0.75
    jp, jm = torch.floor(t1 - t2).long(), torch.floor(t1 + t2).long()
    ir = ns + 1 + jp - jm
    ip = torch.remainder(torch.div(jp + jm - ns + 1 + (1 - ir % 2) + 8 * ns, 2,
                                   rounding_mode="floor"), 4 * ns)
    eq = 2 * ns * (ns - 1) + (ir - 1) * 4 * ns + ip
    tp = tt - torch.floor(tt)
    tmp = ns * torch.sqrt(3.0 * (1.0 - za))
    cr = torch.floor(tp * tmp).long() + torch.floor((1.0 - tp) * tmp).long() + 1
    cip = torch.floor(tt * cr.double()).long()
    cap = torch.where(z > 0, 2 * cr * (cr - 1) + cip, 12 * ns * ns - 2 * cr * (cr + 1) + cip)
    return torch.where(za <= 2.0 / 3.0, eq, cap)


def _exact_map(case, seed):
    ns, npix = case["nside"], 12 * case["nside"] ** 2
    ra, dec, pa = _scan("ces", case["samples"], seed)
    pol, data = _map_data(case, seed)
    pix = _map_pixels(ns, ra, dec)
    sums = torch.zeros((9, npix), dtype=torch.float64, device="cuda")
    one = torch.ones(pix.numel(), dtype=torch.float64, device="cuda")
    for k in range(case["ndet"]):
        psi2 = -2.0 * (pol[k].double() + pa.double())
        c, s, d = torch.cos(psi2), torch.sin(psi2), data[k].double()
        for j, v in enumerate((one, c, s, c * c, c * s, s * s, d, c * d, s * d)):
            sums[j].index_add_(0, pix, v)
    use = sums[0] >= 3
    n, c, s, cc, cs, ss, d, cd, sd = (x[use] for x in sums)
    m = torch.stack([n, c, s, c, cc, cs, s, cs, ss], 1).reshape(-1, 3, 3)
    x = torch.linalg.solve(m, torch.stack([d, cd, sd], 1))
    out = torch.zeros((3, npix), dtype=torch.float64, device="cuda")
    out[:, use] = x.T
    return [out[0], out[1], out[2], None]      # the hit counts are whole numbers


def exact(case, seed):
    kind, n = case["kind"], case["samples"]
    if kind == "map":
        return _exact_map(case, seed)
    sky = _sky(case["nside"], seed)
    if kind in ("pair", "host"):
        ba, bb = _beam(case["nside"], case["nside_beam"], case["cap"], case["fwhm"],
                       case["cross"], seed, 0)
        scan = _scan(case["scan"], n, seed)
        if kind == "host":
            tod, _, _ = _exact_pair(case["nside"], case["nside_beam"], sky, ba, bb, scan)
            return [tod["ab".index(d)].cpu().numpy() for d in _dets(case)]
        tod, gs, gb = _exact_pair(case["nside"], case["nside_beam"], sky, ba, bb, scan,
                                  (_normal(n, seed, 21), _normal(n, seed, 22)), case["vterm"],
                                  case["sky_grad"], case["beam_grad"])
        out = [tod[0], tod[1]]
        if case["sky_grad"]:
            out += list(gs if case["vterm"] else gs[:3])
        if case["beam_grad"]:
            out += [gb[0], gb[1]]
        return out
    if kind == "batch":
        scan = _scan("ces", n, seed)
        g = _normal((case["npairs"], 2, n), seed, 21)
        out = torch.zeros((case["npairs"], 2, n), dtype=torch.float64, device="cuda")
        grad = torch.zeros((3, 12 * case["nside"] ** 2), dtype=torch.float64, device="cuda")
        for k, (a, b, nb, off) in enumerate(_batch_specs(case, seed)):
            ptg = (scan[0], scan[1], scan[2] + np.float32(off).item())
            tod, gs, _ = _exact_pair(case["nside"], nb, sky, a, b, ptg, g[k], sky_grad=True)
            out[k] = tod
            grad += gs[:3]
        return [out, grad[0], grad[1], grad[2]]
    ptg = _exact_focal_plane(*_focal_plane(case, seed))
    p32 = [x.float() for x in ptg]
    out = torch.zeros((case["npairs"], 2, n), dtype=torch.float64, device="cuda")
    for k in range(case["npairs"]):
        a, b = _beam(case["nside"], case["nside_beam"], case["cap"], case["fwhm"], k % 2 == 1,
                     seed, 100 + k)
        out[k] = _exact_pair(case["nside"], case["nside_beam"], sky, a, b,
                             [x[k] for x in p32])[0]
    return list(ptg) + [out]
