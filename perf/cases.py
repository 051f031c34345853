"""The work a user of this package has it do, as cases that can be timed and checked.

Two ways lead from visibilities to dirty images, and both are cases here:

* ``run``: the stage calls in the order CPacerImager::run makes them (the imager class, and any program
  that overrides the class' four stages): geometric and cable corrections in place, gridding into
  grids and counts, ``image`` (FFT, normalisation, shift, grids cleared for the next round) and, when asked
  for, the mean image;
* ``batch``: ``image_batch``, every (timestep, channel) image of one array in one call with the same
  buffers from call to call; ``mixed`` is the same call over many single-image sets of several
  arrays and grid sides.

A case is a dict: the entry, the array ("station": antennas in a 35 m disk, dense in the uv plane; "tiles": a
Gaussian layout of 300 m clipped at 1.5 km), antennas, channels, timesteps, grid side, polarisation,
Kaiser-Bessel footprint (0: nearest cell), transform and whether the mean image is formed.
"""
import math

import numpy as np
import torch

from imager_amd import capi

C_LIGHT = 299792458.0
OVERSAMPLING = 2.0          # the command line's default
MIN_UV = -math.inf          # the class' default
KERNEL_STEPS = 1023         # oversampling of the Kaiser-Bessel kernels
MIXED_SIDES = (128, 180, 256, 512, 1024, 2048)
DEVICE = "cuda:0"
CORRECTIONS = capi.CORR_GEOMETRIC | capi.CORR_CABLE


def _case(name, entry, array, n_ant, n_ch, n_t, side, pol="XX", kernel=0, transform="fft",
          average=False):
    return {"name": name, "entry": entry, "array": array, "n_ant": n_ant, "n_ch": n_ch, "n_t": n_t,
            "side": side, "pol": pol, "kernel": kernel, "transform": transform, "average": average}


def listed():
    return [
        # the command line's single image: one correlation matrix of a 256-antenna station
        _case("run_station_1x180", "run", "station", 256, 1, 1, 180),
        # a coarse channel of the station at an odd side, Stokes I, and its mean image
        _case("run_station_32x225_mean", "run", "station", 256, 32, 1, 225, "I", average=True),
        # a coarse channel of 128 tiles at the ordinary image size, a few dumps
        _case("run_tiles_12x2x1024", "run", "tiles", 128, 12, 2, 1024, "I"),
        # wide-field images of 128 tiles, the largest ordinary side
        _case("run_tiles_4x4096", "run", "tiles", 128, 4, 1, 4096),
        # convolutional gridding through the class
        _case("run_station_16x256_kb7", "run", "station", 256, 16, 1, 256, kernel=7),
        # one image per call in a serving loop
        _case("batch_station_1x180", "batch", "station", 256, 1, 1, 180),
        # a second of 128 tiles: 64 channels of 10 dumps (the benchmark's default workload)
        _case("batch_tiles_64x10x1024", "batch", "tiles", 128, 64, 10, 1024),
        # every fine channel of the band, station all-sky images
        _case("batch_station_768x256", "batch", "station", 256, 768, 1, 256),
        # the same with convolutional gridding
        _case("batch_station_256x256_kb7", "batch", "station", 256, 256, 1, 256, kernel=7),
        # the split-precision transform over the band
        _case("batch_station_768x180_fp16", "batch", "station", 256, 768, 1, 180,
              transform="dft-fp16"),
        # wide-field images, one timestep of 48 channels
        _case("batch_tiles_48x4096", "batch", "tiles", 128, 48, 1, 4096),
        # uneven work in one call: single images of both arrays, six sides, their own flags
        _case("mixed_128", "mixed", "both", 0, 128, 1, 0),
    ]


def _sides(lo, hi, even=False):
    """Grid sides lo .. hi that the FFT takes: prime factors up to 13."""
    found = []
    for n in range(lo, hi + 1):
        m = n
        for p in (2, 3, 5, 7, 11, 13):
            while m % p == 0:
                m //= p
        if m == 1 and not (even and n % 2):
            found.append(n)
    return found


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _near(rng, sides):
    """One of `sides`, evenly over their logarithm."""
    want = math.exp(rng.uniform(math.log(sides[0]), math.log(sides[-1])))
    return min(sides, key=lambda n: abs(math.log(n / want)))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(("run", "run", "run", "run_kb", "batch", "batch", "batch", "batch_kb", "batch_dft",
                       "mixed"))
    if kind == "mixed":
        return {k: v for k, v in _case("", "mixed", "both", 0, _log_int(rng, 16, 128), 1,
                                       0).items() if k != "name"}
    array = "station" if kind in ("run_kb", "batch_kb", "batch_dft") else rng.choice(("station", "tiles"))
    n_ant = rng.randint(160, 256) if array == "station" else rng.randint(96, 128)
    pol = rng.choice(("XX", "XX", "YY", "I", "V"))
    n_t, kernel, transform = 1, 0, "fft"
    power = rng.random() < 0.4  # sides that are powers of two are the usual choice
    if array == "station":
        lo, hi = 128, 512
    else:
        lo, hi = 512, 4096
    sides = [n for n in (128, 256, 512, 1024, 2048, 4096) if lo <= n <= hi] if power else \
        _sides(lo, hi, even=kind not in ("run", "batch"))
    if kind == "batch_kb" or kind == "run_kb":
        sides = [n for n in sides if n <= 300]
        kernel = rng.choice((5, 7, 9))
    if kind == "batch_dft":
        sides = [n for n in sides if n <= 256]
        transform = rng.choice(("dft-bf16", "dft-fp16"))
    side = rng.choice(sides) if power else _near(rng, sides)
    if kind == "run":
        # images of one call: up to a coarse channel's worth, at most 64 Mpixel
        most = max(1, min(32, (1 << 26) // (side * side)))
        n_ch = _log_int(rng, 1, most)
        n_t = rng.randint(1, max(1, min(4, most // n_ch)))
    elif kind == "run_kb":
        n_ch = _log_int(rng, 1, 24)
    elif kind == "batch_kb":
        n_ch = _log_int(rng, 8, 256)
    elif kind == "batch_dft":
        n_ch = _log_int(rng, 32, 512)
    else:
        # at most 512 Mpixel, and for the station 768 channels
        most = max(1, min(768, (1 << 29) // (side * side)))
        n_img = _log_int(rng, 1, most)
        n_t = rng.choice((1, 1, 2, 4, 10))
        n_ch = max(1, n_img // n_t)
    c = _case("", "run" if kind.startswith("run") else "batch", array, n_ant, n_ch, n_t, side, pol,
              kernel, transform, average=kind in ("run", "batch") and rng.random() < 0.2)
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs


def _antennas(n_ant):
    a1 = np.repeat(np.arange(n_ant), np.arange(1, n_ant + 1))
    a2 = np.concatenate([np.arange(i + 1) for i in range(n_ant)])
    return a1, a2


class _Array:
    """One array's host-side geometry, flags and grid scalars (small: made with numpy)."""

    def __init__(self, rng, array, n_ant, side, flag_fraction=0.0):
        if array == "station":
            r, th = 17.5 * np.sqrt(rng.random(n_ant)), 2 * np.pi * rng.random(n_ant)
            x, y = r * np.cos(th), r * np.sin(th)
        else:
            x, y = np.empty(0), np.empty(0)
            while len(x) < n_ant:
                px, py = rng.normal(0, 300.0, (2, 2 * n_ant))
                keep = px * px + py * py <= 1500.0 ** 2
                x, y = np.concatenate([x, px[keep]]), np.concatenate([y, py[keep]])
            x, y = x[:n_ant], y[:n_ant]
        z = rng.normal(0, 0.5, n_ant)
        a1, a2 = _antennas(n_ant)
        self.a1, self.a2 = a1, a2
        self.u, self.v, self.w = ((-(p[a1] - p[a2])).astype(np.float32) for p in (x, y, z))
        bad = rng.choice(n_ant, 2, replace=False)  # two dead antennas
        flags = (a1 == a2) | np.isin(a1, bad) | np.isin(a2, bad)
        flags |= rng.random(len(flags)) < flag_fraction
        self.flags = flags.astype(np.int32)
        self.cable = rng.uniform(50.0, 300.0, n_ant)
        ok = self.flags == 0
        self.du, self.dv = (OVERSAMPLING * float(np.max(np.abs(p[ok].astype(np.float64)))) / side
                            for p in (self.u, self.v))
        self.n_bl = len(flags)
        self.sources = rng.uniform(-0.6, 0.6, (2, 20 if array == "tiles" else 5))
        self.flux = rng.uniform(1.0, 10.0, self.sources.shape[1])
        self.noise = 0.5 if array == "tiles" else 0.1


def _frequencies(array, n_ch):
    if array == "tiles" and n_ch > 1:
        return 170e6 + 30e6 * np.arange(n_ch) / (n_ch - 1)
    return (169.60 + 0.04 * np.arange(n_ch)) * 1e6  # 40 kHz fine channels


def _visibilities(a, freq, n_t, gen):
    """complex64 [n_t][n_ch][n_bl][4]: point sources seen through the array, cable delays and w-terms
    included, and noise; one dump in ten thousand records is lost (NaN)."""
    dev = lambda p: torch.from_numpy(np.ascontiguousarray(p)).to(DEVICE)
    f = dev(freq)
    u, v = dev(a.u).double(), dev(a.v).double()
    delay = dev(a.w).double() - (dev(a.cable)[dev(a.a2)] - dev(a.cable)[dev(a.a1)])
    n_ch = len(freq)
    vis = torch.empty((n_t, n_ch, a.n_bl, 4, 2), dtype=torch.float32, device=DEVICE)
    vis.normal_(0.0, a.noise, generator=gen)
    for lo in range(0, n_ch, 64):
        k = (-2 * math.pi / C_LIGHT) * f[lo:lo + 64, None]
        re = torch.zeros((k.shape[0], a.n_bl), dtype=torch.float32, device=DEVICE)
        im = torch.zeros_like(re)
        for (l, m), s in zip(a.sources.T, a.flux):
            turns = k * (u * l + v * m + delay)[None] / (2 * math.pi)
            ph = ((turns - torch.round(turns)) * (2 * math.pi)).float()
            re.add_(torch.cos(ph), alpha=s)
            im.add_(torch.sin(ph), alpha=s)
        sky = torch.stack((re, im), -1)
        vis[:, lo:lo + 64, :, 0] += sky
        vis[:, lo:lo + 64, :, 3] += 0.9 * sky
    n_rec = n_t * n_ch * a.n_bl
    lost = torch.randint(0, n_rec, (max(1, n_rec // 10000),), device=DEVICE, generator=gen)
    vis.view(n_rec, 8)[lost] = math.nan
    return torch.view_as_complex(vis)


def _inputs(array, n_ant, n_ch, n_t, side, seed, gen, flag_fraction=0.0, freq=None):
    a = _Array(np.random.default_rng(seed), array, n_ant, side, flag_fraction)
    f = _frequencies(array, n_ch) if freq is None else freq
    dev = lambda p: torch.from_numpy(np.ascontiguousarray(p)).to(DEVICE)
    return a, {"vis": _visibilities(a, f, n_t, gen), "u": dev(a.u), "v": dev(a.v), "w": dev(a.w),
               "flags": dev(a.flags), "freq": dev(f), "cable": dev(a.cable),
               "n_ant": n_ant, "n_ch": n_ch, "n_t": n_t, "side": side}


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _mixed_observations(case, seed):
    """The single-image observations of a mixed call, one after another."""
    rng = np.random.default_rng(seed)
    gen = _generator(seed)
    for i in range(case["n_ch"]):
        array = ("tiles", "station")[i // len(MIXED_SIDES) % 2]  # every side with both arrays
        side = MIXED_SIDES[i % len(MIXED_SIDES)]
        freq = np.array([(169.60 + 0.04 * int(rng.integers(768))) * 1e6])
        flagged = float(rng.uniform(0.0, 0.3))
        yield _inputs(array, 128 if array == "tiles" else 256, 1, 1, side, int(rng.integers(1 << 31)),
                      gen, flagged, freq)


_contexts = []


def _context():
    """The process' imaging context: a program keeps one for all it images."""
    if not _contexts:
        _contexts.append(capi.Context(0))
    return _contexts[0]


def _image_set(a, d, images, pol="XX", transform=capi.TRANSFORM_FFT, average=None, kernel=0):
    return capi.make_set(d["vis"], d["n_ant"], d["n_ch"], d["n_t"], d["u"], d["v"], d["w"], d["flags"],
                         d["freq"], d["cable"], CORRECTIONS, a.du, a.dv, MIN_UV, d["side"], pol, images,
                         transform=transform, average=average, kernel_size=kernel)


TRANSFORMS = {"fft": capi.TRANSFORM_FFT, "dft-bf16": capi.TRANSFORM_DFT_BF16X3,
              "dft-fp16": capi.TRANSFORM_DFT_FP16X3}


def prepare(case, seed):
    ctx = _context()
    if case["entry"] == "mixed":
        obs = list(_mixed_observations(case, seed))
        out = torch.empty(sum(d["side"] ** 2 for _, d in obs), dtype=torch.complex64, device=DEVICE)
        sets, at = [], 0
        for a, d in obs:
            n = d["side"] ** 2
            sets.append(_image_set(a, d, out[at:at + n]))
            at += n
        return {"ctx": ctx, "case": case, "sets": sets, "keep": [d for _, d in obs], "out": {"images": out}}
    n, n_ch, n_t = case["side"], case["n_ch"], case["n_t"]
    a, d = _inputs(case["array"], case["n_ant"], n_ch, n_t, n, seed, _generator(seed))
    images = torch.empty((n_t, n_ch, n, n), dtype=torch.complex64, device=DEVICE)
    mean = torch.empty((n, n), dtype=torch.complex64, device=DEVICE) if case["average"] else None
    state = {"ctx": ctx, "case": case, "a": a, "d": d, "mean": mean}
    if case["entry"] == "run":
        # the class keeps its grids; it clears them when it allocates them, and imaging clears them again
        state["images"] = images
        state["grids"] = torch.zeros((n_t, n_ch, n, n), dtype=torch.complex64, device=DEVICE)
        state["counts"] = torch.zeros((n_t, n_ch, n, n), dtype=torch.float32, device=DEVICE)
        return state
    # a batched call that wants the mean alone does not form the images
    alone = mean is not None and n % 2 == 0 and case["transform"] == "fft"
    images = None if alone else images
    state["sets"] = [_image_set(a, d, images, case["pol"], TRANSFORMS[case["transform"]], mean,
                                case["kernel"])]
    state["out"] = {k: t for k, t in (("images", images), ("mean", mean)) if t is not None}
    return state


def run(state):
    ctx = state["ctx"]
    if "sets" in state:
        ctx.image_batch(state["sets"])
        return state["out"]
    case, a, d = state["case"], state["a"], state["d"]
    shape = (d["n_ant"], d["n_ch"], d["n_t"])
    n, n_img = d["side"], d["n_ch"] * d["n_t"]
    # in place, as the stages are defined: a second pass over the same dump turns its phases further
    ctx.apply_geometric_corrections(d["vis"], *shape, d["w"], d["freq"])
    ctx.apply_cable_corrections(d["vis"], *shape, d["cable"], d["freq"])
    if case["kernel"]:
        ctx.gridding_kernel(d["vis"], *shape, d["u"], d["v"], d["flags"], d["freq"], a.du, a.dv, MIN_UV, n,
                            case["pol"], capi.WEIGHTING_NATURAL, case["kernel"], state["grids"],
                            state["counts"])
    else:
        ctx.gridding(d["vis"], *shape, d["u"], d["v"], d["flags"], d["freq"], a.du, a.dv, MIN_UV, n,
                     case["pol"], capi.WEIGHTING_NATURAL, state["grids"], state["counts"])
    ctx.image(state["grids"], state["counts"], n, n_img, state["images"])
    out = {"vis": d["vis"], "images": state["images"]}
    if case["average"]:
        ctx.image_averaging(state["images"], n * n, n_img, state["mean"])
        out["mean"] = state["mean"]
    return out


# ------------------------------------------------------------------ work


def work(case):
    """Bytes: the inputs read once, the outputs written once.  A ``run`` pass also owes the caller the
    corrected visibilities, and grids and counts that are read (what gridding left) and cleared.
    Operations: the FFT of every image, and the Kaiser-Bessel footprints."""
    def fft(n):
        return 2 * 5.0 * n * n * math.log2(n)

    if case["entry"] == "mixed":
        # half of the images from each array, the sides in equal numbers
        bl = 0.5 * (128 * 129 / 2 + 256 * 257 / 2)
        px = sum(n * n for n in MIXED_SIDES) / len(MIXED_SIDES)
        return {"bytes": case["n_ch"] * (bl * (8 + 16) + 8.0 * px),
                "flops": case["n_ch"] * sum(fft(n) for n in MIXED_SIDES) / len(MIXED_SIDES)}
    n, n_img = case["side"], case["n_ch"] * case["n_t"]
    n_bl = case["n_ant"] * (case["n_ant"] + 1) // 2
    products = 1 if case["pol"] in ("XX", "YY") else 2
    flops = n_img * (fft(n) + 8.0 * n_bl * max(1, case["kernel"]) ** 2)
    if case["entry"] == "run":
        nbytes = n_img * (2 * 32.0 * n_bl + 8.0 * n * n + 2 * 12.0 * n * n)
        nbytes += 8.0 * n * n if case["average"] else 0.0
    else:
        formed = 0 if case["average"] and n % 2 == 0 and case["transform"] == "fft" else n_img
        nbytes = n_img * 8.0 * products * n_bl + 8.0 * n * n * (formed + (1 if case["average"] else 0))
    return {"bytes": nbytes + 16.0 * n_bl, "flops": flops}


# ----------------------------------------------------------------- exact


def _shift_source(n):
    """source[o] = p with fft_shift(p) = o: halves swapped, the middle of an odd side kept."""
    h, odd = n // 2, n % 2
    p = np.arange(n)
    to = np.where(p < h, p + h + odd, p - h - odd)
    if odd:
        to[h] = h
    source = np.empty(n, np.int64)
    source[to] = p
    return torch.from_numpy(source).to(DEVICE)


def _bessel_i0(x):
    total = term = 1.0
    d = 0.0
    while term > total * 1e-8:  # the kernels are defined by the series stopped here
        d += 2.0
        term *= x * x / (d * d)
        total += term
    return total


def _kernel_table(K):
    """[1023][K]: the oversampled Kaiser-Bessel (alpha 8.6) times sinc kernel of every fractional cell position."""
    n, os_ = K * KERNEL_STEPS, KERNEL_STEPS
    mid = n // 2
    k1 = np.zeros(n)
    norm = os_ / _bessel_i0(8.6)
    for i in range(mid + 1):
        sinc = 1.0 / os_ if i == 0 else math.sin(math.pi * i / os_) / (math.pi * i)
        t = i / mid
        if mid + i < n:
            k1[mid + i] = sinc * _bessel_i0(8.6 * math.sqrt(1.0 - t * t)) * norm
    k1[:mid] = k1[n - mid:][::-1]
    return torch.from_numpy(np.ascontiguousarray(k1.reshape(K, os_).T[::-1])).to(DEVICE)


def _round_away(x):
    t = torch.trunc(x)
    return t + torch.where((x - t).abs() >= 0.5, torch.sign(x), torch.zeros_like(x))


def _exact_images(a, d, pol, kernel, corrected=None):
    """The images of one observation in 64 bits, [n_t][n_ch][N][N]; `corrected`: list that takes the corrected
    visibilities."""
    n = d["side"]
    delay = d["w"].double() - (d["cable"][torch.from_numpy(a.a2).to(DEVICE)] -
                               d["cable"][torch.from_numpy(a.a1).to(DEVICE)])
    source = _shift_source(n)
    table = _kernel_table(kernel) if kernel else None
    images = torch.empty((d["n_t"], d["n_ch"], n, n), dtype=torch.complex128, device=DEVICE)
    unflagged = d["flags"] == 0
    for ch in range(d["n_ch"]):
        nu = d["freq"][ch]
        wavelength = C_LIGHT / nu
        ue, ve = d["u"].double() / wavelength / a.du, d["v"].double() / wavelength / a.dv
        up, vp = _round_away(ue).long(), _round_away(ve).long()
        turns = delay * nu / C_LIGHT
        turn = torch.polar(torch.ones_like(delay), 2 * math.pi * (turns - torch.round(turns)))
        for t in range(d["n_t"]):
            vis = d["vis"][t, ch].to(torch.complex128) * turn[:, None]
            if corrected is not None:
                corrected[0][t, ch] = vis
            val = {"XX": lambda: vis[:, 0], "YY": lambda: vis[:, 3],
                   "I": lambda: 0.5 * (vis[:, 0] + vis[:, 3]),
                   "V": lambda: 0.5j * (vis[:, 1] - vis[:, 2])}[pol]()
            ok = unflagged & ~torch.isnan(val.real) & ~torch.isnan(val.imag)
            val, x0, y0 = val[ok], up[ok], vp[ok]
            grid = torch.zeros((n * n, 2), dtype=torch.float64, device=DEVICE)
            if kernel:
                row = lambda e, p: table[(_round_away((e[ok] - p) * 1023.0).long() + 1534) % 1023]
                wx, wy = row(ue, x0), row(ve, y0)
            for s in (1, -1):
                v = torch.view_as_real(val if s > 0 else val.conj().resolve_conj())
                if not kernel:
                    grid.index_add_(0, ((s * y0) % n) * n + (s * x0) % n, v)
                    continue
                for j in range(kernel):
                    for c in range(kernel):
                        at = []
                        for p in (y0 - kernel // 2 + j, x0 - kernel // 2 + c):
                            i = s * p + n // 2
                            at.append(torch.where(i < n // 2, i + n // 2, i - n // 2))
                        w = wy[:, j] * wx[:, c]
                        inside = (at[0] >= 0) & (at[0] < n) & (at[1] >= 0) & (at[1] < n)
                        grid.index_add_(0, torch.where(inside, at[0] * n + at[1], 0),
                                        v * (w * inside)[:, None])
            plane = torch.fft.ifft2(torch.view_as_complex(grid).view(n, n), norm="forward")
            images[t, ch] = plane[source][:, source] / (2.0 * val.numel())
    return images


def exact(case, seed):
    if case["entry"] == "mixed":
        return {"images": torch.cat([_exact_images(a, d, "XX", 0).flatten()
                                     for a, d in _mixed_observations(case, seed)])}
    n, n_ch, n_t = case["side"], case["n_ch"], case["n_t"]
    a, d = _inputs(case["array"], case["n_ant"], n_ch, n_t, n, seed, _generator(seed))
    if case["entry"] == "run":
        corrected = [torch.empty(d["vis"].shape, dtype=torch.complex128, device=DEVICE)]
        images = _exact_images(a, d, case["pol"], case["kernel"], corrected)
        out = {"vis": corrected[0], "images": images}
        if case["average"]:
            out["mean"] = images.mean((0, 1))
        return out
    images = _exact_images(a, d, case["pol"], case["kernel"])
    # a batched call's images are exactly real
    out = {}
    if not (case["average"] and n % 2 == 0 and case["transform"] == "fft"):
        out["images"] = images.real.to(torch.complex128)
    if case["average"]:
        out["mean"] = images.mean((0, 1)).real.to(torch.complex128)
    return out
