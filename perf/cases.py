"""The calls this framework is measured by, over the ranges they are used in.

A case is one pass through the public entry points of rexlib_amd: insertions
of spectra and of images into half-complex accumulators (the hot path), whole
reconstructions, and the steps beside the path (background standardization,
transforms over any axes, density compensation, its training). ``listed`` holds
the fixed cases, ``draw`` makes more of the same ranges, ``exact`` computes
the results in float64 with plain torch or numpy.
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch

import rexlib_amd
from rexlib_amd import batched, em, fourier, learned, tune

OPTICS = (300.0, 2.7, 0.1)  # kV, mm, amplitude contrast
PIXEL = 1.5  # Angstrom
KAISER_BESSEL = (2.0, 9.0)  # half-width and shape of the reference's benchmark
LOSS_SCALE = 1024.0


def listed():
    return [
        # The smallest benchmark shape of the reference (64^2 into 128^3, 64
        # slices, linear): a handful of launches, so latency counts.
        dict(name="slices_64_plain", kind="slices", variant="plain", n=64, big=128, count=64, window="linear",
             views="uniform", source="spectra"),
        # The reference's benchmark with the Kaiser-Bessel window (128^2 into
        # 256^3, 256 slices): 64 taps per sample.
        dict(name="slices_128_kb", kind="slices", variant="ctf", n=128, big=256, count=256,
             window="kaiser_bessel", views="uniform", source="spectra"),
        # The reference's largest benchmark shape (256^2 into 512^3) as the
        # two calls of rexlib's API, rfft2 and insert_ctf_slices: few images
        # into a volume of 1.6 GB of accumulators.
        dict(name="slices_256_to_512", kind="slices", variant="ctf", n=256, big=512, count=256, window="linear",
             views="uniform", source="images"),
        # Per-element weights, odd extents (no Nyquist, tabulated volume phase).
        dict(name="slices_99_weighted_odd", kind="slices", variant="weighted", n=99, big=199, count=300,
             window="linear", views="cone", source="spectra"),
        # One launch of the headline workload: 4,096 float32 images 256^2
        # into 256^3.
        dict(name="images_256_f32", kind="images", m=256, padded=0, big=256, count=4096, dtype="f32",
             window="linear", views="uniform"),
        # One launch of the reduced-precision workload: 128^2 bfloat16 images
        # zero-padded on chip to 256^2, into 256^3.
        dict(name="images_128_bf16_padded", kind="images", m=128, padded=256, big=256, count=4096, dtype="bf16",
             window="linear", views="uniform"),
        # A smaller particle set of preferred orientation in scaled float16,
        # with a box (180) that is no power of two.
        dict(name="images_180_f16_cone", kind="images", m=180, padded=0, big=180, count=1000, dtype="f16",
             window="linear", views="cone"),
        # A whole reconstruction of the batched workload's largest box: 1,000
        # images 320^2, insertion, quotient, irfft3, gridding correction.
        dict(name="reconstruct_320", kind="reconstruct", n=320, count=1000, views="uniform"),
        # Background standardization of a micrograph's worth of particles
        # before they are inserted.
        dict(name="standardize_256", kind="standardize", n=256, count=2048),
        # Real transforms there and back over images of a box with a factor 7
        # (no 2-3-5 length).
        dict(name="fourier_252", kind="fourier", form="real", depth=200, rows=252, columns=252),
        # Both density compensations of one weight volume (the iterative one
        # and the shipped perceptron's), as the first reconstruction of a set
        # of orientations computes them.
        dict(name="compensation_256", kind="compensation", big=256),
        # The gradients of one training batch of the perceptron.
        dict(name="gradients_8192", kind="gradients", rows=8192),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choices(["slices", "images", "reconstruct", "standardize", "fourier", "compensation", "gradients"],
                       [5, 5, 3, 2, 2, 1, 1])[0]
    views = rng.choice(["uniform", "cone"])
    if kind == "slices":
        variant = rng.choice(["plain", "weighted", "ctf"])
        n = rng.randint(48, 224)
        big = rng.choice([n, 2 * n, n + rng.randint(1, n)])
        window = rng.choice(["linear", "linear", "kaiser_bessel"])
        # About half the taps of the largest listed case at most.
        most = min(4096, int(4e8 / (n * n * (64 if window == "kaiser_bessel" else 8))))
        source = "spectra"
        if variant == "ctf" and rng.random() < 0.4:
            source = "images"
            n, big = rng.choice([(64, 128), (96, 96), (128, 128), (160, 256), (192, 192), (200, 300)])
        return dict(kind=kind, variant=variant, n=n, big=big, count=_log_int(rng, 16, max(17, most)),
                    window=window, views=views, source=source)
    if kind == "images":
        m = rng.choice([64, 80, 96, 100, 120, 128, 144, 150, 162, 180, 192, 200, 216, 240, 250, 256])
        padded = rng.choice([0, 0, 2 * m]) if m <= 128 else 0
        n = padded or m
        big = rng.choice([n, n, n + rng.randint(0, 31)])
        return dict(kind=kind, m=m, padded=padded, big=big, count=_log_int(rng, 32, int(1.3e8 / (n * n))),
                    dtype=rng.choice(["f32", "bf16", "f16"]), window="linear", views=views)
    if kind == "reconstruct":
        n = rng.choice([64, 72, 96, 100, 128, 135, 160, 192, 225, 256, 320])
        return dict(kind=kind, n=n, count=_log_int(rng, 200, max(400, int(6e7 / (n * n)))), views=views)
    if kind == "standardize":
        n = rng.randint(48, 400)
        return dict(kind=kind, n=n, count=_log_int(rng, 8, max(16, int(6e7 / (n * n)))))
    if kind == "fourier":
        form = rng.choice(["real", "complex", "volume"])
        if form == "volume":
            depth, rows, columns = (rng.randint(32, 200) for _ in range(3))
        else:
            rows, columns = rng.randint(32, 500), rng.randint(32, 500)
            depth = _log_int(rng, 4, max(8, int(1.2e7 / (rows * columns))))
        return dict(kind=kind, form=form, depth=depth, rows=rows, columns=columns)
    if kind == "compensation":
        return dict(kind=kind, big=2 * rng.randint(32, 128))
    return dict(kind=kind, rows=_log_int(rng, 500, 100000))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _rotations(count, views, rng):
    """Uniform orientations, or 80 % of the views in a cone around the top
    view (von Mises-Fisher, concentration 10) and the rest uniform."""
    q = rng.normal(size=(count, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    if views == "cone":
        some = rng.uniform(size=count) < 0.8
        u = rng.uniform(size=count)
        tilt = np.arccos(np.clip(1.0 + np.log(u + (1.0 - u) * math.exp(-20.0)) / 10.0, -1, 1))
        about, spin = rng.uniform(0, 2 * math.pi, count), rng.uniform(0, 2 * math.pi, count)
        # Rz(about) Ry(tilt) Rz(spin) as a quaternion.
        c, s = np.cos(tilt / 2), np.sin(tilt / 2)
        cone = np.stack([c * np.cos((about + spin) / 2), s * np.sin((spin - about) / 2),
                         s * np.cos((spin - about) / 2), c * np.sin((about + spin) / 2)], axis=1)
        q = np.where(some[:, None], cone, q)
    w, x, y, z = q.T
    return np.stack([
        np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)], axis=1),
        np.stack([2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x)], axis=1),
        np.stack([2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], axis=1)], axis=1)


def _geometry(case, seed):
    """Transforms with shifts of a few pixels, CTF parameters: float32 on the device."""
    rng = np.random.default_rng(seed)
    count = case["count"]
    t = np.zeros((count, 3, 4), np.float32)
    t[:, :, :3] = _rotations(count, case["views"], rng)
    t[:, :2, 3] = rng.uniform(-3, 3, (count, 2))
    mean = rng.uniform(10000, 30000, count)
    delta = rng.uniform(0, 1000, count)
    ctf = np.stack([mean + delta / 2, mean - delta / 2, rng.uniform(0, math.pi, count), np.zeros(count)],
                   axis=1).astype(np.float32)
    return torch.from_numpy(t).cuda(), torch.from_numpy(ctf).cuda()


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _images(count, n, g):
    """Particle images: white noise over a centred blob of a tenth of its variance."""
    images = torch.randn((count, n, n), dtype=torch.float32, device="cuda", generator=g)
    r = torch.arange(n, device="cuda", dtype=torch.float32) - n // 2
    blob = torch.exp(-r * r / (2 * (n / 10.0) ** 2))
    return images.add_(blob[:, None] * blob[None, :] * torch.rand((count, 1, 1), device="cuda", generator=g))


def _stage(images, dtype):
    if dtype == "bf16":
        return images.to(torch.bfloat16), None
    if dtype == "f16":
        scales = images.abs().amax(dim=(-2, -1)) / 32768.0
        return (images / scales[:, None, None]).to(torch.float16), scales
    return images, None


def _window(name):
    return em.GriddingWindow.linear() if name == "linear" else em.GriddingWindow.kaiser_bessel(*KAISER_BESSEL)


def _accumulators(big, g):
    """Sums of earlier insertions."""
    shape = (big, big, big // 2 + 1)
    return (torch.randn(shape, dtype=torch.complex64, device="cuda", generator=g),
            torch.rand(shape, dtype=torch.float32, device="cuda", generator=g))


def _weight_volume(big, g):
    """A weight volume as an insertion leaves it: the sampling density falls
    as 1 / |g|, each voxel a few squared CTFs, empty corners."""
    f = torch.fft.fftfreq(big, d=1.0 / big, device="cuda")
    x = torch.arange(big // 2 + 1, device="cuda", dtype=torch.float32)
    r = torch.sqrt(f[:, None, None] ** 2 + f[None, :, None] ** 2 + x[None, None, :] ** 2)
    noise = 0.25 + torch.rand(r.shape, device="cuda", generator=g)
    return torch.where(r < big / 2 + 1, noise * (20.0 * big) / torch.clamp(r, min=1.0), torch.zeros_like(r))


def _coverage(g):
    table = torch.rand((8, 33, 64, 8), device="cuda", generator=g) ** 2
    return table / table.sum(dim=-1, keepdim=True)


def prepare(case, seed):
    kind = case["kind"]
    g = _generator(seed)
    state = dict(case=case)
    if kind in ("slices", "images", "reconstruct"):
        # A program hands the library its tuning table once.
        tune.apply_all()
        state["transforms"], state["ctf"] = _geometry(case, seed)
    if kind == "slices":
        n, h, count = case["n"], case["n"] // 2 + 1, case["count"]
        state["num"], state["den"] = _accumulators(case["big"], g)
        if case["source"] == "images":
            state["images"] = _images(count, n, g)
        else:
            state["slices"] = torch.randn((count, n, h), dtype=torch.complex64, device="cuda", generator=g) * n
        if case["variant"] == "weighted":
            state["weights"] = torch.rand((count, n, h), device="cuda", generator=g) * 2
        # A falling radial weight (an envelope).
        state["radial"] = torch.linspace(1.0, 0.5, h, device="cuda")
        state["window"] = _window(case["window"])
    elif kind == "images":
        n = case["padded"] or case["m"]
        state["images"], state["scales"] = _stage(_images(case["count"], case["m"], g), case["dtype"])
        state["num"], state["den"] = _accumulators(case["big"], g)
        state["radial"] = torch.ones(n // 2 + 1, device="cuda")
        state["window"] = _window(case["window"])
    elif kind == "reconstruct":
        r = batched.Reconstruction(_images(case["count"], case["n"], g), state["transforms"], state["ctf"], PIXEL)
        r.allocate()
        state["reconstruction"] = r
    elif kind == "standardize":
        n, count = case["n"], case["count"]
        images = _images(count, n, g) * 7.0 + 40.0
        # A few hot pixels per image.
        spots = torch.randint(0, n * n, (count, 4), device="cuda", generator=g)
        images.view(count, n * n).scatter_(1, spots, 900.0)
        state["images"] = images
        state["key"] = torch.randint(0, 2 ** 62, (count,), dtype=torch.int64, device="cuda", generator=g)
    elif kind == "fourier":
        dtype = torch.float32 if case["form"] == "real" else torch.complex64
        shape = (case["depth"], case["rows"], case["columns"])
        state["x"] = torch.randn(shape, dtype=dtype, device="cuda", generator=g)
    elif kind == "compensation":
        state["den"] = _weight_volume(case["big"], g)
        state["table"] = _coverage(g)
        state["model"] = learned.shipped_model()
    else:
        rows = case["rows"]
        x = torch.zeros((rows, learned.FEATURES), device="cuda")
        x[:, 0] = torch.rand(rows, device="cuda", generator=g)
        x[:, 1] = torch.rand(rows, device="cuda", generator=g) * 3
        x[:, 2:10] = torch.softmax(torch.randn((rows, 8), device="cuda", generator=g), dim=1)
        state["rows"] = x.to(torch.float16)
        state["target"] = torch.randn(rows, device="cuda", generator=g) * 0.2
        state["model"] = learned.shipped_model()
    return state


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "slices":
        optics = em.CtfOptics(*OPTICS)
        slices = rexlib_amd.rfft2(state["images"]) if case["source"] == "images" else state["slices"]
        if case["variant"] == "plain":
            return em.insert_slices(state["num"], state["den"], slices, state["transforms"], state["radial"],
                                    state["window"])
        if case["variant"] == "weighted":
            return em.insert_weighted_slices(state["num"], state["den"], slices, state["weights"],
                                             state["transforms"], state["radial"], state["window"])
        return em.insert_ctf_slices(state["num"], state["den"], slices, state["transforms"], state["ctf"],
                                    state["radial"], state["window"], optics, PIXEL)
    if kind == "images":
        state["num"].zero_()
        state["den"].zero_()
        return em.insert_ctf_images(state["num"], state["den"], state["images"], state["transforms"], state["ctf"],
                                    state["radial"], state["window"], em.CtfOptics(*OPTICS), PIXEL,
                                    image_scales=state["scales"], padded=case["padded"])
    if kind == "reconstruct":
        r = state["reconstruction"]
        batched.run_one(r)
        return [r.numerator, r.denominator, r.volume]
    if kind == "standardize":
        return em.standardize_background(state["images"], state["key"], 0.4 * case["n"], -6.0, 6.0)
    if kind == "fourier":
        if case["form"] == "real":
            spectra = fourier.rfftn(state["x"], axes=(-2, -1))
            return [spectra, fourier.irfftn(spectra, s=(case["rows"], case["columns"]), axes=(-2, -1))]
        axes = (-2, -1) if case["form"] == "complex" else (-3, -2, -1)
        spectra = fourier.fftn(state["x"], axes=axes)
        return [spectra, fourier.ifftn(spectra, axes=axes)]
    if kind == "compensation":
        return [learned.iterative_weights(state["den"]), state["model"].weights(state["den"], state["table"])]
    gradients, loss = state["model"].gradients(state["rows"], state["target"], LOSS_SCALE)
    return [gradients, loss]


# ---------------------------------------------------------------------------
# Work and tolerances
# ---------------------------------------------------------------------------

def _insertion_work(n, big, count, taps, with_accumulators=24):
    """Bytes of the accumulators (read and written once) and the geometry;
    operations: three sums per tap of the stored samples within the Nyquist
    disk (each lands once in the stored half of the volume)."""
    samples = count * math.pi / 8 * n * n
    return (with_accumulators * big * big * (big // 2 + 1) + count * 64, samples * taps ** 3 * 6)


def work(case):
    kind = case["kind"]
    if kind in ("slices", "images", "reconstruct"):
        count = case["count"]
        if kind == "slices":
            n, big = case["n"], case["big"]
            image = 4 * n * n if case["source"] == "images" else 8 * n * (n // 2 + 1)
            image += 4 * n * (n // 2 + 1) if case["variant"] == "weighted" else 0
            transform = case["source"] == "images"
            taps = 2 if case["window"] == "linear" else 4
        elif kind == "images":
            n, big, taps, transform = case["padded"] or case["m"], case["big"], 2, True
            image = (4 if case["dtype"] == "f32" else 2) * case["m"] ** 2
        else:
            n, big, taps, transform = case["n"], case["n"], 2, True
            image = 4 * n * n
        # In place on zeros nothing is read of the accumulators.
        data, flops = _insertion_work(n, big, count, taps, 24 if kind == "slices" else 12)
        data += count * image
        if transform:
            flops += count * 2.5 * n * n * math.log2(n * n)
        if kind == "reconstruct":
            data += 4 * big ** 3
            flops += 2.5 * big ** 3 * math.log2(big ** 3)
        return dict(bytes=data, flops=flops)
    if kind == "standardize":
        elements = case["count"] * case["n"] ** 2
        return dict(bytes=8 * elements, flops=12 * elements)
    if kind == "fourier":
        a, b, c = case["depth"], case["rows"], case["columns"]
        elements = a * b * c
        points = b * c if case["form"] != "volume" else elements
        if case["form"] == "real":
            half = a * b * (c // 2 + 1)
            return dict(bytes=8 * elements + 16 * half, flops=5.0 * elements * math.log2(points))
        return dict(bytes=32 * elements, flops=10.0 * elements * math.log2(points))
    if kind == "compensation":
        voxels = case["big"] ** 2 * (case["big"] // 2 + 1)
        # The weight volume in, two weight volumes out; ten separable passes
        # and the perceptron.
        return dict(bytes=12 * voxels, flops=voxels * (10 * 20 + 2 * (10 * 64 + 2 * 64 * 64 + 64)))
    return dict(bytes=case["rows"] * 36, flops=case["rows"] * 6 * (10 * 64 + 2 * 64 * 64 + 64))


# Largest relative errors against ``exact`` over the listed cases and two dozen
# drawn ones, times about four. The sums are float32; sample positions round at
# 1e-5 of a voxel (and the Kaiser-Bessel window steps by 1e-3 at its edge, which
# a rounded position can fall on either side of). A finished volume divides by weights down to 1e-3 of one
# sample, and the iterative compensation divides by the density where it
# vanishes, so both amplify the sums' rounding; the perceptron rounds its
# activations and gradients to float16.
TOLERANCE = dict(slices=4e-5, images=3e-5, reconstruct=7e-3, standardize=1e-6, fourier=3e-6, compensation=5e-3,
                 gradients=3e-2)


def tolerance(case):
    if case.get("window") == "kaiser_bessel":
        return dict(rel=4e-4)
    return dict(rel=TOLERANCE[case["kind"]])


# ---------------------------------------------------------------------------
# The results in float64
# ---------------------------------------------------------------------------

def _kaiser_bessel64(d, half_width, shape):
    ratio = torch.clamp(1.0 - (d / half_width) ** 2, min=0.0)
    value = torch.special.i0(shape * torch.sqrt(ratio)) / float(np.i0(shape))
    return torch.where(d.abs() <= half_width, value, torch.zeros_like(value))


def _insert64(num, den, spectra_of, case, n, big, transforms, ctf, radial, weights, window):
    """The insertion's contract, slice group by slice group: `spectra_of(a,
    b)` gives the float64 spectra of slices [a, b)."""
    device = "cuda"
    h, half = n // 2 + 1, big // 2
    count = transforms.shape[0]
    ky = torch.fft.fftfreq(n, d=1.0 / n, device=device, dtype=torch.float64)
    if n % 2 == 0:
        ky[n // 2] = n // 2
    kx = torch.arange(h, device=device, dtype=torch.float64)
    ky, kx = (a.reshape(-1) for a in torch.meshgrid(ky, kx, indexing="ij"))
    shell = torch.floor(torch.sqrt(kx * kx + ky * ky) + 0.5).to(torch.int64)
    inside = shell < h
    if n % 2 == 0:
        inside &= (kx != n // 2) & (ky != n // 2)
    inside = inside.nonzero().squeeze(1)
    kx, ky, r = kx[inside], ky[inside], radial.double()[shell[inside]]
    # Signed frequency of each stored voxel, for the volume's phase.
    f = torch.arange(big, device=device, dtype=torch.float64)
    f = torch.where(f <= half, f, f - big)
    phase = torch.polar(torch.ones_like(f), -2 * math.pi * half * f / big)
    out = torch.zeros((big ** 2 * (half + 1), 3), dtype=torch.float64, device=device)
    half_width, shape = (1.0, 0.0) if window == "linear" else KAISER_BESSEL
    taps = int(math.ceil(2 * half_width))
    group = max(1, (1 << 23) // (inside.numel() * taps))
    for a in range(0, count, group):
        b = min(a + group, count)
        t = transforms[a:b].double()
        x = spectra_of(a, b).reshape(b - a, -1)[:, inside]
        turn = 2 * math.pi / n * (kx * (n // 2 + t[:, 0, 3:4]) + ky * (n // 2 + t[:, 1, 3:4]))
        value = x * torch.polar(torch.ones_like(turn), turn)
        weight = torch.ones_like(turn)
        if case.get("variant", "ctf") == "ctf":
            volts = OPTICS[0] * 1e3
            lam = 12.2643247 / math.sqrt(volts * (1.0 + 0.978466e-6 * volts))
            scale = 1.0 / (n * PIXEL) ** 2
            du, dv, angle, shift = (ctf[a:b, i:i + 1].double() for i in range(4))
            k2 = kx * kx + ky * ky
            defocus = 0.5 * (du + dv) * k2 + 0.5 * (du - dv) * (
                torch.cos(2 * angle) * (kx * kx - ky * ky) + 2 * torch.sin(2 * angle) * kx * ky)
            chi = (math.pi * lam * scale * defocus - 0.5 * math.pi * OPTICS[1] * 1e7 * lam ** 3 * (scale * k2) ** 2
                   + shift + math.asin(OPTICS[2]))
            c = torch.sin(chi)
            value, weight = value * c, c * c
        elif case["variant"] == "weighted":
            weight = weights[a:b].double().reshape(b - a, -1)[:, inside]
        value, weight = value * r, weight * r
        position = (big / n) * (kx[None, :, None] * t[:, 0, None, :3] + ky[None, :, None] * t[:, 1, None, :3])
        for sign in (1.0, -1.0):
            # The mirrored copies of column 0 are its own other rows.
            keep = torch.ones_like(weight, dtype=torch.bool) if sign > 0 else (kx > 0).expand_as(weight)
            p = sign * position
            keep = keep & (p[..., 0] > -half_width)
            p, w = p[keep], weight[keep]
            v = value[keep] if sign > 0 else value[keep].conj()
            first = torch.floor(p) if window == "linear" else torch.floor(p - half_width) + 1
            terms = torch.stack([v.real, v.imag, w], dim=1)
            axis_weights = []
            for tap in range(taps):
                d = (first + tap - p).abs()
                axis_weights.append(1.0 - d if window == "linear" else _kaiser_bessel64(d, half_width, shape))
            first = first.to(torch.int64)
            for tz in range(taps):
                for ty in range(taps):
                    for tx in range(taps):
                        gx, gy, gz = first[:, 0] + tx, first[:, 1] + ty, first[:, 2] + tz
                        ok = (gx >= 0) & (gx <= half) & (gy.abs() <= half) & (gz.abs() <= half)
                        wt = torch.where(ok, axis_weights[tx][:, 0] * axis_weights[ty][:, 1] * axis_weights[tz][:, 2],
                                         torch.zeros_like(w))
                        index = torch.where(ok, ((gz % big) * big + gy % big) * (half + 1) + gx, 0)
                        out.index_add_(0, index, terms * wt[:, None])
    out = out.reshape(big, big, half + 1, 3)
    sums = torch.view_as_complex(out[..., :2].contiguous())
    sums = sums * phase[:, None, None] * phase[None, :, None] * phase[None, None, :half + 1]
    return num.to(torch.complex128) + sums, den.double() + out[..., 2]


def _padded_spectra64(images, scales, n):
    m = images.shape[-1]

    def spectra_of(a, b):
        x = images[a:b].double()
        if scales is not None:
            x = x * scales[a:b, None, None].double()
        if n != m:
            o = n // 2 - m // 2
            x = torch.nn.functional.pad(x, (o, n - m - o, o, n - m - o))
        return torch.fft.rfft(x, dim=-1) if n == 1 else torch.fft.fft(torch.fft.rfft(x, dim=-1), dim=-2)

    return spectra_of


def _philox_normal(key, counter):
    """The standard normal value of a counter of a key's Philox4x32-10 stream
    (Salmon et al., SC 2011), by Box-Muller; uint64 arrays."""
    low = np.uint64(0xFFFFFFFF)
    block = counter >> np.uint64(1)
    c = [block & low, block >> np.uint64(32), np.zeros_like(block), np.zeros_like(block)]
    k = [key & low, key >> np.uint64(32)]
    for i in range(10):
        if i:
            k = [(k[0] + np.uint64(0x9E3779B9)) & low, (k[1] + np.uint64(0xBB67AE85)) & low]
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ k[0], p1 & low, (p0 >> np.uint64(32)) ^ c[3] ^ k[1], p0 & low]
    u = [(((c[2 * j + 1] << np.uint64(32)) | c[2 * j]) >> np.uint64(11)).astype(np.float64) + 1.0 for j in range(2)]
    radius = np.sqrt(-2.0 * np.log(u[0] * 2.0 ** -53))
    angle = 2 * math.pi * u[1] * 2.0 ** -53
    return np.where(counter & np.uint64(1), radius * np.sin(angle), radius * np.cos(angle))


def _standardize64(images, key, n):
    x = images.double()
    r = torch.arange(n, device=x.device, dtype=torch.float64) - n // 2
    background = (r[:, None] ** 2 + r[None, :] ** 2 > (0.4 * n) ** 2)[None]
    valid = background & torch.isfinite(x)
    for _ in range(2):
        weight = valid.double()
        total = weight.sum(dim=(1, 2), keepdim=True)
        mean = (x * weight).sum(dim=(1, 2), keepdim=True) / total
        deviation = torch.sqrt(((x - mean) ** 2 * weight).sum(dim=(1, 2), keepdim=True) / total)
        out = (x - mean) / deviation
        valid = background & (out.abs() <= 6.0)
    out_of_bounds = (out.abs() > 6.0).reshape(-1).nonzero().squeeze(1).cpu().numpy()
    image, counter = np.divmod(out_of_bounds, n * n)
    keys = key.cpu().numpy().astype(np.uint64)[image]
    draws = torch.from_numpy(_philox_normal(keys, counter.astype(np.uint64))).to(out.device)
    out.view(-1)[torch.from_numpy(out_of_bounds).to(out.device)] = draws
    return out


def _full_spectrum(half_grid, big):
    """The full grid of a real Hermitian field stored on x <= N/2."""
    mirror = torch.roll(torch.flip(half_grid, (0, 1)), (1, 1), (0, 1))
    return torch.cat([half_grid, torch.flip(mirror[..., 1:big - big // 2], (2,))], dim=2)


def _iterative64(den):
    big = den.shape[0]
    d = _full_spectrum(den.double(), big)
    w = torch.ones_like(d)
    for _ in range(learned.PASSES):
        c = w * d
        for axis in range(3):
            c = c * (2.0 / 3.0) + (torch.roll(c, 1, axis) + torch.roll(c, -1, axis)) / 6.0
        w = torch.where(d > 0, w / torch.clamp(c, min=learned.FLOOR), torch.zeros_like(w))
    return w[..., :big // 2 + 1]


def _parameters64():
    """The shipped perceptron: the float16 weights it multiplies with, the float32 biases."""
    path = os.path.join(os.path.dirname(os.path.abspath(learned.__file__)), "compensation_model.npz")
    with np.load(path, allow_pickle=False) as f:
        flat = torch.from_numpy(np.asarray(f["parameters"], np.float32)).cuda()
    shapes = [(16, 64), (64, 64), (64, 64), (64, 16), (64,), (64,), (64,), (16,)]
    out, at = [], 0
    for shape in shapes:
        size = int(np.prod(shape))
        part = flat[at:at + size].reshape(shape)
        out.append((part.half() if len(shape) == 2 else part).double())
        at += size
    return out


def _perceptron64(x, p):
    for layer in range(3):
        x = torch.relu(x @ p[layer] + p[4 + layer])
    return x @ p[3][:, 0] + p[7][0]


def _learned64(den, table):
    big = den.shape[0]
    d = den.double()
    f = torch.fft.fftfreq(big, d=1.0 / big, device=d.device, dtype=torch.float64)
    x = torch.arange(big // 2 + 1, device=d.device, dtype=torch.float64)
    r = torch.sqrt(f[:, None, None] ** 2 + f[None, :, None] ** 2 + x[None, None, :] ** 2)
    z = f[:, None, None].expand_as(r)
    theta = torch.where(r > 0, torch.acos(torch.clamp(z / torch.clamp(r, min=1e-9), -1, 1)), torch.zeros_like(r))
    phi = torch.atan2(f[None, :, None].expand_as(r), x[None, None, :].expand_as(r)) % (2 * math.pi)
    bins = torch.clamp((8 * r / (big / 2)).to(torch.int64), max=7)
    entry = (bins * 33 + (theta * (32 / math.pi) + 0.5).to(torch.int64)) * 64 + (
        phi * (64 / (2 * math.pi)) + 0.5).to(torch.int64) % 64
    p = _parameters64()
    mean = d[d > 0].mean()
    correction = torch.empty_like(d)
    table = table.double().reshape(-1, 8)
    for a in range(big):
        rows = torch.zeros((r[a].numel(), 16), dtype=torch.float64, device=d.device)
        rows[:, 0] = r[a].reshape(-1) / (big / 2)
        rows[:, 1] = torch.log1p(d[a].reshape(-1) / mean)
        rows[:, 2:10] = table[entry[a].reshape(-1)]
        correction[a] = _perceptron64(rows, p).reshape(r[a].shape)
    correction = torch.where(r <= big // 2, correction, torch.zeros_like(r))
    return torch.where(d > 0, torch.exp(correction) / torch.where(d > 0, d, torch.ones_like(d)), torch.zeros_like(d))


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind == "slices":
        spectra_of = (_padded_spectra64(s["images"], None, case["n"]) if case["source"] == "images"
                      else lambda a, b: s["slices"][a:b].to(torch.complex128))
        return list(_insert64(s["num"], s["den"], spectra_of, case, case["n"], case["big"], s["transforms"], s["ctf"],
                              s["radial"], s.get("weights"), case["window"]))
    if kind == "images":
        n = case["padded"] or case["m"]
        s["num"].zero_()
        s["den"].zero_()
        return list(_insert64(s["num"], s["den"], _padded_spectra64(s["images"], s["scales"], n), case, n,
                              case["big"], s["transforms"], s["ctf"], s["radial"], None, case["window"]))
    if kind == "reconstruct":
        n = case["n"]
        images = s["reconstruction"].images
        num = torch.zeros((n, n, n // 2 + 1), dtype=torch.complex64, device="cuda")
        num, den = _insert64(num, num.real, _padded_spectra64(images, None, n), case, n, n, s["transforms"], s["ctf"],
                             torch.ones(n // 2 + 1, device="cuda"), None, "linear")
        quotient = torch.where(den > 1e-3, num / torch.where(den > 1e-3, den, 1.0), torch.zeros_like(num))
        lines = torch.fft.ifft(torch.fft.ifft(quotient, dim=0), dim=1)
        lines.imag[..., 0] = 0
        if n % 2 == 0:
            lines.imag[..., n // 2] = 0
        volume = torch.fft.irfft(lines, n=n, dim=2)
        u = (torch.arange(n, device="cuda", dtype=torch.float64) - n // 2) / n
        taper = torch.sinc(u) ** 2
        return [num, den, volume / (taper[:, None, None] * taper[None, :, None] * taper)]
    if kind == "standardize":
        return _standardize64(s["images"], s["key"], case["n"])
    if kind == "fourier":
        axes = (-3, -2, -1) if case["form"] == "volume" else (-2, -1)
        x = s["x"].cpu().numpy()
        if case["form"] == "real":
            return [np.fft.rfftn(x.astype(np.float64), axes=axes), x.astype(np.float64)]
        return [np.fft.fftn(x.astype(np.complex128), axes=axes), x.astype(np.complex128)]
    if kind == "compensation":
        return [_iterative64(s["den"]), _learned64(s["den"], s["table"])]
    p = [a.requires_grad_(True) for a in _parameters64()]
    loss = ((_perceptron64(s["rows"].double(), p) - s["target"].double()) ** 2).mean()
    loss.backward()
    return [torch.cat([a.grad.reshape(-1) for a in p]), loss.detach().reshape(1)]
