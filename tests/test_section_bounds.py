"""The brick kernel's section bound (bound_section and bound_rows in
rexlib_amd/csrc/insertion.hip), restated in float32 numpy, against brute force
over random planes and bricks: every row that holds a sample whose first tap
lies in the brick is kept, for both copies of a slice, and few others are."""
import numpy as np
import pytest

f32 = np.float32
LARGE = f32(3.0e38)


def rotation(rng):
    q = rng.normal(size=4)
    a, b, c, d = q / np.linalg.norm(q)
    return np.array([[a * a + b * b - c * c - d * d, 2 * (b * c - a * d), 2 * (b * d + a * c)],
                     [2 * (b * c + a * d), a * a - b * b + c * c - d * d, 2 * (c * d - a * b)],
                     [2 * (b * d - a * c), 2 * (c * d + a * b), a * a - b * b - c * c + d * d]])


def narrowed(p, q, i, j, lower, upper, inv, bounds):
    p0, p1, q0, q1 = f32(p * lower[i]), f32(p * upper[i]), f32(q * lower[j]), f32(q * upper[j])
    l = f32(f32(min(p0, p1) - max(q0, q1)) * inv)
    u = f32(f32(max(p0, p1) - min(q0, q1)) * inv)
    return max(bounds[0], min(l, u)), min(bounds[1], max(l, u))


def section(xs, ys, lower, upper):
    kx = ky = (-LARGE, LARGE)
    for c in range(3):
        a, b = (c + 1) % 3, (c + 2) % 3
        normal = f32(f32(xs[a] * ys[b]) - f32(xs[b] * ys[a]))
        if abs(normal) > 1e-30:
            inv = f32(f32(1) / normal)
            ky = narrowed(xs[a], xs[b], b, a, lower, upper, inv, ky)
            kx = narrowed(ys[b], ys[a], a, b, lower, upper, inv, kx)
    return kx, ky


def rows(xs, ys, lower, upper, kx, ky, first, widest):
    k_low, k_high = np.ceil(max(kx[0], f32(first))), np.floor(min(kx[1], f32(widest)))
    low, high = max(ky[0], f32(-widest)), min(ky[1], f32(widest))
    if k_low > k_high:
        return 0, 0
    for a in range(3):
        at_first, at_last = f32(k_low * xs[a]), f32(k_high * xs[a])
        lo, hi = f32(lower[a] - max(at_first, at_last)), f32(upper[a] - min(at_first, at_last))
        if ys[a] == 0:
            if not lo <= 0 <= hi:
                return 0, 0
        else:
            l, u = f32(lo * f32(1 / ys[a])), f32(hi * f32(1 / ys[a]))
            low, high = max(low, min(l, u)), min(high, max(l, u))
    return (int(np.ceil(low)), int(np.floor(high)) + 1) if low <= high else (0, 0)


@pytest.mark.parametrize("scale", [1.0, 2.0, 0.7])
@pytest.mark.parametrize("axes", [False, True])
def test_every_row_with_a_sample_is_kept(scale, axes):
    rng = np.random.default_rng(11)
    n, widest, edge = 256, 127, 8
    kept = held = 0
    for case in range(300):
        r = rotation(rng)
        if axes:
            # Planes along the lattice's axes: zero steps and zero normals.
            r = np.eye(3)[rng.permutation(3)] * rng.choice([-1, 1], 3)[:, None]
        xs, ys = (scale * r[0]).astype(f32), (scale * r[1]).astype(f32)
        centre = rng.uniform(-100, 100, 2) @ (scale * r[:2]) + rng.uniform(-2, 2) * r[2]
        lo = np.floor(centre) - edge // 2
        lower, upper = (lo - 0.01).astype(f32), (lo + edge + 0.01).astype(f32)
        kx, ky = section(xs, ys, lower, upper)
        for mirrored in (False, True):
            if mirrored:
                r0, r1 = rows(xs, ys, -upper, -lower, (-kx[1], -kx[0]), (-ky[1], -ky[0]), 1, widest)
            else:
                r0, r1 = rows(xs, ys, lower, upper, kx, ky, 0, widest)
            k_y = np.arange(-widest, widest + 1)[:, None]
            k_x = np.arange(1 if mirrored else 0, widest + 1)[None, :]
            sign = f32(-1 if mirrored else 1)
            base = (k_y.astype(np.float64)[..., None] * (sign * ys.astype(np.float64))).astype(f32)
            position = base + (k_x.astype(f32)[..., None] * (sign * xs)).astype(f32)
            cell = np.floor(position)
            inside = np.all((cell >= lo) & (cell < lo + edge), axis=-1) & (k_x * k_x + k_y * k_y <= (n // 2) ** 2)
            found = np.unique(np.nonzero(inside)[0] - widest)
            assert np.all((found >= r0) & (found < r1)), (case, mirrored, found, r0, r1)
            kept += max(r1 - r0, 0)
            held += found.size
    # On generic planes at most one row in three holds no sample.
    assert held > 300 and (axes or kept < 1.5 * held)
