"""Insertions on either side of the density at which the bricks own voxels
rather than first-tap cells (sparse calls write each voxel once, input plus
sum), and the Kaiser-Bessel bricks whose lanes are the taps of one sample:
against the float64 oracle at volume extents that cut the bricks short, in
place and out of place, with strided and batched accumulators."""
import numpy as np
import pytest
import torch

import oracle
from cases import make_case
from gpu_helpers import OPTICS, hip_insert, hip_window, to_device
from rexlib_amd import em, tune

pytestmark = pytest.mark.gpu

# The reference's float32 bar (max-abs 1e-4 of accumulators of order one).
BAR = 1e-4


def geometry(inputs, rng):
    """Rotations with shifts in place of the fixture's random matrices."""
    from rexlib_amd import synthetic
    count = inputs[2].shape[0]
    inputs[3][...] = synthetic.transforms_of(synthetic.uniform_rotations(count, rng))
    inputs[3][:, :2, 3] = rng.uniform(-2, 2, (count, 2))
    return inputs


# 1.6 samples per voxel of the stored half divide the two: n = N = 16 with 5
# slices (0.4: bucket 8) and with 60 (3.1); N around 7 (voxels per brick), 8 and
# 14; odd and even. At N = 145 and 146 the inputs exceed the L2s: out of place, 60
# slices (0.06 samples per voxel) let the bricks copy them, 20 (0.02) do not.
@pytest.mark.parametrize("n,big,slices", [(16, 16, 5), (16, 16, 60), (6, 7, 2), (7, 13, 3), (8, 14, 3), (9, 15, 1),
                                          (12, 24, 9), (12, 29, 9), (20, 33, 4), (64, 145, 60), (64, 146, 60),
                                          (64, 146, 20)])
@pytest.mark.parametrize("in_place", [True, False])
def test_sparse_and_dense_insertions_match_the_oracle(n, big, slices, in_place):
    inputs = geometry(make_case("plain", n, big, seed=n + big, slices=slices), np.random.default_rng(big))
    ref = oracle.insert_f64("plain", inputs, oracle.Window.linear())
    num, den = hip_insert("plain", inputs, oracle.Window.linear(), in_place=in_place)
    scale = max(1.0, float(np.abs(ref[0]).max()))
    assert np.abs(num - ref[0]).max() <= BAR * scale
    assert np.abs(den - ref[1]).max() <= BAR * max(1.0, float(np.abs(ref[1]).max()))


# (Two volumes of 116^3 exceed the L2s: the bricks copy the inputs.)
@pytest.mark.parametrize("n,big,slices", [(10, 20, 3), (64, 116, 30)])
def test_sparse_insertion_into_strided_batched_accumulators(n, big, slices):
    kept = 2
    rng = np.random.default_rng(4)
    inputs = make_case("plain", n, big, seed=9, slices=slices, accumulator_batch=(kept, 1))
    inputs = geometry(inputs, rng)
    inputs[2] = rng.uniform(-1, 1, (kept, slices, n, n // 2 + 1)) + 0j
    ref = oracle.insert_f64("plain", inputs, oracle.Window.linear())
    t = [to_device(a) for a in inputs]
    # The accumulators transposed in memory, the outputs padded along x.
    num = t[0].transpose(-3, -2).contiguous().transpose(-3, -2)
    den = t[1].transpose(-3, -2).contiguous().transpose(-3, -2)
    num_out = torch.full((kept, 1, big, big, big // 2 + 4), 7.0, dtype=torch.complex64, device="cuda")
    den_out = torch.full((kept, 1, big, big, big // 2 + 4), 7.0, device="cuda")
    em.insert_slices(num, den, t[2], t[3], t[4], em.GriddingWindow.linear(),
                     numerator_out=num_out[..., :big // 2 + 1], denominator_out=den_out[..., :big // 2 + 1])
    torch.cuda.synchronize()
    assert np.abs(num_out[..., :big // 2 + 1].cpu().numpy() - ref[0]).max() <= BAR
    assert np.abs(den_out[..., :big // 2 + 1].cpu().numpy() - ref[1]).max() <= BAR
    assert bool((num_out[..., big // 2 + 1:] == 7.0).all()) and bool((den_out[..., big // 2 + 1:] == 7.0).all())
    assert np.array_equal(num.cpu().numpy(), inputs[0].astype(np.complex64))


# 3 and 4 taps, one sample per wavefront step; more samples than a wavefront.
@pytest.mark.parametrize("half_width,shape", [(1.2, 4.0), (1.5, 6.0), (2.0, 9.0)])
@pytest.mark.parametrize("n,big,slices", [(5, 9, 1), (12, 16, 7), (24, 37, 20)])
def test_kaiser_bessel_bricks_match_the_oracle(half_width, shape, n, big, slices):
    window = oracle.Window.kaiser_bessel(half_width, shape)
    inputs = geometry(make_case("plain", n, big, seed=3 * n, slices=slices), np.random.default_rng(n))
    ref = oracle.insert_f64("plain", inputs, window)
    num, den = hip_insert("plain", inputs, window)
    # The reference's bar for this window (5e-4: its table and its edge).
    assert np.abs(num - ref[0]).max() <= 5e-4 * max(1.0, float(np.abs(ref[0]).max()))
    assert np.abs(den - ref[1]).max() <= 5e-4 * max(1.0, float(np.abs(ref[1]).max()))


# 2 taps (half-width 1), 3 (1.2, 1.5) and 4 of the layout's 4.
@pytest.mark.parametrize("half_width", [1.0, 1.2, 1.5, 2.0])
@pytest.mark.parametrize("big", [16, 17])
def test_an_infinite_sample_stays_within_its_kaiser_bessel_window(half_width, big):
    n = 8
    taps = int(np.ceil(2 * half_width))
    inputs = make_case("plain", n, big, seed=1, slices=1, zero_accumulators=True)
    inputs[2][...] = 0.0
    inputs[2][0, 1, 2] = np.inf  # k = (2, 1)
    inputs[3][...] = [[[0.9, 0.1, 0.0, 0.0], [-0.1, 0.8, 0.3, 0.0], [0.0, 0.0, 1.0, 0.0]]]
    inputs[4][...] = 1.0
    position = (big / n) * (2 * inputs[3][0, 0, :3] + inputs[3][0, 1, :3])
    reach = [{int(f) % big for f in np.floor(c - half_width) + 1 + np.arange(taps)} for c in position]
    num, _ = hip_insert("plain", inputs, oracle.Window.kaiser_bessel(half_width, 6.0))
    spoilt = np.argwhere(~np.isfinite(num))
    assert len(spoilt) > 0
    for z, y, x in spoilt:
        assert x in reach[0] and y in reach[1] and z in reach[2]


# The rounds of a Kaiser-Bessel brick: claimed (3 taps in every brick shape; 4
# taps, sparse into 200^3 and more), one sample at a time (4 taps; 3 into twice
# the slices' extent).
@pytest.mark.parametrize("half_width,n,big,slices", [(1.5, 24, 37, 20), (1.0, 20, 40, 12), (1.2, 16, 32, 9),
                                                     (1.5, 17, 35, 9), (2.0, 100, 200, 13), (2.0, 100, 201, 13)])
def test_kaiser_bessel_rounds_match_the_oracle(half_width, n, big, slices):
    # (The same positions: the window steps at its edge, by 1 / I0(6) = 0.015 of a sample.)
    window = oracle.Window.kaiser_bessel(half_width, 6.0)
    inputs = geometry(make_case("plain", n, big, seed=n, slices=slices), np.random.default_rng(n))
    inputs = [a.astype(np.complex64 if np.iscomplexobj(a) else np.float32) for a in inputs]
    ref = oracle.insert_f64("plain", inputs, window, float32_positions=True)
    shapes = tune.SHAPES if big < 40 else (None,)
    tune.clear_tuning()
    try:
        for shape in shapes:
            if shape is not None:
                tune.set_tuning(big, shape, 64)
            num, den = hip_insert("plain", inputs, window)
            assert np.abs(num - ref[0]).max() <= 5e-4 * max(1.0, float(np.abs(ref[0]).max())), shape
            assert np.abs(den - ref[1]).max() <= 5e-4 * max(1.0, float(np.abs(ref[1]).max())), shape
    finally:
        tune.clear_tuning()
