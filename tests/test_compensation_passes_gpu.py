"""The density compensation's tiled passes and the predicted weights in one
pass, at extents that cut the tiles: even and odd N, rows shorter and longer
than a tile, a group of 64 voxels that ends a plane."""
import numpy as np
import pytest
import torch

import oracle
from rexlib_amd import learned

pytestmark = pytest.mark.gpu


def weight_volume(big, seed):
    """Positive densities with empty voxels, Hermitian where the stored half
    mirrors itself (x = 0, and x = N/2 of an even N)."""
    rng = np.random.default_rng(seed)
    full = rng.uniform(0.2, 4.0, (big, big, big)) * (rng.uniform(size=(big, big, big)) < 0.8)
    index = (-np.arange(big)) % big
    full = 0.5 * (full + full[np.ix_(index, index, index)])
    return full[..., :big // 2 + 1].astype(np.float32)


@pytest.mark.parametrize("big", [4, 9, 16, 33, 78, 82, 121])
@pytest.mark.parametrize("passes", [1, 2, 10])
def test_tiled_passes_match_the_oracle(big, passes):
    den = weight_volume(big, big)
    got = learned.iterative_weights(torch.from_numpy(den).cuda(), passes=passes).cpu().numpy()
    ref = oracle.density_compensation(den, passes=passes, floor=learned.FLOOR)
    # Ten divisions of float32 sums of 27 products: about 10 eps relative.
    assert oracle.rel_l2(got, ref) < 5e-6


# (At 49, 98 and 214 fftfreq's frequencies are not whole: the sphere's edge.)
@pytest.mark.parametrize("big", [6, 15, 32, 45, 49, 98, 214])
def test_predicted_weights_equal_features_then_perceptron(big):
    den = torch.from_numpy(weight_volume(big, 7 * big)).cuda()
    g = torch.Generator(device="cuda")
    g.manual_seed(big)
    table = torch.rand((8, 33, 64, 8), device="cuda", generator=g)
    model = learned.CompensationModel(seed=3)
    with torch.no_grad():
        model.f32[learned.parameter_count() - 16 - 3 * 64:] += 0.3
    correction = model.predict(learned.features(den, table).reshape(-1, learned.FEATURES)).reshape(den.shape)
    correction = torch.where(learned.inside_nyquist(big, den.device), correction, torch.zeros_like(correction))
    expected = torch.where(den > 0, torch.exp(correction.double()) / den.double(), torch.zeros_like(den).double())
    got = model.weights(den, table)
    # The same float16 features and perceptron; exp and the division in float32.
    assert oracle.rel_l2(got.cpu().numpy(), expected.cpu().numpy()) < 1e-6


def test_density_scale_is_the_reciprocal_mean_of_the_positive_weights():
    den = torch.from_numpy(weight_volume(33, 2)).cuda()
    den[0, 0, :5] = -1.0
    positive = den[den > 0].double()
    assert abs(learned.density_scale(den) * float(positive.mean()) - 1.0) < 1e-12
    assert learned.density_scale(torch.zeros((4, 4, 3), device="cuda")) == 1.0


# Index N/2 of an odd N is the frequency +N/2 (of an even N, -N/2).
@pytest.mark.parametrize("big", [15, 16, 33, 45])
def test_features_of_odd_and_even_extents_match_the_oracle(big):
    den = weight_volume(big, big)
    table = np.random.default_rng(big).uniform(size=(8, 33, 64, 8)).astype(np.float32)
    got = learned.features(torch.from_numpy(den).cuda(), torch.from_numpy(table).cuda(), 0.7).float().cpu().numpy()
    ref = oracle.compensation_features(den, table, 0.7)
    np.testing.assert_allclose(got[..., :2], ref[..., :2], rtol=2e-3, atol=2e-3)  # float16
    # (A direction within a float32 rounding of two grid directions may take either.)
    same = np.all(np.abs(got[..., 2:10] - ref[..., 2:]) <= 2e-3, axis=-1)
    assert same.mean() > 0.999


@pytest.mark.parametrize("big", [15, 16, 33])
def test_predicted_weights_of_a_plane_that_mirrors_itself(big):
    # A table that depends on the radius alone: (0, y, z) and (0, -y, -z) have
    # the same features, so the same weights, to the last bit.
    den = torch.from_numpy(weight_volume(big, 5)).cuda()
    table = torch.rand((8, 1, 1, 8), generator=torch.Generator().manual_seed(2)).expand(8, 33, 64, 8).contiguous().cuda()
    plane = learned.CompensationModel(seed=3).weights(den, table)[..., 0]
    index = (-torch.arange(big)) % big
    assert torch.equal(plane, plane[index][:, index])
