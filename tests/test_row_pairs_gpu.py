"""Real transforms share a complex line only between rows of one transform: a
row beside a row of another transform that is a million times larger, or not
finite, comes out as if it were alone. Lengths of every row kernel: radix
stages (30, 2048), 256 points, two factors (64, 75, 252), chirp-z in one kernel (101)
and through memory (521); odd numbers of rows. Each row or image is compared
against numpy (float64) on its own scale; float32 DFTs round at a few eps
sqrt(log2 n), so 2e-6 relative L2 holds them (a shared line leaves 5e-2)."""
import numpy as np
import pytest
import torch

import rexlib_amd
from gpu_helpers import OPTICS
from rexlib_amd import em, fourier

pytestmark = pytest.mark.gpu

BAR = 2e-6


def uneven(shape, kept, seed):
    """Normal values; each element of the first `kept` axes (one transform) has
    a scale of its own, 1 and 1e6 in turn."""
    x = np.random.default_rng(seed).normal(size=shape)
    turns = np.arange(int(np.prod(shape[:kept]))).reshape(shape[:kept] + (1,) * (len(shape) - kept))
    return (x * np.where(turns % 2, 1e6, 1.0)).astype(np.float32)


def worst(got, want, kept):
    got = got.reshape((-1,) + got.shape[kept:])
    want = want.reshape((-1,) + want.shape[kept:])
    return max(float(np.linalg.norm(g - w) / np.linalg.norm(w)) for g, w in zip(got, want))


# One transform per row; per image (odd numbers of rows, so that pairs would
# cross images); the row axis not next to a transformed one (moved to the back
# for the comparison).
@pytest.mark.parametrize("n", [30, 64, 75, 101, 252, 256, 521, 2048])
@pytest.mark.parametrize("shape,kept,axes", [((5,), 1, (-1,)), ((4, 7), 1, (-2, -1)), ((3, 1, 5), 2, (-2, -1)),
                                             ((4, 1), 1, (-2, -1))])
def test_rows_of_other_transforms_leave_no_trace(n, shape, kept, axes):
    x = uneven(shape + (n,), kept, n)
    full = x.astype(np.float64)
    spectra = fourier.rfftn(torch.from_numpy(x).cuda(), axes=axes)
    assert worst(spectra.cpu().numpy(), np.fft.rfftn(full, axes=axes), kept) <= BAR
    sizes = [x.shape[a] for a in axes]
    back = fourier.irfftn(spectra, s=sizes, axes=axes)
    assert worst(back.cpu().numpy(), full, kept) <= 2 * BAR  # there and back
    # A transform that is not finite leaves the others as they are, bit for bit.
    x.reshape((-1,) + x.shape[kept:])[1, ..., 3] = np.inf
    again = fourier.rfftn(torch.from_numpy(x).cuda(), axes=axes)
    others = [i for i in range(int(np.prod(shape[:kept]))) if i != 1]
    assert torch.equal(again.reshape((-1,) + again.shape[kept:])[others],
                       spectra.reshape((-1,) + spectra.shape[kept:])[others])
    again = fourier.irfftn(again, s=sizes, axes=axes)
    assert torch.equal(again.reshape((-1,) + again.shape[kept:])[others],
                       back.reshape((-1,) + back.shape[kept:])[others])


@pytest.mark.parametrize("n", [60, 252])
def test_a_batch_axis_between_the_transformed_ones(n):
    x = np.random.default_rng(n).normal(size=(4, 3, n))
    x = (x * np.array([1.0, 1e6, 1.0])[None, :, None]).astype(np.float32)
    full = x.astype(np.float64)
    spectra = fourier.rfftn(torch.from_numpy(x).cuda(), axes=(0, 2))
    assert worst(np.moveaxis(spectra.cpu().numpy(), 1, 0), np.moveaxis(np.fft.rfftn(full, axes=(0, 2)), 1, 0), 1) <= BAR
    back = fourier.irfftn(spectra, s=(4, n), axes=(0, 2))
    assert worst(np.moveaxis(back.cpu().numpy(), 1, 0), np.moveaxis(full, 1, 0), 1) <= 2 * BAR


@pytest.mark.parametrize("n", [27, 75, 225])
def test_image_stacks_of_odd_extents(n):
    x = uneven((4, n, n), 1, n)
    full = x.astype(np.float64)
    spectra = rexlib_amd.rfft2(torch.from_numpy(x).cuda())
    assert worst(spectra.cpu().numpy(), np.fft.rfft2(full), 1) <= BAR
    assert worst(rexlib_amd.irfft2(spectra).cpu().numpy(), full, 1) <= 2 * BAR


def test_volumes_of_odd_extents():
    n = 27
    x = uneven((3, n, n, n), 1, n)
    spectra = np.fft.rfftn(x.astype(np.float64), axes=(1, 2, 3))
    back = rexlib_amd.irfft3(torch.from_numpy(spectra.astype(np.complex64)).cuda())
    assert worst(back.cpu().numpy(), x.astype(np.float64), 1) <= BAR


# Odd images on odd and even grids, through every row kernel of the insertion.
@pytest.mark.parametrize("m,n", [(45, 90), (27, 27), (45, 75), (135, 256), (75, 75), (25, 30)])
@pytest.mark.parametrize("schedule", ["brick", "scatter"])
def test_an_image_of_one_volume_stays_out_of_another(m, n, schedule, monkeypatch):
    monkeypatch.setenv("REXLIB_HIP_INSERTION_SCHEDULE", schedule)
    g = torch.Generator().manual_seed(m)
    images = torch.randn((2, m, m), generator=g)
    transforms = torch.eye(3, 4).expand(2, 3, 4).contiguous().cuda()
    ctf = torch.tensor([[15000.0, 14000.0, 0.3, 0.0]]).expand(2, 4).contiguous().cuda()
    radial = torch.ones(n // 2 + 1, device="cuda")

    def insert(stack):
        num = torch.zeros((2, n, n, n // 2 + 1), dtype=torch.complex64, device="cuda")
        den = torch.zeros((2, n, n, n // 2 + 1), device="cuda")
        em.insert_ctf_images(num, den, stack.cuda(), transforms, ctf, radial, em.GriddingWindow.linear(), OPTICS, 1.5,
                             padded=0 if n == m else n)
        return num

    clean = insert(images)
    images[0, -1, 2] = float("nan")  # the last row, which a pair across images would share
    spoilt = insert(images)
    assert bool(torch.isfinite(torch.view_as_real(spoilt[1])).all())
    error = torch.linalg.vector_norm(spoilt[1] - clean[1]) / torch.linalg.vector_norm(clean[1])
    assert float(error) <= 1e-6  # sums in another order
    assert not bool(torch.isfinite(torch.view_as_real(spoilt[0])).all())
