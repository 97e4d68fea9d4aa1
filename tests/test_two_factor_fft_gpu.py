"""Transforms whose lengths are two register factors: the shortest and longest
of each register class, equal and unequal factors, primes 7, 11 and 13, odd
lengths, fewer lines than a block takes and one more, contiguous and strided
lines, in place and out of place; against numpy.fft (float64). float32 DFTs of
n points round at a few eps sqrt(log2 n), so 2e-6 relative L2 holds them."""
import numpy as np
import pytest
import torch

import rexlib_amd
from rexlib_amd import fourier

pytestmark = pytest.mark.gpu

BAR = 2e-6
# 48 = 6 x 8, 49 = 7 x 7, 256 = 16 x 16 | 144.., 162 = 9 x 18, 441 = 21 x 21,
# 484 = 22 x 22 | 240.., 250 = 10 x 25, 729 = 27 x 27, 1024 = 32 x 32; 47, 125 and
# 243 are taken by the other kernels.
LENGTHS = [47, 48, 49, 64, 65, 99, 121, 125, 143, 162, 169, 200, 225, 243, 250, 256, 260, 286, 300, 320, 441, 484, 512,
           529, 625, 676, 729, 1024]


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("count", [1, 17])
def test_complex_lines_match_numpy(n, count):
    g = torch.Generator().manual_seed(n + count)
    x = torch.randn((count, n, 3), dtype=torch.complex64, generator=g)
    for axis, operand in ((1, x), (2, x.transpose(1, 2).contiguous())):
        device = operand.cuda()
        ref = np.fft.fft(operand.numpy().astype(np.complex128), axis=axis)
        assert rel(fourier.fftn(device, axes=(axis,)).cpu().numpy(), ref) <= BAR
        inverse = np.fft.ifft(operand.numpy().astype(np.complex128), axis=axis)
        assert rel(fourier.ifftn(device, axes=(axis,), out=device).cpu().numpy(), inverse) <= BAR


@pytest.mark.parametrize("n", [48, 54, 72, 75, 90, 150, 162, 200, 225, 250, 256, 270, 300, 320, 384, 486, 512])
def test_real_images_match_numpy(n):
    # Rows loaded 4, 2 and 1 elements at a time: n of every remainder, and a
    # view whose rows start at odd elements.
    g = torch.Generator().manual_seed(n)
    x = torch.randn((3, n, n + 1), generator=g)
    for operand in (x[..., :n].contiguous(), x[..., 1:]):
        device = operand.cuda() if operand.is_contiguous() else x.cuda()[..., 1:]
        ref = np.fft.rfft2(operand.numpy().astype(np.float64))
        spectra = rexlib_amd.rfft2(device)
        assert rel(spectra.cpu().numpy(), ref) <= BAR
        back = rexlib_amd.irfft2(spectra)
        assert rel(back.cpu().numpy(), operand.numpy().astype(np.float64)) <= BAR


def test_lengths_of_other_primes_stay_refused():
    images = torch.zeros((1, 252, 252), device="cuda")
    with pytest.raises(rexlib_amd.UnsupportedOperationError):
        rexlib_amd.rfft2(images)
    with pytest.raises(rexlib_amd.UnsupportedOperationError):
        rexlib_amd.irfft2(torch.zeros((1, 252, 127), dtype=torch.complex64, device="cuda"))
