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
# Chirp-z lengths: convolutions of 48 points (the shortest) to 1,024 in one
# kernel, and one (521) whose steps pass through memory.
CHIRP_LENGTHS = [7, 17, 37, 101, 127, 251, 383, 509, 511, 521]


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("n", LENGTHS + CHIRP_LENGTHS)
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


# Even, odd and prime halved axes; a strided and a batched other axis; an odd
# number of rows (one left without a partner); every normalisation.
@pytest.mark.parametrize("shape,axes", [((3, 7, 64), (-1,)), ((5, 252, 60), (-2, -1)), ((1, 101, 127), (-2, -1)),
                                        ((3, 50, 251), (0, 2)), ((9, 256, 256), (-2, -1)), ((48, 49, 54), (0, 1, 2)),
                                        ((2, 33, 521), (-2, -1)), ((60, 5, 48), (2, 0)), ((6, 70, 5), (0, 1))])
@pytest.mark.parametrize("norm", ["backward", "ortho", "forward"])
def test_real_transforms_over_any_axes_match_numpy(shape, axes, norm):
    g = torch.Generator().manual_seed(sum(shape))
    x = torch.randn(shape, generator=g)
    ref = np.fft.rfftn(x.numpy().astype(np.float64), axes=axes, norm=norm)
    spectra = fourier.rfftn(x.cuda(), axes=axes, norm=norm)
    assert rel(spectra.cpu().numpy(), ref) <= BAR
    sizes = [shape[a] for a in axes]
    # Imaginary parts of self-conjugate coefficients do not count.
    noisy = ref + 1j * 0.1 * np.abs(ref).max()
    expected = np.fft.irfft(
        np.fft.ifftn(noisy, axes=axes[:-1], norm=norm) if len(axes) > 1 else noisy, n=sizes[-1], axis=axes[-1], norm=norm)
    got = fourier.irfftn(torch.from_numpy(noisy.astype(np.complex64)).cuda(), s=sizes, axes=axes, norm=norm)
    assert rel(got.cpu().numpy(), expected) <= BAR


def test_overlapping_real_operands_take_the_general_path():
    # The output starts inside the input's memory.
    n, count = 60, 7
    buffer = torch.zeros(count * n + 2 * count * (n // 2 + 1), device="cuda")
    x = torch.randn((count, n), generator=torch.Generator().manual_seed(1))
    buffer[:count * n] = x.reshape(-1).cuda()
    out = torch.view_as_complex(buffer[count * n // 2:count * n // 2 + 2 * count * (n // 2 + 1)].view(-1, 2))
    fourier.rfftn(buffer[:count * n].view(count, n), axes=(-1,), out=out.view(count, n // 2 + 1))
    assert rel(out.view(count, -1).cpu().numpy(), np.fft.rfft(x.numpy().astype(np.float64))) <= BAR


def test_lengths_of_other_primes_stay_refused():
    images = torch.zeros((1, 252, 252), device="cuda")
    with pytest.raises(rexlib_amd.UnsupportedOperationError):
        rexlib_amd.rfft2(images)
    with pytest.raises(rexlib_amd.UnsupportedOperationError):
        rexlib_amd.irfft2(torch.zeros((1, 252, 127), dtype=torch.complex64, device="cuda"))
