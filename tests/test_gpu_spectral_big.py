"""Spectral convolutions of images of 4 GiB, which the column kernels address by groups of rows."""
import pytest
import torch

import afft
from afft import Mode

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(torch.linalg.vector_norm(a - b) / torch.linalg.vector_norm(b))


@pytest.mark.parametrize("dtype,h,w,tol", [(torch.complex64, 32, 1 << 24, 3e-5), (torch.complex128, 16, 1 << 24, 1e-12)])
def test_images_of_4_gib(gpu, dtype, h, w, tol):
    real = torch.float32 if dtype == torch.complex64 else torch.float64
    g = torch.Generator(device=gpu).manual_seed(3)
    x = torch.randn(1, h, w, dtype=dtype, device=gpu, generator=g)
    # a filter of unit phases: the convolution moves the image by (5, 12345)
    k = torch.arange(h, device=gpu, dtype=torch.float64)[:, None] * (5 / h)
    l = (torch.arange(w, device=gpu, dtype=torch.int64) * 12345 % w).to(torch.float64)[None, :] / w
    turns = torch.frac(k + l)
    H = torch.polar(torch.ones((), dtype=real, device=gpu).expand(h, w), (turns * (-2 * torch.pi)).to(real)).to(dtype).contiguous()
    del k, l, turns
    # Complex Float: about 3e-7 each for two transforms, the filter and its angles; 100 times that is
    # still below any misplaced row or column (1 or more)
    y, spec = afft.spectral_conv(x, H, save_spectrum=True)
    assert rel(y, torch.roll(x, (5, 12345), (1, 2))) <= tol
    assert rel(spec, afft.fft2D(Mode.Forward, x[0])[None]) <= tol
    # the adjoint moves it back, and the filter's gradient is conj(F x) F g / (h w)
    gx, gH = afft.spectral_conv_vjp(None, H, y, spectrum=spec)
    assert rel(gx, x) <= tol
    assert rel(gH, spec[0].conj() * afft.fft2D(Mode.Forward, y[0]) / (h * w)) <= tol
    del gx, gH
    gx, gH = afft.spectral_conv_vjp(x, H, y)  # with the spectrum of x formed again
    assert rel(gx, x) <= tol
    assert rel(gH, spec[0].conj() * afft.fft2D(Mode.Forward, y[0]) / (h * w)) <= tol
