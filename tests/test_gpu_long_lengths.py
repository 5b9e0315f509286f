"""Lengths beyond one workgroup whose most balanced factors have no kernel: less balanced ones, or
chirp-z."""
import pytest
import torch

import afft
import oracle as O
from afft import Mode
from conftest import tolerance

pytestmark = pytest.mark.gpu


# 2 * 13^6 (no Complex Double tile of 4394), 11^7 (no two factors), and a longer Complex Float one
@pytest.mark.parametrize("dtype,n", [(torch.complex128, 9653618), (torch.complex128, 19487171),
                                     (torch.complex64, 33587736)])
def test_long_lengths(gpu, dtype, n):
    g = torch.Generator(device=gpu).manual_seed(n)
    x = torch.randn(n, dtype=dtype, device=gpu, generator=g)
    xr = x.cpu().numpy()
    tol = tolerance(dtype == torch.complex128, n)
    y = afft.fft1D(Mode.Forward, x)
    assert O.rel_l2(y.cpu().numpy(), O.fft1D(O.Mode.Forward, xr)) <= tol
    z = afft.fft1D(Mode.Inverse, y)
    assert O.rel_l2(z.cpu().numpy(), xr) <= 2 * tol  # two transforms
