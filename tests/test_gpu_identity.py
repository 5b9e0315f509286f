"""Transforms over extents of 1: copies, of many elements to a workgroup."""
import pytest
import torch

import afft
from afft import Mode

pytestmark = pytest.mark.gpu


# one element; around a workgroup's tile (1536 Complex Float, 768 Complex Double); an odd large count
@pytest.mark.parametrize("count", [1, 767, 768, 769, 1535, 1536, 1537, (1 << 24) + 3])
@pytest.mark.parametrize("dtype", [torch.complex64, torch.complex128])
def test_extents_of_one(gpu, dtype, count):
    g = torch.Generator(device=gpu).manual_seed(count)
    x = torch.randn(count, 1, dtype=dtype, device=gpu, generator=g)
    for mode in Mode:
        assert torch.equal(afft.fft(mode, x), x)
    p = afft.Plan((count, 1), dtype)
    y = x.clone()
    p.execute(y, direction=+1, scale=0.5, out=y)  # in place, scaled by a power of two: exact
    assert torch.equal(y, 0.5 * x)
    p.close()
