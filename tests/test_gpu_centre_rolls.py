"""Rolls before and after a transform of even extents, both folded into signs: the roll of the output
moves the sign that stands for the roll of the input, which leaves a factor of -1 where the extents'
halves add up to an odd number."""
import itertools

import numpy as np
import pytest
import torch

import oracle as O
from afft import Mode, centre as C
from conftest import tolerance

pytestmark = pytest.mark.gpu

OPS = {None: lambda a: a, "centre": O.centre, "shift": O.shift, "ishift": O.ishift}


@pytest.mark.parametrize("dtype", [torch.complex64, torch.complex128])
@pytest.mark.parametrize("shape", [(2,), (6,), (8,), (4098,), (10, 4), (6, 10), (36, 6), (6, 6, 10), (4, 6, 2)])
def test_rolls_on_both_sides(gpu, dtype, shape):
    x = torch.from_numpy(O.normal(9, shape)).to(dtype).to(gpu)
    xr = x.cpu().numpy().astype(np.complex128)
    fftn = {1: O.fft1D, 2: O.fft2D, 3: O.fft3D}[len(shape)]
    tol = tolerance(dtype == torch.complex128, int(np.prod(shape)))
    for pre, post in itertools.product(OPS, OPS):
        for mode, omode in ((Mode.Forward, O.Mode.Forward), (Mode.Inverse, O.Mode.Inverse)):
            want = OPS[post](fftn(omode, OPS[pre](xr)))
            got = C.fft_centred(mode, x, pre=pre, post=post).cpu().numpy()
            assert O.rel_l2(got, want) <= tol, f"pre={pre} post={post} {mode}"
