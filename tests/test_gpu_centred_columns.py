"""Centring signs in the strided kernels whose threads hold 32 elements: odd and even numbers of butterflies a
pass, which decide whether a thread's elements alternate in sign."""
import numpy as np
import pytest
import torch

import oracle as O
from afft import Mode, centre as C
from conftest import tolerance

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.complex64, torch.complex128])
@pytest.mark.parametrize("shape", [(1080, 66), (3645, 9), (2430, 35), (5000, 16), (4050, 33), (16, 1080, 12)])
def test_centred_columns(gpu, dtype, shape):
    x = torch.from_numpy(O.normal(9, shape)).to(dtype).to(gpu)
    xr = x.cpu().numpy().astype(np.complex128)
    fftn = {2: O.fft2D, 3: O.fft3D}[len(shape)]
    tol = tolerance(dtype == torch.complex128, int(np.prod(shape)))
    for mode, omode in ((Mode.Forward, O.Mode.Forward), (Mode.Inverse, O.Mode.Inverse)):
        got = C.fft_centred(mode, x, pre="centre", post="centre").cpu().numpy()
        assert O.rel_l2(got, O.centre(fftn(omode, O.centre(xr)))) <= tol
