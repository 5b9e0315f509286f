"""Rounding errors of transforms against FP64 (Complex Float) and extended precision (Complex Double).

The bounds are the errors of kernels that read every twiddle, rounded once from FP64, from a table, as
measured with them on an MI355X (relative L2, normally distributed samples), and 5% for other samples."""
import numpy as np
import pytest
import scipy.fft
import torch

import afft
from afft import Mode

pytestmark = pytest.mark.gpu

CASES = [
    (torch.complex64, 16384, 32, 7.40e-8),
    (torch.complex64, 4096, 128, 8.69e-8),
    (torch.complex64, 519, 1009, 1.78e-7),
    (torch.complex64, 8, 120000, 1.53e-7),     # two strided passes
    (torch.complex128, 1, 262144, 2.89e-16),
    # chirp-z, whose tables hold angles that are no binary fractions of a turn
    (torch.complex128, 64, 1009, 5.04e-16),
    (torch.complex128, 83, 783, 4.59e-16),
    (torch.complex128, 19, 3428, 4.83e-16),
    # chirp-z with a choice of padded lengths
    (torch.complex64, 12787, 41, 1.31e-7),
    (torch.complex64, 495, 1059, 1.62e-7),
    (torch.complex64, 240, 2177, 1.71e-7),
    (torch.complex128, 79, 824, 4.71e-16),
    # rows through the split exchange
    (torch.complex128, 260, 8192, 2.36e-16),
    # two passes or three
    (torch.complex64, 1, 3732480, 1.79e-7),
]


def exact(x):
    """The forward transform of the last axis, in FP64 for complex64 and in extended precision for complex128."""
    if x.dtype == torch.complex64:
        return np.fft.fft(x.cpu().numpy().astype(np.complex128))
    return scipy.fft.fft(x.cpu().numpy().astype(np.clongdouble))


def error(y, want):
    d = y.cpu().numpy().astype(want.dtype) - want
    return float(np.sqrt((np.abs(d) ** 2).sum() / (np.abs(want) ** 2).sum()))


@pytest.mark.parametrize("dtype,rows,n,bound", CASES)
def test_rounding_errors(gpu, dtype, rows, n, bound):
    g = torch.Generator(device=gpu).manual_seed(n)
    x = torch.randn(rows, n, dtype=dtype, device=gpu, generator=g)
    assert error(afft.fft(Mode.Forward, x), exact(x)) <= 1.05 * bound
    if rows > 1:  # the items of ragged batches
        plan = afft.RaggedPlan([n] * rows, dtype)
        assert error(plan.execute(Mode.Forward, x.reshape(-1)).reshape(rows, n), exact(x)) <= 1.05 * bound
        plan.close()
