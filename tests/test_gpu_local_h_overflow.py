"""A line value that overflows stays the infinity that the division by the grid's
points makes of it (and is no NaN)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# few columns (one-wave workgroups) and many; a z axis whose register DFT exceeds 10
@pytest.mark.parametrize("shape,columns", [((32, 32, 32), 1), ((32, 32, 32), 700), ((8, 8, 96), 3), ((8, 8, 96), 700)])
@pytest.mark.parametrize("precision", [0, 1])
def test_overflow_of_the_last_sum(hip_ctx, shape, columns, precision):
    # one coefficient at G = 0 in a constant potential: every line is constant, every
    # difference zero and every partial sum a fraction of the last, which alone passes
    # the largest number by a tenth
    largest = float(np.finfo(np.float64 if precision == 0 else np.float32).max)
    indices = np.array([0, 1, shape[2] - 1], dtype=np.uint64)
    x = np.zeros((3, columns), dtype=np.complex128)
    count = int(np.prod(shape))
    x[0, ::2] = 1.1 * (largest / count)
    x[0, 1::2] = -1.1 * (largest / count)
    got = hip_ctx.local_hamiltonian(shape, indices, np.zeros(3), np.ones(count), x, precision=precision)
    infinite = np.isposinf(got[0, ::2].real).sum() + np.isneginf(got[0, 1::2].real).sum()
    assert infinite == columns and np.count_nonzero(got[0].imag) == 0
    # half of it is exact up to rounding
    half = hip_ctx.local_hamiltonian(shape, indices, np.zeros(3), np.ones(count), 0.5 * x, precision=precision)
    eps = 2.0 ** -53 if precision == 0 else 2.0 ** -24
    assert np.abs(half - 0.5 * x).max() <= 64 * eps * np.abs(x).max()
