"""A block longer than the sphere: what the library does not write is zero."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_local_hamiltonian_of_a_longer_column(hip_ctx):
    rng = np.random.default_rng(6)
    shape, n, more = (8, 8, 8), 40, 25000  # past what an allocator hands out cleared
    indices = rng.permutation(512)[:n].astype(np.uint64)
    kinetic, potential = rng.uniform(0, 5, n), rng.standard_normal(512)
    x = rng.standard_normal((n + more, 1)) + 1j * rng.standard_normal((n + more, 1))
    want = hip_ctx.local_hamiltonian(shape, indices, kinetic, potential, x[:n])
    for _ in range(20):
        junk = np.full(n + more, 7.0 + 7.0j)
        del junk
        got = hip_ctx.local_hamiltonian(shape, indices, kinetic, potential, x)
        assert np.array_equal(got[:n], want) and np.count_nonzero(got[n:]) == 0
