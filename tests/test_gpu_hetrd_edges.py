"""The one-launch tridiagonalisation at the edges of its launch rules."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(n, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    return (a + a.conj().T) / 2


# one, two and four entries a thread (512, 1024), one and two rows a workgroup (72,
# 73), rows limited by the LDS (1025); after the largest, smaller ones reuse its buffers
@pytest.mark.parametrize("n", [1025, 2, 3, 72, 73, 144, 145, 511, 512, 513, 1023, 1024, 5])
def test_orders(hip_ctx, n):
    a = _matrix(n, n)
    k = min(n, 40)
    w, v, fused = hip_ctx.hermitian_eigen(a, k)
    assert fused == 1
    scale = max(1.0, np.abs(a).max())
    # backward error of a Householder reduction: eps sqrt(n) |A| with room; |A|_2 of a
    # random matrix is about 2 sqrt(n) times its entries
    bound = 1e-13 * scale * n
    assert np.abs(w - np.linalg.eigvalsh(a)).max() <= bound
    assert np.abs(a @ v - v * w[:k]).max() <= 10 * bound
    assert np.abs(v.conj().T @ v - np.eye(k)).max() <= 1e-11

