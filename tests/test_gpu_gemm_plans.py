"""Every tile plan of the complex GEMM, at the edges of its tiles and splits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 64 x 64 tiles (wide, 1200 tiles or more) with and without ragged edges; 64 x 32
# tiles split along K (ragged last split, K remainder); 32 x 32 tiles at one
# element, one full tile and its neighbours; K of one slab, one more, one less
SHAPES = [(2400, 2048, 20), (2399, 2018, 33), (500, 150, 6001), (640, 96, 4096), (1, 1, 2), (32, 32, 16), (33, 31, 17),
          (31, 33, 15), (64, 33, 4000)]


def _operand(rng, rows, cols, ld):
    a = np.full((ld, cols), np.nan + 1j * np.nan, dtype=np.complex128, order="F")
    a[:rows] = rng.standard_normal((rows, cols)) + 1j * rng.standard_normal((rows, cols))
    return a


@pytest.mark.parametrize("mnk", SHAPES)
@pytest.mark.parametrize("ops", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("precision", [0, 1])
def test_plans(hip_ctx, mnk, ops, precision):
    m, n, k = mnk
    rng = np.random.default_rng(3)
    a = _operand(rng, *((m, k) if not ops[0] else (k, m)), ld=(m if not ops[0] else k) + 2)
    b = _operand(rng, *((k, n) if not ops[1] else (n, k)), ld=(k if not ops[1] else n) + 1)
    left = a[:m, :k] if not ops[0] else a[:k, :m].conj().T
    right = b[:k, :n] if not ops[1] else b[:n, :k].conj().T
    ref = left @ right
    c = np.zeros(m * n, dtype=np.complex128)
    hip_ctx.zgemm_strided(ops[0], ops[1], m, n, k, a.ravel(order="F"), a.shape[0], b.ravel(order="F"), b.shape[0], c, m,
                          precision=precision)
    # three real products of K terms: eps sqrt(K) times the operands' scale, with
    # room for the largest of the entries
    eps = 2.0 ** -53 if precision == 0 else 2.0 ** -24
    assert np.abs(c.reshape((m, n), order="F") - ref).max() <= 32 * eps * k ** 0.5 * np.log2(k + 1) + 32 * eps


@pytest.mark.parametrize("ops", [(0, 0), (1, 0)])
def test_far_leading_dimension(hip_ctx, ops):
    # a leading dimension past the reach of a tile's 32-bit offsets
    m, n, k, ld = 5, 3, 4, (1 << 20) + 3
    rng = np.random.default_rng(4)
    a = _operand(rng, *((m, k) if not ops[0] else (k, m)), ld=ld)
    b = _operand(rng, k, n, ld=ld)
    left = a[:m, :k] if not ops[0] else a[:k, :m].conj().T
    c = np.zeros(m * n, dtype=np.complex128)
    hip_ctx.zgemm_strided(ops[0], 0, m, n, k, a.ravel(order="F"), ld, b.ravel(order="F"), ld, c, m)
    assert np.abs(c.reshape((m, n), order="F") - left @ b[:k, :n]).max() <= 1e-13


# one operand past that reach: planned as 64 x 32 tiles in 46 splits whose last is ragged
# (then run as 32 x 32 with the same K ranges), with the other operand normal and
# adjoint; several tiles and slabs along the far operand's columns; an adjoint B
@pytest.mark.parametrize("far,ops,mnk", [("a", (1, 0), (5, 512, 12301)), ("a", (1, 1), (5, 512, 12301)),
                                         ("a", (0, 0), (70, 40, 17)), ("b", (0, 1), (40, 70, 17)),
                                         ("b", (1, 0), (70, 5, 6001))])
@pytest.mark.parametrize("precision", [0, 1])
def test_one_far_operand(hip_ctx, far, ops, mnk, precision):
    m, n, k = mnk
    rng = np.random.default_rng(5)
    shape_a, shape_b = (m, k) if not ops[0] else (k, m), (k, n) if not ops[1] else (n, k)
    a = _operand(rng, *shape_a, ld=(1 << 20) + 3 if far == "a" else shape_a[0])
    b = _operand(rng, *shape_b, ld=(1 << 20) + 5 if far == "b" else shape_b[0])
    left = a[:m, :k] if not ops[0] else a[:k, :m].conj().T
    right = b[:k, :n] if not ops[1] else b[:n, :k].conj().T
    c = np.zeros(m * n, dtype=np.complex128)
    hip_ctx.zgemm_strided(*ops, m, n, k, a.ravel(order="F"), a.shape[0], b.ravel(order="F"), b.shape[0], c, m,
                          precision=precision)
    eps = 2.0 ** -53 if precision == 0 else 2.0 ** -24
    assert np.abs(c.reshape((m, n), order="F") - left @ right).max() <= 32 * eps * k ** 0.5 * np.log2(k + 1) + 32 * eps
