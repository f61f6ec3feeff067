"""The onsite products of an application, bit for bit: the sum of the projection's
partial sums and the compensated products of it."""
import numpy as np
import pyoracle
import pytest

pytestmark = pytest.mark.gpu

ROWS = {"one": [1], "full": [64], "over": [65], "groups": [3, 5, 60, 1, 40], "si": [8] * 8}


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


def _sum(partials):
    """Quarters of the partials in order, then the four sums in order."""
    splits = len(partials)
    total = None
    for quarter in range(4):
        part = np.zeros_like(partials[0])
        for s in range(splits * quarter // 4, splits * (quarter + 1) // 4):
            part = part + partials[s]
        total = part if total is None else total + part
    return total


# one partial; fewer than the four quarters; quarters of one, of unequal and of many
# partials (four at a time and the rest)
@pytest.mark.parametrize("splits", [1, 2, 3, 4, 7, 16, 37, 64])
@pytest.mark.parametrize("rows", sorted(ROWS))
def test_products_of_partial_sums(hip_ctx, rows, splits):
    rng = np.random.default_rng(splits)
    draw = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)  # noqa: E731
    hermitian = lambda r: (lambda a: (a + a.conj().T) / 2)(draw(r, r))  # noqa: E731
    atoms = ROWS[rows]
    d, q = [hermitian(r) for r in atoms], [hermitian(r) for r in atoms]
    partials = draw(splits, sum(atoms), 5)
    p = _sum(partials)
    w = hip_ctx.onsite_partials(atoms, d, q, partials)
    whole = hip_ctx.onsite_blocks(atoms, d, q, p)
    assert np.array_equal(_bits(w), _bits(whole))
    o = 0
    for r, db, qb in zip(atoms, d, q):
        assert np.array_equal(_bits(w[o:o + r, :5]), _bits(pyoracle.compensated_product(0, db, p[o:o + r])))
        assert np.array_equal(_bits(w[o:o + r, 5:]), _bits(pyoracle.compensated_product(0, qb, p[o:o + r])))
        o += r


def test_atoms_beyond_the_kernel(hip_ctx):
    d = [np.eye(1025, dtype=np.complex128)]
    p = np.ones((1, 1025, 1), dtype=np.complex128)
    with pytest.raises(ValueError):
        hip_ctx.onsite_partials([1025], d, d, p)
    assert np.array_equal(hip_ctx.onsite_blocks([1025], d, d, p[0]), np.ones((1025, 2)))
