"""The local Hamiltonian's kernels over grids and spheres at the edges of their
launch rules, against numpy transforms in FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# ball: centred, empty in the middle of every axis; wide: a ball over most of the
# axis (no empty middle); shifted: lines that start off the origin (two runs from
# the ends of the axis no more); dense: every point
SPHERES = {
    "ball": lambda f: (np.abs(f) < 0.24).all(axis=1) & ((f * f).sum(axis=1) < 0.23 ** 2 * 1.5),
    "wide": lambda f: (f * f).sum(axis=1) < 0.46 ** 2,
    "shifted": lambda f: (np.abs(f - 0.2) < 0.15).all(axis=1),
    "dense": lambda f: np.ones(len(f), dtype=bool),
}


def _case(shape, sphere, columns, seed):
    rng = np.random.default_rng(seed)
    grids = np.stack(np.meshgrid(*[np.arange(s) for s in shape], indexing="ij"), axis=-1).reshape(-1, 3)
    signed = np.where(grids > np.array(shape) // 2, grids - np.array(shape), grids)
    keep = SPHERES[sphere](signed / np.array(shape))
    indices = rng.permutation(np.flatnonzero(keep)).astype(np.uint64)
    n = len(indices)
    x = rng.standard_normal((n, columns)) + 1j * rng.standard_normal((n, columns))
    kinetic, potential = rng.uniform(0, 5, n), rng.standard_normal(int(np.prod(shape)))
    out = kinetic[:, None] * x
    for c in range(columns):
        g = np.zeros(int(np.prod(shape)), dtype=np.complex128)
        g[indices] = x[:, c]
        r = np.fft.ifftn(g.reshape(shape)) * potential.reshape(shape)
        out[:, c] += np.fft.fftn(r).ravel()[indices]
    return indices, kinetic, potential, x, out


# 72 x 72 and 96 x 16: the benchmark plane and a register DFT above 10; 2 x 3 and
# 7 x 5: one digit; 100 x 20 / 20 x 100: long rows, long columns; 30 x 35, 63 x 70:
# remainders in the lines a wave takes
@pytest.mark.parametrize("shape", [(72, 72, 6), (96, 16, 8), (16, 96, 5), (2, 3, 4), (7, 5, 3), (100, 20, 4),
                                   (20, 100, 4), (30, 35, 27), (63, 70, 2)])
@pytest.mark.parametrize("sphere", sorted(SPHERES))
@pytest.mark.parametrize("precision", [0, 1])
def test_local_hamiltonian_grid_and_sphere(hip_ctx, shape, sphere, precision):
    indices, kinetic, potential, x, ref = _case(shape, sphere, 3, 11)
    if not len(indices):
        pytest.skip("no plane wave in this sphere")
    got = hip_ctx.local_hamiltonian(shape, indices, kinetic, potential, x, precision=precision)
    # rounding of six line transforms of at most 128 points: a few eps times
    # log2 of the grid, on the scale of the largest entry
    eps = 2.0 ** -53 if precision == 0 else 2.0 ** -24
    assert np.abs(got - ref).max() <= 64 * eps * np.abs(ref).max()


# 96 x 96: with every line touched, a plane and its waves' buffers pass the LDS of a
# workgroup in FP64 (98 rows of 97 and 4 x 480 values of 16 bytes: 183 kB) and the
# in-place kernel takes over
@pytest.mark.parametrize("sphere", sorted(SPHERES))
@pytest.mark.parametrize("precision", [0, 1])
def test_local_hamiltonian_plane_beyond_the_lds(hip_ctx, sphere, precision):
    indices, kinetic, potential, x, ref = _case((96, 96, 3), sphere, 2, 12)
    got = hip_ctx.local_hamiltonian((96, 96, 3), indices, kinetic, potential, x, precision=precision)
    eps = 2.0 ** -53 if precision == 0 else 2.0 ** -24
    assert np.abs(got - ref).max() <= 64 * eps * np.abs(ref).max()


# z-lines with a register DFT above 10 (5 x 15, 8 x 12, 9 x 14, 8 x 16), by one-wave
# workgroups and, from 512 of four waves on, by those
@pytest.mark.parametrize("shape", [(4, 5, 75), (12, 10, 96), (3, 4, 126), (6, 8, 128)])
@pytest.mark.parametrize("sphere", sorted(SPHERES))
@pytest.mark.parametrize("columns", [3, 400])
@pytest.mark.parametrize("precision", [0, 1])
def test_local_hamiltonian_long_lines(hip_ctx, shape, sphere, columns, precision):
    indices, kinetic, potential, x, ref = _case(shape, sphere, columns, 13)
    got = hip_ctx.local_hamiltonian(shape, indices, kinetic, potential, x, precision=precision)
    eps = 2.0 ** -53 if precision == 0 else 2.0 ** -24
    assert np.abs(got - ref).max() <= 64 * eps * np.abs(ref).max()
