"""Application of H and S over atoms at the edges of the onsite kernel's groups."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one projector; a group of 64 rows exactly, one more, and several atoms whose sum
# passes 64; many small atoms; the largest atom of the kernel and one beyond it
ROWS = {"one": [1], "full": [64], "over": [65], "groups": [3, 5, 60, 1, 40], "many": [1] * 130, "largest": [1024, 2],
        "beyond": [3, 1025]}


def _problem(si8, rows):
    rng = np.random.default_rng(len(rows) + rows[0])
    draw = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    hermitian = lambda r: (lambda a: (a + a.conj().T) / (2 * r ** 0.5))(draw(r, r))
    return dataclasses.replace(si8, atom_rows=np.array(rows, dtype=np.int64),
                               amplitudes=[draw(r, si8.n) / si8.n ** 0.5 for r in rows],
                               d_blocks=[hermitian(r) for r in rows], q_blocks=[0.01 * hermitian(r) for r in rows])


@pytest.fixture(scope="module")
def local(si8):
    from sdft_amd import synthetic
    bare = dataclasses.replace(si8, atom_rows=np.array([1]), amplitudes=[np.zeros((1, si8.n), dtype=np.complex128)],
                               d_blocks=[np.eye(1)], q_blocks=[np.eye(1)])
    return synthetic.dense_operator(bare)[0]


# chunk 4: H in passes of 4 columns at most, S in one
@pytest.mark.parametrize("rows,chunk", [(r, None) for r in sorted(ROWS)] + [("groups", "4")])
def test_onsite_groups(hip_ctx, si8, local, rows, chunk, monkeypatch):
    from sdft_amd import native
    if chunk:
        monkeypatch.setenv("SDFT_HIP_APPLY_CHUNK", chunk)
    prob = _problem(si8, ROWS[rows])
    b, d, q = prob.all_b(), prob.block_d(), prob.block_q()
    op = native.Operator(hip_ctx, prob)
    for columns in (1, 21):
        rng = np.random.default_rng(columns)
        x = rng.standard_normal((prob.n, columns)) + 1j * rng.standard_normal((prob.n, columns))
        theta = rng.standard_normal(columns)
        want = dict(h=local @ x + b.conj().T @ (d @ (b @ x)),
                    s=(1 + prob.regularization) * x + b.conj().T @ (q @ (b @ x)))
        want["shifted"] = want["h"] - want["s"] * theta
        for precision in (0, 1):
            # chains of n terms in the projection and of the atom's rows twice over, by steps
            # that grow like a random walk
            tol = 8 * (2.0 ** -53 if precision == 0 else 2.0 ** -24) * prob.n ** 0.5
            near = lambda got, key: np.linalg.norm(got - want[key]) <= tol * np.linalg.norm(want[key])
            hy, sy = op.apply(x, precision=precision)
            assert near(hy, "h") and near(sy, "s"), (columns, precision)
            assert near(op.apply(x, which="h", precision=precision), "h"), (columns, precision)
            assert near(op.apply(x, which="s", precision=precision), "s"), (columns, precision)
            assert near(op.apply_shifted(x, theta, precision=precision), "shifted"), (columns, precision)
    op.close()
