"""Host blocks of the accelerator calls at the edges of the transfer chunks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one element, a chunk of 1 MiB and its neighbours, all chunks of the ring in use, more than the ring
@pytest.mark.parametrize("npw,columns", [(1, 1), (65535, 1), (65536, 1), (65537, 1), (65536, 4), (65537, 4), (32771, 19)])
def test_pair_of_blocks(hip_ctx, npw, columns):
    rng = np.random.default_rng(npw + columns)
    draw = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    b, d, q = draw(2, npw) / npw ** 0.5, draw(2, 2), draw(2, 2)
    for call in range(3):  # the ring starts each call at another chunk
        x = draw(npw, columns)
        h, s = hip_ctx.paw_pair(7001, b, d, q, x, projector_identity=7001 * npw + columns)
        p = b @ x
        for got, block in ((h, d), (s, q)):
            want = b.conj().T @ (block @ p)
            # two products of at most npw terms each
            assert np.linalg.norm(got - want) <= 64 * 2.0 ** -53 * (npw + 1) ** 0.5 * np.linalg.norm(want), call
