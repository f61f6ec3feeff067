"""A batch whose launch shape comes from the plan cache uses nothing of the batch
that was tuned: that one's operators may be gone and their memory reused."""
import numpy as np
import pytest

from sdft_amd import native
from sdft_amd import synthetic as syn

pytestmark = pytest.mark.gpu


def test_cached_plan_after_its_operators_are_gone(hip_ctx, si8):
    columns = 3
    x = syn.initial_psi(si8, columns, 0)

    def batch():
        ops = [native.Operator(hip_ctx, si8) for _ in range(2)]
        return ops, native.Batch(hip_ctx, ops, columns)

    ops, b = batch()
    b.apply([x, x])
    b.close()
    for op in ops:
        op.close()
    # blocks of many sizes take the freed memory and overwrite it
    taken = [native.DeviceBlock(rows, 1).upload(np.full((rows, 1), np.nan + 0j))
             for rows in (16, 32, 64, 256, 1024, 4096, 32768, 131072) for _ in range(8)]
    ops, b = batch()
    assert b.plan()["from_cache"]
    h, s = b.apply([x, x])
    ref_h, ref_s = ops[0].apply(x)
    # one rounding order against another: the tolerance of the batch's parity tests
    for got, ref in ((h, ref_h), (s, ref_s)):
        for block in got:
            assert np.abs(block - ref).max() <= 1e-12 * np.abs(ref).max()
    b.close()
    for op in ops:
        op.close()
    for block in taken:
        block.close()
