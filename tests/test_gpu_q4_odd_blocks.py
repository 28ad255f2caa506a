"""GPU: Q4_0 GEMV on rows of an odd number of blocks (every other row starts in the middle of a pair of blocks): the
narrowest and widest rows of each split, matrices of one row up to several rounds, blocks beside a row that are not
numbers, guard bytes behind the last row."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("blocks", [1, 3, 7, 9, 23, 75, 127, 129, 255, 257, 385, 511])
@pytest.mark.parametrize("rows", [1, 2, 3, 31, 32, 33, 65, 9003])
def test_odd_block_counts(rows, blocks):
    from leviathan_amd import ops
    if rows > 1000 and blocks > 129:
        rows = 1501
    ctx = ops.Context(0)
    cols = 32 * blocks
    w = O.synth_q4_0(rows + blocks, rows * blocks, 0.02)
    x = O.normal(cols, blocks)
    y = torch.full((rows + 1,), -7.0, device="cuda")
    got = ctx.q4_0_gemv(dev(w), dev(x), cols, rows, y=y).cpu().numpy()
    assert got[rows] == -7.0
    assert O.max_rel_err(got[:rows], O.q4_0_matvec_f64(w, rows, cols, x)) < 1e-4
    if rows > 2:            # a row whose scales are not numbers makes its own output NaN and no other's
        bad = rows // 2
        w.reshape(rows, blocks, 18)[bad, :, 0:2] = np.frombuffer(np.float16(np.nan).tobytes(), np.uint8)
        again = ctx.q4_0_gemv(dev(w), dev(x), cols, rows, y=y).cpu().numpy()[:rows]
        assert np.isnan(again[bad]) and np.array_equal(np.delete(again, bad), np.delete(got[:rows], bad))
    ctx.close()
