"""GPU: Q4_K GEMV of three to eight columns on rows of more than sixteen superblocks, cut into slices that meet in
scratch: the narrowest and widest of two, three and four slices, part of a row group up to many of them a workgroup, the
norm in front, a column that is not a number; repeated calls give the same bits."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("blocks", [17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("rows,ncol", [(1, 3), (15, 8), (17, 5), (1000, 4), (4113, 8), (9001, 3)])
def test_q4k_sliced_rows(rows, ncol, blocks):
    from leviathan_amd import ops
    if rows > 2000 and blocks not in (17, 33):
        rows = 1300
    ctx = ops.Context(0)
    cols = 256 * blocks
    w = O.synth_q4_k(blocks + rows, rows * blocks, 0.01)
    x = O.normal(ncol * cols, ncol).reshape(ncol, cols)
    gain = O.normal(cols, 9, 1.0, 0.1) if blocks % 2 else None
    x[-1, cols - 1] = np.inf if rows == 17 else x[-1, cols - 1]
    y = torch.full((ncol, rows), -7.0, device="cuda")
    dw, dx, dg = dev(w), dev(x), dev(gain) if gain is not None else None
    got = ctx.q4_k_gemv_ncol(dw, dx, cols, rows, ncol, gain=dg, y=y).cpu().numpy()
    for c in range(ncol):
        if not np.isfinite(x[c]).all():
            assert np.isnan(got[c]).all()
            continue
        xc = O.rmsnorm(x[c], gain, 1e-6) if gain is not None else x[c]
        assert O.max_rel_err(got[c], O.q4_k_matvec_f64(w, rows, cols, xc)) < 1e-4, (rows, ncol, blocks, c)
    for _ in range(3):
        again = ctx.q4_k_gemv_ncol(dw, dx, cols, rows, ncol, gain=dg).cpu().numpy()
        assert np.array_equal(again.view(np.uint32), got.view(np.uint32))
    ctx.close()
