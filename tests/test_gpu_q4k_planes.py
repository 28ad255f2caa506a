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


@pytest.mark.parametrize("blocks,rows,ncol", [(17, 700, 5), (33, 300, 3), (47, 1000, 8), (64, 50, 6)])
def test_q4_k_wide_columns_record_the_eager_values(blocks, rows, ncol):
    """Recorded on a context without scratch, where the planes have no room, a row too wide to be staged by fours is
    taken by ones and twos.  Both ways a sum is exact but for the order of f64 additions in front of its one rounding to
    f32 (2^-53 against 2^-24: the same bits for all but one value in 10^8)."""
    from leviathan_amd import ops
    cols = 256 * blocks
    w = dev(O.synth_q4_k(blocks + rows, rows * blocks, 0.01))
    x = dev(O.normal(ncol * cols, 7 + ncol).reshape(ncol, cols))
    gain = dev(O.normal(cols, 3, 1.0, 0.1))
    want, y = (torch.full((ncol, rows), float("nan"), device="cuda") for _ in range(2))
    eager, fresh = ops.Context(0), ops.Context(0, own_stream=True)
    eager.q4_k_gemv_ncol(w, x, cols, rows, ncol, gain=gain, y=want)
    torch.cuda.synchronize()
    fresh.program_begin()
    fresh.q4_k_gemv_ncol(w, x, cols, rows, ncol, gain=gain, y=y)
    program = fresh.program_end()
    for _ in range(3):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        program.run()
        fresh.sync()
        assert torch.equal(y.view(torch.int32), want.view(torch.int32))
    program.destroy()
    fresh.close()
    eager.close()
