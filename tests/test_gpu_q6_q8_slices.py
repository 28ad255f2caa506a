"""GPU: int8-activation Q6_K GEMV on rows wider than a workgroup's waves, which are cut into slices: the first width with
two slices, a last slice that is shorter than the others, more row groups than workgroups; every width of the operand."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("ncol", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("blocks,rows", [(9, 17), (17, 1), (17, 4099), (19, 2000), (33, 48), (48, 31), (64, 1040)])
def test_q6_q8_sliced_rows(blocks, rows, ncol):
    from leviathan_amd import ops
    ctx = ops.Context(0)
    cols = 256 * blocks
    w = O.synth_q6_k(blocks + rows, rows * blocks)
    x = O.normal(ncol * cols, 7 + ncol).reshape(ncol, cols)
    q = [O.quantize_q8(v) for v in x]
    xq = np.stack([a for a, *_ in q])
    d = np.stack([b for _, b, *_ in q])
    xs = np.stack([d, d * xq.reshape(ncol, -1, 32).sum(2)], axis=2).astype(np.float32)
    outs = []
    for _ in range(2):                              # the second call finds the arrival counters as the first left them
        y = torch.full((ncol, rows), float("nan"), device="cuda")
        ctx.q6_k_gemv_q8(dev(w), dev(xq), dev(xs), cols, rows, ncol, y=y)
        ctx.sync()
        outs.append(y.cpu().numpy())
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    pick = sorted({0, rows - 1, rows // 2, min(rows - 1, 15), min(rows - 1, 16)})
    ww = w.reshape(rows, -1)[pick].reshape(-1)
    for c in range(ncol):
        ref = O.q6_k_matvec_q8_f64(ww, len(pick), cols, xq[c], d[c])
        assert np.allclose(outs[0][c][pick], ref, rtol=1e-4, atol=1e-4 * np.abs(ref).max() + 1e-6), (blocks, rows, ncol, c)
    ctx.close()


@pytest.mark.parametrize("ncol", [4, 9, 16])
@pytest.mark.parametrize("blocks,rows", [(10, 4096), (10, 12288), (17, 4096), (17, 16016), (18, 2064)])
def test_q6_q8_sliced_or_staged(blocks, rows, ncol):
    """Either side of the line from which wide rows are left to the kernel that stages the activations: by rows, by
    columns, and by width where it no longer holds sixteen columns in one pass."""
    test_q6_q8_sliced_rows(blocks, rows, ncol)


@pytest.mark.parametrize("blocks,rows,ncol", [(17, 300, 1), (19, 2000, 4), (33, 48, 8), (9, 17, 9), (48, 1000, 16)])
def test_q6_q8_sliced_rows_record_the_eager_bits(blocks, rows, ncol):
    """Recorded on a context without scratch the slices are launched one after the other: the same sums in the same
    order as where they meet in scratch."""
    from leviathan_amd import ops
    cols = 256 * blocks
    w = dev(O.synth_q6_k(blocks + rows, rows * blocks))
    x = O.normal(ncol * cols, 7 + ncol).reshape(ncol, cols)
    q = [O.quantize_q8(v) for v in x]
    xq = np.stack([a for a, *_ in q])
    d = np.stack([b for _, b, *_ in q])
    xs = dev(np.stack([d, d * xq.reshape(ncol, -1, 32).sum(2)], axis=2).astype(np.float32))
    xq = dev(xq)
    want, y = (torch.full((ncol, rows), float("nan"), device="cuda") for _ in range(2))
    eager, fresh = ops.Context(0), ops.Context(0, own_stream=True)
    eager.q6_k_gemv_q8(w, xq, xs, cols, rows, ncol, y=want)
    torch.cuda.synchronize()
    fresh.program_begin()
    fresh.q6_k_gemv_q8(w, xq, xs, cols, rows, ncol, y=y)
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


@pytest.mark.parametrize("ncol", [1, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("blocks,rows", [(17, 15), (18, 4096), (19, 4097), (31, 33), (32, 8200), (33, 2049), (41, 4095), (48, 2064),
                                         (48, 2048), (49, 2056), (63, 4096), (64, 3000), (33, 4097)])
def test_q6_q8_whole_row_groups(blocks, rows, ncol):
    """Rows of which a wave takes two, three or four superblocks: an odd number of them, one short and one more than the
    waves hold, row groups that end inside one, one round and several, and either side of the lines to the slices."""
    test_q6_q8_sliced_rows(blocks, rows, ncol)
