"""GPU: Q4_0 products on the integer matrix cores with activations far above the rest where the row's scale is zero (a block of
zero weights): such a block adds nothing, so the rest of the row has to keep the accuracy that it has without it.

Bound: integers of 31 bits are exact within a block, what is rounded after them is a block's sum (three times), its pair, the
pairs of a lane group, the waves of a row and the store, at most 16 roundings of 2^-25 (rms of a half unit in the last place)
of partial sums no larger than the total: 16 * 2^-25 = 4.8e-7 in the 2-norm."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu
BOUND = 16 * 2.0 ** -25


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def rel(got, want):
    return np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want)


def outlier_columns(n):
    """One column in every other block: the first block of a pair and the second in turn."""
    pairs = np.arange((n // 32 + 1) // 2)
    cols = 64 * pairs + np.where(pairs % 2, 37, 5)
    return cols[cols < n]


def without_scale(w, rows, n, cols):
    w = w.reshape(rows, n // 32, 18).copy()
    w[:, cols // 32, :2] = 0
    return w.reshape(-1)


# whole tasks; a part of one; two tasks a wave; rows of an odd number of blocks (one, two and four tasks a wave)
@pytest.mark.parametrize("in_dim", [256, 2112, 4096, 6144, 1056, 4128, 12320])
@pytest.mark.parametrize("e", [0, 8, 16, 40])
def test_gemv(in_dim, e):
    from leviathan_amd import ops
    ctx = ops.Context(0)
    rows, cols = 300, outlier_columns(in_dim)
    w = without_scale(O.synth_q4_0(in_dim, rows * in_dim // 32, 0.02), rows, in_dim, cols)
    x = O.normal(in_dim, e).astype(np.float32)
    x[cols] = np.ldexp(np.where(np.arange(cols.size) % 3 == 1, -1.0, 1.0), e)
    y = ctx.q4_0_gemv(dev(w), dev(x), in_dim, rows)
    ctx.sync()
    assert rel(y.cpu().numpy(), O.q4_0_matvec_f64(w, rows, in_dim, x)) < BOUND
    ctx.close()


@pytest.mark.parametrize("inter", [64, 320, 1216, 2112])
def test_shared_ffn(inter):
    """Outliers of the input to gate and up, and of the one to the down projection."""
    from leviathan_amd import ops
    ctx = ops.Context(0)
    hidden = 1024
    hc, ic = outlier_columns(hidden), outlier_columns(inter)
    gate = without_scale(O.synth_q4_0(1, inter * hidden // 32, 0.02), inter, hidden, hc)
    up = without_scale(O.synth_q4_0(2, inter * hidden // 32, 0.02), inter, hidden, hc)
    rows = up.reshape(inter, hidden // 32, 18)            # the outliers of act: rows of up with larger scales
    d = rows[ic, :, :2].copy().view(np.float16)
    rows[ic, :, :2] = (d * np.float16(32768)).view(np.uint8)
    down = without_scale(O.synth_q4_0(3, hidden * inter // 32, 0.02), hidden, inter, ic)
    x = O.normal(hidden, 4).astype(np.float32)
    x[hc] = 2.0 ** 16
    _, shared = ctx.shared_expert_ffn(dev(x), None, dev(gate), dev(up), dev(down), None, hidden, inter, eps=0.0,
                                      bufs=(h := torch.empty(hidden, device="cuda"), gu := torch.empty(2 * inter, device="cuda"),
                                            act := torch.empty(inter, device="cuda"), torch.empty(hidden, device="cuda")))
    ctx.sync()
    hf, guf, actf = (t.cpu().numpy() for t in (h, gu, act))   # each stage on the device's own input to it
    assert rel(guf[:inter], O.q4_0_matvec_f64(gate, inter, hidden, hf)) < BOUND
    want = O.q4_0_matvec_f64(up, inter, hidden, hf)
    rest = np.setdiff1d(np.arange(inter), ic)
    assert rel(guf[inter:][rest], want[rest]) < BOUND
    assert np.abs(actf[ic]).max() > 500 * np.abs(actf[rest]).max()
    want = O.q4_0_matvec_f64(down, hidden, inter, actf)
    want /= np.sqrt(np.mean(want ** 2))
    assert rel(shared.cpu().numpy(), want) < BOUND + 3 * 2.0 ** -24   # (the norm: its factor and the product)
    ctx.close()
