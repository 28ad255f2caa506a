"""GPU: two contexts on one device ask for different amounts of LDS of the same kernel, in turn and from two threads."""
import threading

import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def test_two_contexts_share_a_kernel_at_different_lds_sizes():
    from leviathan_amd import ops
    ctxs = [ops.Context(0, own_stream=True) for _ in range(2)]
    rows, ncol = 33, 4
    wide = {}
    for cols in (4096, 8192):                       # the same instantiation: 4 columns staged, SHORT
        w, x = O.synth_q4_k(cols, rows * cols // 256, 0.01), O.normal(ncol * cols, cols + 1).reshape(ncol, cols)
        wide[cols] = (dev(w), dev(x), np.stack([O.q4_k_matvec_f64(w, rows, cols, c) for c in x]))
    torch.cuda.synchronize()
    bad = []

    def run(ctx, order):
        for cols in order:
            w, x, ref = wide[cols]
            y = torch.full((ncol, rows), float("nan"), device="cuda")
            torch.cuda.synchronize()
            ctx.q4_k_gemv_ncol(w, x, cols, rows, ncol, y=y)
            ctx.sync()
            if O.max_rel_err(y.cpu().numpy(), ref) > 1e-4:
                bad.append(cols)
    for ctx, order in ((ctxs[0], (8192,)), (ctxs[1], (4096,)), (ctxs[0], (8192,))):
        run(ctx, order)
    threads = [threading.Thread(target=run, args=(c, o)) for c, o in zip(ctxs, ((8192, 4096) * 8, (4096, 8192) * 8))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for c in ctxs:
        c.close()
