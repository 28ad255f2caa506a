"""GPU: the Q6_K matrix-core GEMVs on rows of an odd number of 210-byte superblocks, where every other row starts off
the dword boundary: one row, a partial and a full task of 16 rows, one row more, many rounds; f32 and int8 activations."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("rows", [1, 2, 15, 16, 17, 12301])
@pytest.mark.parametrize("blocks", [1, 3, 11, 16, 17, 29])
def test_q6_rows_off_the_dword_boundary(rows, blocks):
    from leviathan_amd import ops
    if rows > 1000 and blocks not in (11, 17):
        rows = 513                                  # several rounds on these as well, cheaper to check
    ctx = ops.Context(0)
    cols = 256 * blocks
    w = O.synth_q6_k(blocks + rows, rows * blocks)
    dw = dev(w)
    for ncol in (1, 2, 3):
        x = O.normal(ncol * cols, ncol).reshape(ncol, cols)
        y = ctx.q6_k_gemv_ncol(dw, dev(x), cols, rows, ncol).cpu().numpy() if ncol > 1 else \
            ctx.q6_k_gemv(dw, dev(x[0]), cols, rows).cpu().numpy()[None]
        for c in range(ncol):
            assert O.max_rel_err(y[c], O.q6_k_matvec_f64(w, rows, cols, x[c])) < 1e-5, (rows, blocks, ncol, c)
    for ncol in (1, 5):
        x = O.normal(ncol * cols, 7 + ncol).reshape(ncol, cols)
        q = [O.quantize_q8(v) for v in x]
        xq = np.stack([a for a, *_ in q])
        d = np.stack([b for _, b, *_ in q])
        xs = np.stack([d, d * xq.reshape(ncol, -1, 32).sum(2)], axis=2).astype(np.float32)
        y = ctx.q6_k_gemv_q8(dw, dev(xq), dev(xs), cols, rows, ncol).cpu().numpy()
        for c in range(ncol):
            assert O.max_rel_err(y[c], O.q6_k_matvec_q8_f64(w, rows, cols, xq[c], d[c])) < 1e-4, (rows, blocks, ncol, c)
    ctx.close()
