"""GPU parity of the prefill GEMM for short prompts (a wave decodes its own rows, K cut into slices), at its
edges: token tiles of 32 (one to four a wave, several a call), 32-row waves in 128-row workgroups, slices of
unequal numbers of superblocks, partial sums in scratch.  Gate of the prefill GEMMs: 1e-3, every row and token."""
import numpy as np
import pytest
import torch

import oracle as O
from tests import helpers as H
from tests.test_gpu_moe_gemm import GEMM_TOL, ctx, config4_q6, dev, gemm, gemm6  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["q4_k", "q6_k"])
@pytest.mark.parametrize("rows,cols,tokens", [
    (31, 256, 31),          # less than a wave's rows, one superblock
    (129, 1792, 33),        # a second workgroup of one row; seven superblocks over up to six slices
    (160, 2816, 96), (257, 1536, 97),
    (700, 3328, 128), (96, 4096, 129),
    (400, 2304, 400),       # four token tiles
    (1130, 4864, 643),      # four slices of tiles of 96 tokens: the most LDS a workgroup of either format takes
])
def test_gemm_split_edges(ctx, kind, rows, cols, tokens):
    if kind == "q4_k":
        w, x = H.config4(rows, cols, tokens, seed=rows + tokens)
        got = gemm(ctx, w, x, rows, cols, tokens)
        ref = O.q4_k_gemm_f16_oracle(w, rows, cols, x.view(np.uint16), tokens, 0, 1)
    else:
        w, x = config4_q6(rows, cols, tokens, seed=rows + tokens)
        got = gemm6(ctx, w, x, rows, cols, tokens)
        ref = O.q6_k_gemm_f16_oracle(w, rows, cols, x.view(np.uint16), tokens, 0, 1)
        shifted = gemm6(ctx, np.concatenate([np.zeros(2, np.uint8), w]), x, rows, cols, tokens, w_off=2)
        assert np.array_equal(shifted.view(np.uint32), got.view(np.uint32))
    assert O.max_rel_err(got, ref) < GEMM_TOL


def test_gemm_split_recorded_without_scratch(ctx):
    """Recording never grows the scratch: a call that would want it for partial sums takes all of K instead."""
    from leviathan_amd import ops
    rows, cols, tokens = 512, 4096, 40
    w, x = H.config4(rows, cols, tokens, seed=5)
    wd, xd = dev(w), dev(x)
    eager = gemm(ctx, w, x, rows, cols, tokens)
    fresh = ops.Context(0, own_stream=True)
    y = torch.full((tokens, rows), float("nan"), device="cuda")
    torch.cuda.synchronize()
    fresh.program_begin()
    fresh.q4_k_gemm_prefill(wd, xd, cols, rows, tokens, y=y)
    program = fresh.program_end()
    for _ in range(3):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        program.run()
        fresh.sync()
        got = y.cpu().numpy()
        assert np.linalg.norm(got - eager) < 1e-5 * np.linalg.norm(eager)     # f32 sums in another order
    program.destroy()
    fresh.close()


@pytest.mark.parametrize("kind,rows,cols,tokens", [("q4_k", 512, 4096, 40), ("q4_k", 129, 1792, 33), ("q4_k", 257, 12288, 70),
                                                   ("q6_k", 512, 4096, 40), ("q6_k", 96, 8192, 129), ("q6_k", 33, 11008, 97)])
def test_gemm_split_records_the_eager_bits(ctx, kind, rows, cols, tokens):
    """Slices that workgroups share meet in scratch or, recorded where there is none, one launch after the other in y:
    the same sums in the same order."""
    from leviathan_amd import ops
    w, x = (H.config4 if kind == "q4_k" else config4_q6)(rows, cols, tokens, seed=rows + tokens)
    wd, xd = dev(w), dev(x)
    eager = (gemm if kind == "q4_k" else gemm6)(ctx, w, x, rows, cols, tokens)
    fresh = ops.Context(0, own_stream=True)
    y = torch.empty(tokens, rows, device="cuda")
    torch.cuda.synchronize()
    fresh.program_begin()
    (fresh.q4_k_gemm_prefill if kind == "q4_k" else fresh.q6_k_gemm_prefill)(wd, xd, cols, rows, tokens, y=y)
    program = fresh.program_end()
    for _ in range(3):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        program.run()
        fresh.sync()
        assert np.array_equal(y.cpu().numpy().view(np.uint32), eager.reshape(tokens, rows).view(np.uint32))
    program.destroy()
    fresh.close()
