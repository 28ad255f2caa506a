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


@pytest.mark.parametrize("kind,rows,cols,tokens", [
    ("q6_k", 32000, 1024, 1250),     # 250 row tiles: five token tiles of a workgroup one after the other, the last ragged
    ("q6_k", 16384, 1280, 1510),     # 128 row tiles: two token tiles side by side, three in turn
    ("q6_k", 6140, 1024, 1270),      # one round of 240 workgroups, the last row tile ragged
    ("q4_k", 24570, 2048, 2290),     # nine rounds, ragged in rows and tokens
    ("q4_k", 12288, 2048, 1985),     # eight token tiles, the last one ragged
    ("q4_k", 12288, 2048, 1500),     # three rounds: the estimates within 1.1 of each other
])
def test_gemm_long_prompts_in_256_token_tiles(ctx, kind, rows, cols, tokens):
    """Prompts above 1024 tokens whose 256-token tiles fill the chip: each tile is the product of its tokens alone, which
    the 128-token kernel forms in the same order where it never cuts K (from 768 row tiles, below six superblocks), bit
    for bit; sampled rows meet the gate."""
    w, x = (H.config4 if kind == "q4_k" else config4_q6)(rows, cols, tokens, seed=rows + tokens)
    run = gemm if kind == "q4_k" else gemm6
    got = run(ctx, w, x, rows, cols, tokens)
    whole = rows > 767 * 32 or cols < 6 * 256
    for lo in (0, tokens // 512 * 256, tokens // 256 * 256) if whole else ():
        hi = min(lo + 256, tokens)
        part = run(ctx, w, x[lo:hi].copy(), rows, cols, hi - lo)
        assert np.array_equal(part.view(np.uint32), got[lo:hi].view(np.uint32)), (lo, hi)
    oracle = O.q4_k_gemm_f16_oracle if kind == "q4_k" else O.q6_k_gemm_f16_oracle
    assert O.max_rel_err(got[:, 0::499], oracle(w, rows, cols, x.view(np.uint16), tokens, 0, 499)) < GEMM_TOL


@pytest.mark.parametrize("kind,rows,cols,tokens", [
    ("q4_k", 12200, 2048, 505),     # row tiles of 96, the last ragged; the second token tile ragged
    ("q4_k", 24500, 4352, 241),     # an odd number of superblocks, one token tile; row tiles of 128
    ("q6_k", 12200, 2048, 505),
    ("q6_k", 31990, 2304, 500),     # row tiles of 128, two rounds
    ("q6_k", 12288, 1792, 256),
])
def test_gemm_256_token_tiles(ctx, kind, rows, cols, tokens):
    """Prompts whose 256-token tiles fill the chip: sampled rows meet the gate, and recorded on a context without room for
    X in the order of the fragments the call forms the same sums in the same order."""
    from leviathan_amd import ops
    w, x = (H.config4 if kind == "q4_k" else config4_q6)(rows, cols, tokens, seed=rows + tokens)
    got = (gemm if kind == "q4_k" else gemm6)(ctx, w, x, rows, cols, tokens)
    oracle = O.q4_k_gemm_f16_oracle if kind == "q4_k" else O.q6_k_gemm_f16_oracle
    assert O.max_rel_err(got[:, 0::331], oracle(w, rows, cols, x.view(np.uint16), tokens, 0, 331)) < GEMM_TOL
    assert O.max_rel_err(got[:, rows - 1:], oracle(w, rows, cols, x.view(np.uint16), tokens, rows - 1, rows)) < GEMM_TOL
    wd, xd = dev(w), dev(x)
    fresh = ops.Context(0, own_stream=True)
    y = torch.full((tokens, rows), float("nan"), device="cuda")
    torch.cuda.synchronize()
    fresh.program_begin()
    (fresh.q4_k_gemm_prefill if kind == "q4_k" else fresh.q6_k_gemm_prefill)(wd, xd, cols, rows, tokens, y=y)
    program = fresh.program_end()
    for _ in range(3):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        program.run()
        fresh.sync()
        assert np.array_equal(y.cpu().numpy().view(np.uint32), got.view(np.uint32))
    program.destroy()
    fresh.close()
