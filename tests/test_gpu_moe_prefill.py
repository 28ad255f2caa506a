"""GPU parity of the grouped matrix product that serves prompts and large batches of the MoE layer, at the
edges of its tiles: column tiles of 32 in items of 64 pairs, rows in tiles of 128 (gate/up) and 256 (down)
cut into waves, K in steps of two blocks and weight groups of four.  FP64 chain at the reference's 1e-4."""
import numpy as np
import pytest

import oracle as O
from tests import helpers as H
from tests.test_gpu_moe_gemm import TOL, ctx, run_experts  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,inter,counts", [
    (64, 64, (1, 32)),            # one K-step, one weight group of two blocks
    (192, 320, (33, 31, 0)),      # rows past the last whole wave tile; a last group of two blocks
    (320, 192, (64, 65)),         # a full item; a second item of one pair
    (2816, 704, (97, 7, 128)),
    (4160, 128, (40, 24)),        # rows wider than the few-token kernels take
])
def test_moe_grouped_product_tiles(ctx, hidden, inter, counts):
    """One slot a token: expert e takes exactly counts[e] pairs."""
    experts, tokens = len(counts), sum(counts)
    wr, pool, offs, x = H.config5(hidden, inter, experts, tokens, seed=hidden + inter)
    rng = np.random.default_rng(tokens)
    ids = rng.permutation(np.repeat(np.arange(experts), counts)).astype(np.int32)[:, None]
    wts = rng.random((tokens, 1)).astype(np.float32)
    y, act = run_experts(ctx, pool, offs, hidden, inter, experts, x, ids, wts)
    g, u, d = (pool[offs["gate_off"]:], pool[offs["up_off"]:], pool[offs["down_off"]:])
    for t in range(0, tokens, 1 if hidden < 1000 else 9):
        ref = O.moe_experts_f64(g, u, d, hidden, inter, ids[t], wts[t], x[t])
        assert O.max_rel_err(act[t], ref["act"]) < TOL, t
        y32, _ = O.moe_experts_f32(g, u, d, hidden, inter, ids[t], wts[t], x[t])
        assert O.max_rel_err(y[t], ref["y"]) < max(TOL, 1.5 * O.max_rel_err(y32, ref["y"])), t


@pytest.mark.parametrize("hidden,inter,experts,top_k,tokens", [
    (2816, 704, 14, 8, 9),        # eleven column tasks a row (twelve waves); a last task of three pairs
    (4096, 4096, 4, 2, 6),        # sixteen tasks both ways
    (3136, 1088, 9, 4, 12),       # thirteen, the last of one pair; five, the last of one
])
def test_moe_grouped_integer_kernels_ragged_rows(ctx, hidden, inter, experts, top_k, tokens):
    """The integer grouped kernels on rows that end inside a 256-value task and rows wider than eight tasks."""
    wr, pool, offs, x = H.config5(hidden, inter, experts, tokens, seed=hidden + inter)
    rng = np.random.default_rng(tokens)
    ids = np.stack([rng.permutation(experts)[:top_k] for _ in range(tokens)]).astype(np.int32)
    wts = rng.random((tokens, top_k)).astype(np.float32)
    assert 2 * tokens * top_k <= 11 * experts
    y, act = run_experts(ctx, pool, offs, hidden, inter, experts, x, ids, wts)
    g, u, d = (pool[offs["gate_off"]:], pool[offs["up_off"]:], pool[offs["down_off"]:])
    for t in range(tokens):
        ref = O.moe_experts_f64(g, u, d, hidden, inter, ids[t], wts[t], x[t])
        assert O.max_rel_err(act[t], ref["act"]) < TOL
        y32, _ = O.moe_experts_f32(g, u, d, hidden, inter, ids[t], wts[t], x[t])
        assert O.max_rel_err(y[t], ref["y"]) < max(TOL, 1.5 * O.max_rel_err(y32, ref["y"]))


@pytest.mark.parametrize("hidden,inter,experts,top_k,tokens", [
    (3136, 960, 6, 4, 1),         # thirteen column tasks a row, the last of one pair; four, the last of three
    (2112, 64, 4, 2, 3), (4032, 448, 5, 3, 4), (192, 704, 9, 8, 2),
])
def test_moe_few_tokens_ragged_rows(ctx, hidden, inter, experts, top_k, tokens):
    """The few-token matrix-core kernels on rows that end inside a 256-value task."""
    wr, pool, offs, x = H.config5(hidden, inter, experts, tokens, seed=hidden + inter)
    rng = np.random.default_rng(tokens)
    ids = np.stack([rng.permutation(experts)[:top_k] for _ in range(tokens)]).astype(np.int32)
    wts = rng.random((tokens, top_k)).astype(np.float32)
    y, act = run_experts(ctx, pool, offs, hidden, inter, experts, x, ids, wts)
    g, u, d = (pool[offs["gate_off"]:], pool[offs["up_off"]:], pool[offs["down_off"]:])
    for t in range(tokens):
        ref = O.moe_experts_f64(g, u, d, hidden, inter, ids[t], wts[t], x[t])
        assert O.max_rel_err(act[t], ref["act"]) < TOL
        y32, _ = O.moe_experts_f32(g, u, d, hidden, inter, ids[t], wts[t], x[t])
        assert O.max_rel_err(y[t], ref["y"]) < max(TOL, 1.5 * O.max_rel_err(y32, ref["y"]))
