"""GPU: router scores at the edges of their kernels' tiles (16 and 32 tokens and experts, shares of whole 16 columns), the
grouping of pairs with more than eight slots a token, and a whole layer of the most tokens that the gate/up kernel routes."""
import numpy as np
import pytest

import oracle as O
from tests import helpers as H
from tests.test_gpu_moe_gemm import TOL, ctx, dev, run_experts  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,experts,tokens", [
    (16, 8, 16), (48, 33, 17), (1408, 64, 16), (2944, 32, 40),      # fewer steps than waves; shares of unequal length
    (1040, 129, 513), (96, 128, 1000), (4112, 97, 33),              # tiles of 32 x 32 with a ragged edge on both sides
    (4100, 20, 15), (1026, 9, 6), (5120, 40, 5), (1044, 6, 40),     # few tokens; columns that are not whole 16s
])
def test_router_scores_tiles(ctx, hidden, experts, tokens):
    wr = O.normal(experts * hidden, 7 + hidden, 0.0, 0.02).reshape(experts, hidden)
    x = O.normal(tokens * hidden, 8 + experts).reshape(tokens, hidden)
    ids, wts, scores = ctx.moe_route_topk(dev(wr), dev(x), hidden, experts, 2, tokens, want_scores=True)
    ctx.sync()
    ref = x.astype(np.float64) @ wr.astype(np.float64).T
    assert np.allclose(scores.cpu().numpy(), ref, rtol=1e-6, atol=1e-6 * np.abs(ref).max())


def test_moe_grouping_of_twelve_slots(ctx):
    hidden, inter, experts, top_k, tokens = 64, 64, 16, 12, 1030
    wr, pool, offs, x = H.config5(hidden, inter, experts, tokens, seed=3)
    rng = np.random.default_rng(tokens)
    ids = np.stack([rng.permutation(experts)[:top_k] for _ in range(tokens)]).astype(np.int32)
    wts = rng.random((tokens, top_k)).astype(np.float32)
    y, act = run_experts(ctx, pool, offs, hidden, inter, experts, x, ids, wts)
    g, u, d = (pool[offs["gate_off"]:], pool[offs["up_off"]:], pool[offs["down_off"]:])
    for t in list(range(0, tokens, 101)) + [1023, 1024, tokens - 1]:
        ref = O.moe_experts_f64(g, u, d, hidden, inter, ids[t], wts[t], x[t])
        assert O.max_rel_err(act[t], ref["act"]) < TOL, t


@pytest.mark.parametrize("hidden,inter,experts,top_k,tokens", [(1408, 384, 64, 2, 15), (2112, 192, 200, 4, 9)])
def test_moe_layer_routed_by_the_gate_up_kernel(ctx, hidden, inter, experts, top_k, tokens):
    from leviathan_amd import ops
    wr, pool, offs, x = H.config5(hidden, inter, experts, tokens, seed=hidden)
    pools = ops.Context.moe_pools(dev(pool), hidden, inter, experts, offs["gate_off"], offs["up_off"], offs["down_off"])
    y, ids, wts = ctx.moe_layer_q4_0(pools, dev(wr), dev(x), top_k, tokens)
    rids, rwts, _ = ctx.moe_route_topk(dev(wr), dev(x), hidden, experts, top_k, tokens, want_scores=True)
    ctx.sync()
    y, ids, wts = y.cpu().numpy(), ids.cpu().numpy(), wts.cpu().numpy()
    assert np.array_equal(ids, rids.cpu().numpy()) and np.array_equal(wts, rwts.cpu().numpy())
    g, u, d = (pool[offs["gate_off"]:], pool[offs["up_off"]:], pool[offs["down_off"]:])
    for t in range(tokens):
        ref = O.moe_experts_f64(g, u, d, hidden, inter, ids[t], wts[t], x[t])
        y32, _ = O.moe_experts_f32(g, u, d, hidden, inter, ids[t], wts[t], x[t])
        assert O.max_rel_err(y[t], ref["y"]) < max(TOL, 1.5 * O.max_rel_err(y32, ref["y"])), t


@pytest.mark.parametrize("hidden,inter,experts,top_k,tokens", [
    (64, 64, 64, 64, 1), (64, 64, 65, 65 - 1, 2),                   # every slot of a wave; fewer tasks than waves
    (2048, 64, 128, 1, 1), (4096, 1024, 256, 8, 1), (2816, 2048, 129, 6, 3),   # 8, 16 and 12 waves, one row group and more
])
def test_moe_layer_lists_ids_and_weights_as_the_router(ctx, hidden, inter, experts, top_k, tokens):
    """The list that the gate/up kernel makes is the stand-alone router's, bit for bit: equal scores (lower index first) and
    an expert's scale."""
    from leviathan_amd import ops
    rng = np.random.default_rng(hidden + experts)
    wr = np.zeros((experts, hidden), np.float32)
    wr[:, 1] = rng.integers(-6, 7, experts) * 0.25                  # many ties, one-hot activations: the scores themselves
    x = np.zeros((tokens, hidden), np.float32)
    x[:, 1] = np.linspace(1.0, 0.5, tokens)
    scale = dev(rng.random(experts).astype(np.float32) + 0.5)
    pool = rng.integers(0, 256, experts * 3 * inter * hidden // 32 * 18, dtype=np.uint8)
    pool.reshape(-1, 18)[:, 1] = 0x20                               # fp16 scales of ordinary size
    step = experts * inter * hidden // 32 * 18
    pools = ops.Context.moe_pools(dev(pool), hidden, inter, experts, 0, step, 2 * step)
    for s in (None, scale):
        _, ids, wts = ctx.moe_layer_q4_0(pools, dev(wr), dev(x), top_k, tokens, expert_scale=s)
        rids, rwts = ctx.moe_route_topk(dev(wr), dev(x), hidden, experts, top_k, tokens, expert_scale=s)
        ctx.sync()
        assert np.array_equal(ids.cpu().numpy(), rids.cpu().numpy())
        assert np.array_equal(wts.cpu().numpy(), rwts.cpu().numpy())
    order = np.lexsort((np.arange(experts), -wr[:, 1]))[:top_k]
    assert ids.cpu().numpy()[0].tolist() == order.tolist()
