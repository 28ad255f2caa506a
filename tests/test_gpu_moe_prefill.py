"""GPU parity of the grouped matrix product that serves prompts and large batches of the MoE layer, at the
edges of its tiles: column tiles of 32 in items of 64 pairs, workgroups of four, eight and twelve waves of 16
(gate/up) and 32 (down) rows, K in steps of two blocks and weight groups of four.  FP64 chain at the reference's 1e-4."""
import numpy as np
import pytest
import torch

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


@pytest.mark.parametrize("hidden,inter,experts,tokens", [
    (1024, 512, 2, 100),          # 32 blocks a row: one chain
    (1088, 512, 2, 100),          # 34: two parts and two blocks
    (4096, 256, 2, 64),           # 128: eight parts, workgroups of four waves
    (1088, 384, 128, 1200),       # workgroups of twelve waves; rows past the last whole workgroup
    (256, 1088, 2, 260),          # down folded
])
def test_moe_grouped_product_folded_sums(ctx, hidden, inter, experts, tokens):
    """The f32 sums of the grouped product against 64 bits, on positive weights and activations, where a chain's
    partial sums grow evenly: n additions leave sqrt(n / 3) roundings u = 2^-24 / sqrt(3) of the whole (rms), 3.3 at
    32 blocks and 6.5 at 128, parts of 16 blocks folded at most 2.0 (8 parts).  gelu is the identity here, so
    act = g * u has sqrt(2) times that and some two roundings of its own: 5.1 u, held to 5.5; y adds its own row and
    some two: 6.4 u, held to 7.  One chain of 128 blocks leaves 9.4 u in act."""
    u = 2.0 ** -24 / 3 ** 0.5
    wr, pool, offs, x = H.config5(hidden, inter, experts, tokens, seed=hidden + inter)
    blocks = pool.reshape(-1, 18)
    blocks[:, 1] &= 0x7F
    blocks[:, 2:] |= 0x88
    x = np.abs(x)
    rng = np.random.default_rng(tokens)
    ids = rng.permutation(np.arange(tokens) % experts).astype(np.int32)[:, None]
    wts = np.ones((tokens, 1), np.float32)
    y, act = run_experts(ctx, pool, offs, hidden, inter, experts, x, ids, wts)
    g, up, d = (pool[offs["gate_off"]:], pool[offs["up_off"]:], pool[offs["down_off"]:])
    off = {"act": [], "y": []}
    for t in range(0, tokens, max(1, tokens // 24)):
        ref = O.moe_experts_f64(g, up, d, hidden, inter, ids[t], wts[t], x[t])
        for k, got in (("act", act[t]), ("y", y[t])):
            r = np.asarray(ref[k], np.float64).ravel()
            off[k].append((np.linalg.norm(got.astype(np.float64).ravel() - r) / np.linalg.norm(r)) ** 2)
    act_off, y_off = (np.sqrt(np.mean(off[k])) / u for k in ("act", "y"))
    print(f"act {act_off:.2f} u, y {y_off:.2f} u")
    assert act_off < 5.5
    assert y_off < 7


@pytest.mark.parametrize("x_exp,d_exp", [
    (68, -24),      # act near 2^127.6: its own power of two scales it
    (-63, 12),      # act near 2^-135, a subnormal number
])
def test_moe_grouped_product_range_of_act(ctx, x_exp, d_exp):
    """Rows of act whose maximum is at either end of f32's range are operands like any other.  g = u = 7 d x[0] with
    the gate's and the up matrix's only weights in column 0; every weight of down is 7 * 2^d_exp."""
    hidden = inter = 320
    experts, tokens = 2, 700
    gu, dn = inter * hidden // 32 * 18, hidden * inter // 32 * 18
    one = np.zeros((inter * hidden // 32, 18), np.uint8)
    one[:, 2:] = 0x88                                                # weight zero
    one[:, 0:2] = np.array([2.0 ** -7], np.float16).view(np.uint8)
    one.reshape(inter, hidden // 32, 18)[:, 0, 2] = 0x8F             # element 0: 7
    down = np.empty((hidden * inter // 32, 18), np.uint8)
    down[:, 2:] = 0xFF
    down[:, 0:2] = np.array([2.0 ** d_exp], np.float16).view(np.uint8)
    pool = np.concatenate([np.tile(one.ravel(), 2 * experts), np.tile(down.ravel(), experts)])
    offs = dict(gate_off=0, up_off=experts * gu, down_off=2 * experts * gu, gate_stride=gu, up_stride=gu, down_stride=dn)
    x = np.zeros((tokens, hidden), np.float32)
    x[:, 0] = np.ldexp(1.0 + np.arange(tokens) / 8192.0, x_exp)
    ids = (np.arange(tokens) % experts).astype(np.int32)[:, None]
    y, act = run_experts(ctx, pool, offs, hidden, inter, experts, x, ids, np.ones((tokens, 1), np.float32))
    g = 7 * 2.0 ** -7 * x[:, :1].astype(np.float64)
    want = (g if x_exp > 0 else 0.5 * g) * g
    quantum = 2.0 ** -149
    assert np.all(np.abs(act[:, 0] - want) <= 1e-6 * want + quantum)
    # against the act that was stored, whose subnormal numbers have fewer bits
    y_want = act[:, 0].astype(np.float64).sum(axis=1, keepdims=True) * 7 * 2.0 ** d_exp
    assert np.all(np.isfinite(y)) and np.all(y > 0)
    assert np.all(np.abs(y - y_want) <= 1e-6 * y_want)


def test_moe_experts_with_their_own_act_record_on_a_fresh_context(ctx):
    """A caller that brings `act` needs no scratch of the context's but for grouping: recorded on a context that has
    none, where nothing may be allocated, the pairs are taken one by one."""
    from leviathan_amd import capi, ops
    import ctypes as C
    hidden, inter, experts, tokens = 320, 192, 2, 700
    wr, pool, offs, x = H.config5(hidden, inter, experts, tokens, seed=9)
    rng = np.random.default_rng(9)
    ids = (np.arange(tokens) % experts).astype(np.int32)[:, None]
    wts = rng.random((tokens, 1)).astype(np.float32)
    want_y, want_act = run_experts(ctx, pool, offs, hidden, inter, experts, x, ids, wts)      # grouped
    fresh = ops.Context(0, own_stream=True)
    pool_d, x_d, ids_d, wts_d = (torch.from_numpy(a).cuda() for a in (pool, x, ids, wts))
    pools = ops.Context.moe_pools(pool_d, hidden, inter, experts, offs["gate_off"], offs["up_off"], offs["down_off"])
    y, act = torch.empty(tokens, hidden, device="cuda"), torch.empty(tokens, 1, inter, device="cuda")
    torch.cuda.synchronize()
    fresh.program_begin()
    st = fresh.lib.lev_hip_moe_experts_q4_0(fresh.ctx, C.byref(pools), *(C.c_void_p(t.data_ptr()) for t in (x_d, ids_d, wts_d, y, act)),
                                            1, tokens)
    program = fresh.program_end()
    assert st == capi.OK
    for _ in range(3):
        y.fill_(float("nan")), act.fill_(float("nan"))
        torch.cuda.synchronize()
        program.run()
        fresh.sync()
        assert O.max_rel_err(act.cpu().numpy().ravel(), want_act.ravel()) < 1e-4
        assert O.max_rel_err(y.cpu().numpy().ravel(), want_y.ravel()) < 1e-4
    program.destroy()
    fresh.close()


@pytest.mark.parametrize("hidden,inter,counts", [
    (64, 64, (1, 32)), (192, 320, (33, 31, 0)), (320, 192, (64, 65)), (4160, 128, (40, 24)), (4160, 64, (97, 7, 128)),
])
def test_moe_grouped_product_tiles_of_small_experts(ctx, hidden, inter, counts):
    """The tiles of test_moe_grouped_product_tiles where experts are so small that pairs are only grouped when there are
    thousands: one expert more takes as many as the rule asks for (65 MB of weights that grouping saves reading, ten
    experts' worth counted in; lev_moe_grouped_usable), twelve of them checked."""
    nbytes = 3 * hidden * inter * 18 // 32
    counts = counts + (int(65e6 / nbytes) + 70,)
    experts, tokens = len(counts), sum(counts)
    assert (tokens - experts + 10) * nbytes >= 65e6 and tokens > 8 * experts
    wr, pool, offs, x = H.config5(hidden, inter, experts, tokens, seed=hidden + inter)
    rng = np.random.default_rng(tokens)
    ids = rng.permutation(np.repeat(np.arange(experts), counts)).astype(np.int32)[:, None]
    wts = rng.random((tokens, 1)).astype(np.float32)
    y, act = run_experts(ctx, pool, offs, hidden, inter, experts, x, ids, wts)
    g, u, d = (pool[offs["gate_off"]:], pool[offs["up_off"]:], pool[offs["down_off"]:])
    filler = np.flatnonzero(ids[:, 0] == experts - 1)
    for t in np.concatenate([np.flatnonzero(ids[:, 0] != experts - 1), filler[::max(1, len(filler) // 12)]]):
        ref = O.moe_experts_f64(g, u, d, hidden, inter, ids[t], wts[t], x[t])
        assert O.max_rel_err(act[t], ref["act"]) < TOL, t
        y32, _ = O.moe_experts_f32(g, u, d, hidden, inter, ids[t], wts[t], x[t])
        assert O.max_rel_err(y[t], ref["y"]) < max(TOL, 1.5 * O.max_rel_err(y32, ref["y"])), t


# hidden, inter, experts, tokens, (pairs an item, form of gate/up, form of down) on 256 CUs: test_moe_rules.py holds the forms
FORMS = [
    (1024, 1088, 64, 832, (64, 0, 3)),
    (1088, 1088, 64, 832, (64, 1, 1)),        # 17 steps a row: a last group of two blocks; waves past the last row
    (1280, 640, 32, 7200, (64, 2, 0)),        # experts of four items
    (1088, 2176, 40, 560, (64, 1, 3)),
    (1088, 512, 16, 800, (64, 3, 0)),
    (1088, 1088, 32, 640, (32, 4, 4)),
    (2304, 1280, 32, 2000, (64, 2, 2)),
]


@pytest.mark.parametrize("hidden,inter,experts,tokens,forms", FORMS)
def test_moe_grouped_product_forms(ctx, hidden, inter, experts, tokens, forms):
    """Every form of the product, with lists at the edges of column tiles and items: one pair, and one more and less than
    32 and 64.  Tokens of those lists and some others are checked."""
    edges = [1, 31, 32, 33, 63, 64, 65]
    wr, pool, offs, x = H.config5(hidden, inter, experts, tokens, seed=hidden + inter)
    rng = np.random.default_rng(tokens)
    rest = rng.multinomial(tokens - sum(edges), [1 / (experts - len(edges))] * (experts - len(edges)))
    ids = rng.permutation(np.repeat(np.arange(experts), edges + rest.tolist())).astype(np.int32)[:, None]
    wts = rng.random((tokens, 1)).astype(np.float32)
    y, act = run_experts(ctx, pool, offs, hidden, inter, experts, x, ids, wts)
    assert np.isfinite(y).all() and np.isfinite(act).all()
    g, u, d = (pool[offs["gate_off"]:], pool[offs["up_off"]:], pool[offs["down_off"]:])
    checked = np.concatenate([np.flatnonzero(ids[:, 0] == e)[[0, -1]] for e in range(experts)])
    for t in checked:
        ref = O.moe_experts_f64(g, u, d, hidden, inter, ids[t], wts[t], x[t])
        assert O.max_rel_err(act[t], ref["act"]) < TOL, t
        y32, _ = O.moe_experts_f32(g, u, d, hidden, inter, ids[t], wts[t], x[t])
        assert O.max_rel_err(y[t], ref["y"]) < max(TOL, 1.5 * O.max_rel_err(y32, ref["y"])), t


@pytest.mark.parametrize("hidden,inter,experts,tokens", [f[:4] for f in FORMS])
def test_moe_grouped_product_gives_a_pair_the_same_bits_anywhere(ctx, hidden, inter, experts, tokens):
    """The order of an expert's pairs is that of atomics, so where a pair lies (its item, its column tile, the tiles of its
    item) must not show in a bit: equal activations have equal outputs in all of an expert's lists of 1 to 65 pairs and more."""
    edges = [1, 31, 32, 33, 63, 64, 65]
    wr, pool, offs, x = H.config5(hidden, inter, experts, tokens, seed=hidden + inter)
    rng = np.random.default_rng(tokens)
    rest = rng.multinomial(tokens - sum(edges), [1 / (experts - len(edges))] * (experts - len(edges)))
    ids = rng.permutation(np.repeat(np.arange(experts), edges + rest.tolist())).astype(np.int32)[:, None]
    x[:] = x[0]
    y, act = run_experts(ctx, pool, offs, hidden, inter, experts, x, ids, np.full((tokens, 1), 0.75, np.float32))
    for e in range(experts):
        mine = np.flatnonzero(ids[:, 0] == e)
        assert (act[mine] == act[mine[0]]).all() and (y[mine] == y[mine[0]]).all(), e


@pytest.mark.parametrize("top_k,tokens,experts", [(8, 70, 24), (12, 40, 24), (3, 1100, 40), (8, 1030, 1100), (8, 1200, 1100)])
def test_moe_prompt_grouping_drops_bad_pairs(ctx, top_k, tokens, experts):
    """Pairs whose id is out of range or repeats another slot of their token are dropped and reported, in the first eight
    slots of a token and behind them, for the first 1024 tokens and for others, with one expert a thread of the grouping
    and with more (1030 tokens of 1100 experts: the integer kernels); every other pair counts."""
    from leviathan_amd import capi, ops
    from leviathan_amd.ops import LevError
    hidden, inter = 256, 256
    wr, pool, offs, x = H.config5(hidden, inter, experts, tokens, seed=top_k)
    rng = np.random.default_rng(top_k + tokens)
    ids = np.stack([rng.permutation(min(experts, 60))[:top_k] for _ in range(tokens)]).astype(np.int32)
    wts = rng.random((tokens, top_k)).astype(np.float32)
    bad = {1: (0, experts), 5: (top_k - 1, -1), tokens - 1: (top_k - 1, ids[tokens - 1, 0]), tokens - 2: (1, ids[tokens - 2, 2])}
    for t, (slot, value) in bad.items():
        ids[t, slot] = value
    pool_d = torch.from_numpy(pool).cuda()
    pools = ops.Context.moe_pools(pool_d, hidden, inter, experts, offs["gate_off"], offs["up_off"], offs["down_off"])
    x_d, ids_d, wts_d = (torch.from_numpy(a).cuda() for a in (x, ids, wts))
    y = ctx.moe_experts_q4_0(pools, x_d, ids_d, wts_d, top_k, tokens)
    with pytest.raises(LevError) as e:
        ctx.sync()
    assert e.value.status == capi.BAD_DIMENSIONS
    y = y.cpu().numpy()
    g, u, d = (pool[offs["gate_off"]:], pool[offs["up_off"]:], pool[offs["down_off"]:])
    for t in sorted(set(bad) | set(range(0, tokens, max(1, tokens // 12)))):
        keep = [k for k in range(top_k) if 0 <= ids[t, k] < experts and np.count_nonzero(ids[t] == ids[t, k]) == 1]
        assert (len(keep) == top_k) == (t not in bad)
        ref = O.moe_experts_f64(g, u, d, hidden, inter, ids[t, keep], wts[t, keep], x[t])
        y32, _ = O.moe_experts_f32(g, u, d, hidden, inter, ids[t, keep], wts[t, keep], x[t])
        assert O.max_rel_err(y[t], ref["y"]) < max(TOL, 1.5 * O.max_rel_err(y32, ref["y"])), t
