"""GPU: a recorded decode step, the shared expert's FFN, the MoE layer on its normalised residual and the norm and residuals
behind both, gives the bits of the operators called one by one on every replay, and replays as the launches that it is meant
to: the scores of the router go into the launch of the shared expert's gate/up, its down projection into the layer's, its norm
into the layer's, that norm and the residuals into the next layer's gate/up, unless what the one writes the other touches."""
import pytest
import torch

from tests.test_gpu_program_norm_adds import launches_of

pytestmark = pytest.mark.gpu


def q4_0(rows, n, g):
    nb = rows * n // 32
    w = torch.randint(0, 256, (nb, 18), dtype=torch.uint8, device="cuda", generator=g)
    w[:, :2] = (torch.randn(nb, 1, device="cuda", generator=g) / (4.6 * n ** 0.5)).abs().half().view(torch.uint8)
    return w.reshape(-1)


@pytest.mark.parametrize("case,launches", [("plain", 4), ("two layers", 7), ("two layers on the same buffers", 7), ("norm in front", 4), ("scores of the sum", 7), ("sum not added", 5), ("added twice", 5),
                                           ("part of the sum", 7), ("result is the sum", 5), ("gain is the sum", 5)])
@pytest.mark.parametrize("hidden,inter,shared,experts,top_k", [
    (2816, 704, 2112, 128, 8), (1024, 256, 512, 32, 2), (4096, 1536, 4096, 256, 8), (1152, 320, 1344, 60, 4), (2048, 768, 1024, 128, 8), (1280, 576, 640, 256, 8),
    (2432, 512, 1280, 60, 6), (3840, 896, 1344, 64, 8), (1024, 1984, 768, 32, 8), (3712, 320, 1408, 64, 4), (1024, 256, 64, 32, 2),
    (1536, 704, 832, 60, 6)])
def test_recorded_decode_step(hidden, inter, shared, experts, top_k, case, launches):
    from leviathan_amd import ops
    ctx = ops.Context(0, own_stream=True)
    g = torch.Generator(device="cuda").manual_seed(hidden + experts)
    normal = lambda *s: torch.randn(s, device="cuda", generator=g)
    gu = inter * (hidden // 32) * 18 * experts
    layers = []
    for _ in range(2 if "two" in case else 1):
        pool = torch.cat([q4_0(experts * inter, hidden, g), q4_0(experts * inter, hidden, g), q4_0(experts * hidden, inter, g)])
        layers.append(dict(
            pools=ops.Context.moe_pools(pool, hidden, inter, experts, 0, gu, 2 * gu), pool=pool, router=0.02 * normal(experts, hidden),
            norm=1 + 0.1 * normal(hidden), gate=q4_0(shared, hidden, g), up=q4_0(shared, hidden, g), down=q4_0(hidden, shared, g),
            post=1 + 0.1 * normal(hidden), post2=1 + 0.1 * normal(hidden),
            bufs=tuple(torch.empty(n, device="cuda") for n in (hidden, 2 * shared, shared, hidden)), y=torch.empty(1, hidden, device="cuda"),
            ids=torch.empty((1, top_k), dtype=torch.int32, device="cuda"), weights=torch.empty(1, top_k, device="cuda"),
            out=torch.empty(hidden, device="cuda")))
    if case == "two layers on the same buffers":
        layers[1]["bufs"], layers[1]["y"] = layers[0]["bufs"], layers[0]["y"]
    x0, before = normal(hidden), normal(2, hidden)

    def step():
        x = x0
        if case == "norm in front":
            ctx.rmsnorm(before[0], hidden, 1, weight=layers[0]["post"], y=x)
            ctx.axpy(before[1], x, 1.0, hidden)
        for m in layers:
            h, s = ctx.shared_expert_ffn(x, m["norm"], m["gate"], m["up"], m["down"], m["post"], hidden, shared, bufs=m["bufs"])
            ctx.moe_layer_q4_0(m["pools"], m["router"], (s if case == "scores of the sum" else h)[None], top_k, 1, y=m["y"], ids=m["ids"],
                               weights=m["weights"])
            out = s if case == "result is the sum" else m["out"]
            ctx.rmsnorm(m["y"], hidden, 1, weight=s if case == "gain is the sum" else m["post2"], y=out)
            if case == "part of the sum":
                ctx.axpy(s[4:], out, 1.0, hidden - 4)
            elif case not in ("sum not added", "result is the sum"):
                ctx.axpy(s, out, 0.5 if case == "added twice" else 1.0, hidden)
            if case == "added twice":
                ctx.axpy(s, out, 0.25, hidden)
            ctx.axpy(x, out, 1.0, hidden)
            x = m["out"]

    def results():
        ctx.sync()
        return [x0.clone()] + [t.clone() for m in layers for t in (*m["bufs"], m["y"], m["ids"], m["weights"], m["out"])]

    def wipe():
        for m in layers:
            for t in (*m["bufs"], m["y"], m["weights"], m["out"]):
                t.fill_(float("nan"))
            m["ids"].fill_(-1)
        torch.cuda.synchronize()

    wipe()
    step()
    want = results()
    torch.cuda.synchronize()
    ctx.program_begin()
    step()
    prog = ctx.program_end()
    for _ in range(3):
        wipe()
        prog.run()
        for a, b in zip(results(), want):
            assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    # (the layer's gate/up takes nothing along where the down projection's workgroups do not fit the chip beside its own)
    crowded = 2 * len(layers) - 1 + (case == "norm in front") if hidden == 4096 and case != "scores of the sum" else 0
    assert launches_of(prog) == launches + crowded
    prog.destroy()
    ctx.close()


@pytest.mark.parametrize("what,buffers,launches", [("norm", "own", 8), ("norm", "shared", 8), ("router", "own", 8), ("router", "shared", 11),
                                                   ("post", "own", 7), ("post", "shared", 7)])
def test_next_layer_reads_the_shared_sum(what, launches, buffers):
    """A layer's `shared` as a weight of the next layer's FFN: what that reads is the normalised sum, so the norm stays in
    front of it, whether the sum is needed behind it (buffers of its own) or the next down projection writes a new one (over the
    router, in one case, so that the second layer's kernels stay as they are).  As the weight of that layer's post norm the sum is
    read behind all of this, and the norm goes along."""
    from leviathan_amd import ops
    ctx = ops.Context(0, own_stream=True)
    hidden, inter, shared, experts, top_k = 2816, 704, 512, 32, 4
    g = torch.Generator(device="cuda").manual_seed(7)
    normal = lambda *s: torch.randn(s, device="cuda", generator=g)
    gu = inter * (hidden // 32) * 18 * experts
    layers = []
    for _ in range(2):
        pool = torch.cat([q4_0(experts * inter, hidden, g), q4_0(experts * inter, hidden, g), q4_0(experts * hidden, inter, g)])
        layers.append(dict(
            pools=ops.Context.moe_pools(pool, hidden, inter, experts, 0, gu, 2 * gu), pool=pool, router=0.02 * normal(experts, hidden),
            norm=1 + 0.1 * normal(hidden), gate=q4_0(shared, hidden, g), up=q4_0(shared, hidden, g), down=q4_0(hidden, shared, g),
            post=1 + 0.1 * normal(hidden), post2=1 + 0.1 * normal(hidden),
            bufs=[torch.empty(n, device="cuda") for n in (hidden, 2 * shared, shared, hidden)], y=torch.empty(1, hidden, device="cuda"),
            ids=torch.empty((1, top_k), dtype=torch.int32, device="cuda"), weights=torch.empty(1, top_k, device="cuda"),
            out=torch.empty(hidden, device="cuda")))
    first, second = layers
    if what == "router":                                  # (of its first expert)
        first["bufs"][3] = second["router"][0]
    else:
        second[what] = first["bufs"][3]
    if buffers == "shared":
        second["bufs"][3] = first["bufs"][3]
    x0 = normal(hidden)

    def step():
        x = x0
        for m in layers:
            h, s = ctx.shared_expert_ffn(x, m["norm"], m["gate"], m["up"], m["down"], m["post"], hidden, shared, bufs=tuple(m["bufs"]))
            ctx.moe_layer_q4_0(m["pools"], m["router"], h[None], top_k, 1, y=m["y"], ids=m["ids"], weights=m["weights"])
            ctx.rmsnorm(m["y"], hidden, 1, weight=m["post2"], y=m["out"])
            ctx.axpy(s, m["out"], 1.0, hidden)
            ctx.axpy(x, m["out"], 1.0, hidden)
            x = m["out"]

    def results():
        ctx.sync()
        return [t.clone() for m in layers for t in (*m["bufs"], m["y"], m["ids"], m["weights"], m["out"])]

    def wipe():
        for m in layers:
            for t in (*m["bufs"], m["y"], m["weights"], m["out"]):
                t.fill_(float("nan"))
            m["ids"].fill_(-1)
        torch.cuda.synchronize()

    wipe()
    step()
    want = results()
    torch.cuda.synchronize()
    ctx.program_begin()
    step()
    prog = ctx.program_end()
    for _ in range(3):
        wipe()
        prog.run()
        for a, b in zip(results(), want):
            assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    assert launches_of(prog) == launches
    prog.destroy()
    ctx.close()
