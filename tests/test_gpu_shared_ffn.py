"""GPU: the shared expert's FFN in one call against the CPU chain, at the edges of its fused gate/up kernel: a wave
per 256-value column task (8, 12 or 16 waves), rows that end inside a task, one and several row groups a workgroup,
sizes it leaves to the separate operators."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("hidden,inter,norms", [(64, 64, True), (2048, 4160, True), (2880, 2112, False), (3136, 192, True),
                                                (4096, 8256, True), (4160, 128, True)])
def test_shared_ffn_shapes(hidden, inter, norms):
    from leviathan_amd import ops
    ctx = ops.Context(0)
    gate, up = (O.synth_q4_0(s, inter * hidden // 32, 0.02) for s in (1, 2))
    down = O.synth_q4_0(3, hidden * inter // 32, 0.02)
    x = O.normal(hidden, 4)
    fn, pn = (O.normal(hidden, s, 1.0, 0.1) if norms else None for s in (5, 6))
    bufs = tuple(torch.full((n,), float("nan"), device="cuda") for n in (hidden, 2 * inter, inter, hidden))
    h, shared = ctx.shared_expert_ffn(dev(x), dev(fn) if norms else None, dev(gate), dev(up), dev(down),
                                      dev(pn) if norms else None, hidden, inter, bufs=bufs)
    ctx.sync()
    ref_h = O.rmsnorm_f64(x, fn, 1e-6)
    assert O.max_rel_err(h.cpu().numpy(), ref_h) < 1e-5
    hf = h.cpu().numpy()                                   # each stage on the device's own input to it
    gu, act = bufs[1].cpu().numpy(), bufs[2].cpu().numpy()
    assert O.max_rel_err(gu[:inter], O.q4_0_matvec_f64(gate, inter, hidden, hf)) < 1e-4
    assert O.max_rel_err(gu[inter:], O.q4_0_matvec_f64(up, inter, hidden, hf)) < 1e-4
    want = np.array([O.gelu_up_f64(float(a), float(b)) for a, b in zip(gu[:inter], gu[inter:])])
    assert O.max_rel_err(act, want) < 1e-5
    ref = O.rmsnorm_f64(O.q4_0_matvec_f64(down, hidden, inter, act).astype(np.float32), pn, 1e-6)
    assert O.max_rel_err(shared.cpu().numpy(), ref) < 1e-4
    ctx.close()


# name: offsets in floats, in one buffer, of x, h, gu, act and shared at hidden 2048, inter 1024
OVERLAPS = {
    "apart": (0, 2048, 4096, 6144, 7168),
    "act over x": (0, 2048, 4096, 1024, 7168),
    "act over h": (0, 2048, 4096, 2064, 7168),
    "act over gu": (0, 2048, 4096, 4096, 7168),
    "act over the up half": (0, 2048, 4096, 5120, 7168),
    "gu over x": (0, 4096, 0, 6144, 7168),
    "gu over a part of x": (0, 4096, 1984, 6144, 7168),
    "h over x": (0, 0, 4096, 6144, 7168),
    "h over a part of x": (0, 1024, 4096, 6144, 7168),
    "shared over x and h": (0, 2048, 4096, 6144, 1024),
}


@pytest.mark.parametrize("name", OVERLAPS)
def test_shared_ffn_buffers_that_overlap(name):
    """Buffers that share memory, as far as the operators one after the other allow it, give what those give: the same
    bits of `shared`, and of h where nothing is written over it."""
    from leviathan_amd import ops
    ctx = ops.Context(0)
    hidden, inter = 2048, 1024
    gate, up = (dev(O.synth_q4_0(s, inter * hidden // 32, 0.02)) for s in (1, 2))
    down = dev(O.synth_q4_0(3, hidden * inter // 32, 0.02))
    x0 = O.normal(hidden, 4)
    fn, pn = (dev(O.normal(hidden, s, 1.0, 0.1)) for s in (5, 6))
    sizes = (hidden, hidden, 2 * inter, inter, hidden)

    def buffers():
        pool = torch.full((9216,), float("nan"), device="cuda")
        parts = [pool[o:o + n] for o, n in zip(OVERLAPS[name], sizes)]
        parts[0].copy_(dev(x0))
        return parts
    x, h, gu, act, shared = buffers()
    ctx.rmsnorm(x, hidden, 1, weight=fn, y=h)
    want_h = h.clone()
    ctx.q4_0_gemv(gate, h, hidden, inter, y=gu)
    ctx.q4_0_gemv(up, h, hidden, inter, y=gu[inter:])
    ctx.gelu_up(gu, inter, y=act)
    ctx.q4_0_gemv(down, act, inter, hidden, y=shared)
    ctx.rmsnorm(shared, hidden, 1, weight=pn, y=shared)
    want = shared.clone()
    for _ in range(4):
        x, h, gu, act, shared = buffers()
        ctx.shared_expert_ffn(x, fn, gate, up, down, pn, hidden, inter, bufs=(h, gu, act, shared))
        assert torch.equal(shared, want)
        if name not in ("act over h", "shared over x and h"):
            assert torch.equal(h, want_h)
    ctx.close()
