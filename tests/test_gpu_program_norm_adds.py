"""GPU: a recorded RMSNorm with axpys behind it gives the bits of the operators called one by one, on every replay: the
chains that one kernel takes (lengths of one, two and four pieces a lane; one to five addends) and those that it may not
(an addend that overlaps the result, another length, another result, several vectors, an unaligned vector)."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("case", ["plain", "five", "alias", "short", "other", "vectors", "unaligned", "no weight", "in place"])
@pytest.mark.parametrize("n", [4, 1024, 2816, 5000, 16384])
def test_recorded_norm_and_adds(n, case):
    from leviathan_amd import ops
    ctx = ops.Context(0, own_stream=True)
    vectors = 3 if case == "vectors" else 1
    off = 1 if case == "unaligned" else 0
    flat = dev(O.normal(vectors * n + 4, n))
    x0 = flat[off:off + vectors * n].clone() if not off else None
    src = torch.empty(vectors * n + 4, device="cuda")[off:off + vectors * n]
    gain = None if case == "no weight" else dev((1 + 0.1 * O.normal(n, 2)).astype(np.float32))
    adds = [dev(O.normal(n, 10 + k)) for k in range(5)]
    y = src if case == "in place" else torch.empty(vectors * n, device="cuda")
    z = torch.zeros(n, device="cuda")

    def chain():
        ctx.rmsnorm(src, n, vectors, weight=gain, y=y)
        ctx.axpy(adds[0], y, 0.5, n)
        if case == "alias":
            ctx.axpy(y, y, 2.0, n)
        elif case == "short":
            ctx.axpy(adds[1], y, -1.5, n - 1 if n > 4 else 3)
        elif case == "other":
            ctx.axpy(y, z, -1.5, n)
        else:
            ctx.axpy(adds[1], y, -1.5, n)
        if case == "five":
            for k in (2, 3, 4):
                ctx.axpy(adds[k], y, 0.25 * k, n)

    def reset():
        src.copy_(flat[:vectors * n] if x0 is None else x0)
        z.zero_()
        torch.cuda.synchronize()

    reset()
    chain()
    ctx.sync()
    want, want_z = y.clone(), z.clone()
    torch.cuda.synchronize()
    ctx.program_begin()
    chain()
    prog = ctx.program_end()
    for _ in range(3):
        reset()
        if case != "in place":
            y.fill_(float("nan"))
            torch.cuda.synchronize()
        prog.run()
        ctx.sync()
        assert torch.equal(y.view(torch.int32), want.view(torch.int32))
        assert torch.equal(z, want_z)
    prog.close() if hasattr(prog, "close") else None
