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


def launches_of(prog):
    """Nodes of the graph that a program replays (the program counts its operators as recorded): the graph is the first
    member of lev_program."""
    import ctypes as C
    hip = C.CDLL("libamdhip64.so")
    graph = C.cast(prog.handle, C.POINTER(C.c_void_p))[0]
    n = C.c_size_t()
    hip.hipGraphGetNodes.argtypes = [C.c_void_p, C.c_void_p, C.POINTER(C.c_size_t)]
    assert hip.hipGraphGetNodes(graph, None, C.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("case,launches", [("plain", 1), ("five", 2), ("alias", 2), ("short", 2), ("other", 2), ("behind", 2),
                                           ("vectors", 3), ("unaligned", 3), ("in place", 1)])
def test_what_a_recorded_norm_takes_along(case, launches):
    """How many kernels a recorded RMSNorm and the axpys behind it replay as: a norm of one aligned vector takes up to
    four of them along, as far as each adds a vector apart from the result to all of it."""
    from leviathan_amd import ops
    ctx = ops.Context(0, own_stream=True)
    n, vectors, off = 2816, 3 if case == "vectors" else 1, 1 if case == "unaligned" else 0
    src = torch.ones(vectors * n + 4, device="cuda")[off:off + vectors * n]
    y = src if case == "in place" else torch.zeros(vectors * n, device="cuda")
    adds = [torch.ones(n, device="cuda") for _ in range(5)]
    torch.cuda.synchronize()
    ctx.program_begin()
    ctx.rmsnorm(src, n, vectors, y=y)
    ctx.axpy(adds[0], y, 0.5, n)
    if case == "alias":
        ctx.axpy(y, y, 2.0, n)
    elif case == "short":
        ctx.axpy(adds[1], y, -1.5, n - 1)
    elif case == "other":
        ctx.axpy(y, adds[1], -1.5, n)
    elif case == "behind":
        ctx.gelu_up(y, n // 2, y=adds[1])
    else:
        ctx.axpy(adds[1], y, -1.5, n)
    if case == "five":
        for k in (2, 3, 4):
            ctx.axpy(adds[k], y, 0.25 * k, n)
    prog = ctx.program_end()
    assert prog.node_count() == (6 if case == "five" else 3)
    assert launches_of(prog) == launches
    prog.destroy()
    ctx.close()
