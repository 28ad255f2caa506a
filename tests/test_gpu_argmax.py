"""GPU: the argmax operator where its split into workgroups changes: one, several and the most workgroups a column, a
last one with a single logit, more columns than it has counters; the best in the last share, ties across shares."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [1, 63, 4096, 4097, 130001, 262144, 262145, 400003])
def test_argmax_splits(vocab):
    from leviathan_amd import ops
    ctx = ops.Context(0)
    for ncol in (1, 3, 16, 17):
        v = O.normal(ncol * vocab, vocab % 97 + ncol).reshape(ncol, vocab)
        v[0, vocab - 1] = 50.0                                  # the very last logit
        v[-1, vocab // 3] = v[-1, vocab // 2] = 60.0            # a tie: the lower index, margin zero
        d = torch.from_numpy(v).cuda()
        for _ in range(2):                                      # the counters are left as they were found
            idx, margin = ctx.argmax(d, vocab, ncol)
            ctx.sync()
            assert idx.cpu().tolist() == [O.argmax(row) for row in v], (vocab, ncol)
            if vocab > 1:
                assert margin.cpu().tolist() == [O.top_margin(row) for row in v], (vocab, ncol)
    ctx.close()
