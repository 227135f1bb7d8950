"""The largest batches of the staged kernels (GPU): those whose launches would
pass 2^32 threads at the usual workgroup size."""

import numpy as np
import pytest

from cabi_robot import REVOLUTE, Balls, Context, Robot, i64

pytestmark = pytest.mark.gpu

PERIOD = 4096


@pytest.mark.parametrize("what", ["valid", "evaluate", "pairs"])
def test_a_billion_configurations(what):
    """2^30 + 70 configurations of one joint, 4,096 of them over and over: every
    one has the result it has in a batch of 4,096."""
    import torch

    robot = Robot([(-1, 0, -1, (0, 0, 0), (0, 0, 0)), (0, REVOLUTE, 0, (0, 0, 0.5), (0, 0, 1))],
                  [(1, (0.5, 0, 0), 0.1, 0)], 1)
    ctx = Context(robot, Balls([((0.4, 0.4, 0.5), 0.15)]))
    B = (1 << 30) + 70
    part = torch.from_numpy(np.random.default_rng(1).uniform(-3, 3, PERIOD)).to("cuda")
    q = part.repeat(B // PERIOD + 1)[:B].contiguous()

    def run(q):
        n = q.numel()
        out = [torch.full((n,), 9, dtype=torch.uint8 if what == "valid" else torch.float32, device="cuda")
               for _ in range(1 if what == "valid" else 2)]
        torch.cuda.synchronize()
        args = (ctx.ctx, ctx._ptr(q), i64(n), i64(n), ctx._ptr(out[0]))
        if what == "valid":
            ctx.ok(ctx.lib.pmp_is_valid_batch(*args, None))
        elif what == "evaluate":
            ctx.ok(ctx.lib.pmp_evaluate_batch(*args, ctx._ptr(out[1])))
        else:
            ctx.ok(ctx.lib.pmp_pair_clearance_batch(*args, ctx._ptr(out[1])))
        torch.cuda.synchronize()
        return out

    for got, ref in zip(run(q), run(part)):
        assert len(torch.unique(ref)) > 1
        whole = B // PERIOD * PERIOD
        same = got[:whole].view(-1, PERIOD) == ref
        assert bool(same.all()), int((~same).sum())
        assert torch.equal(got[whole:], ref[: B - whole])
    torch.cuda.empty_cache()
