"""The edge kernel's own time (GPU) against events around the call: never more,
and most of it where the kernel is nearly all of the call."""

import numpy as np
import pytest

from plainmp_amd import synth
from support import product_cst

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("robot,E", [("fetch_like", 4000), ("panda_like", 40000)])
def test_kernel_time(robot, E):
    """A workgroup per motion and a wave per motion."""
    import torch
    from plainmp_amd.ompl import BoxMotionValidator

    r = getattr(synth, robot)(0)
    rng = np.random.default_rng(1)
    a, b = (torch.from_numpy(np.ascontiguousarray(rng.uniform(r.lower, r.upper, (E, r.dof)).T)).to("cuda")
            for _ in range(2))
    v, n = torch.empty(E, dtype=torch.uint8, device="cuda"), torch.empty(E, dtype=torch.int32, device="cuda")
    mv = BoxMotionValidator(product_cst(synth.Workload("clock", r, synth.mixed_primitives(16, 2))), [0.02] * r.dof)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    kernel, call = [], []
    for _ in range(9):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(stream)
        mv._dev_check_motions(a.data_ptr(), b.data_ptr(), E, E, v.data_ptr(), n.data_ptr(), stream.cuda_stream)
        e1.record(stream)
        kernel.append(mv._dev_edge_kernel_ms(stream.cuda_stream))
        e1.synchronize()
        call.append(e0.elapsed_time(e1))
    assert all(0 < k <= c for k, c in zip(kernel, call))
    assert np.median(kernel) >= 0.5 * np.median(call), (kernel, call)
