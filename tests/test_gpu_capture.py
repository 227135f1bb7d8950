"""Motion checks in a caller's own stream capture (GPU): replays between direct
calls leave both sides' results and counts of FP64 decisions as they are alone."""

import numpy as np
import pytest

from plainmp_amd import synth
from support import product_cst

pytestmark = pytest.mark.gpu


def _edges(r, E, seed):
    import torch

    rng = np.random.default_rng(seed)
    a, b = (rng.uniform(r.lower, r.upper, size=(E, r.dof)) for _ in range(2))
    b = a + 0.3 * (b - a)
    return [torch.from_numpy(np.ascontiguousarray(x.T)).to("cuda") for x in (a, b)]


@pytest.mark.parametrize("n_direct,n_captured", [(64, 300), (300, 64), (64, 1500), (1500, 64), (1500, 2000)])
def test_replays_between_direct_calls(n_direct, n_captured):
    """Both sides of the bound between the two forms of the check (1,024 motions)."""
    import torch
    from plainmp_amd.ompl import BoxMotionValidator

    r = synth.panda_like(0)
    pc = product_cst(synth.Workload("capture", r, synth.mixed_primitives(12, 2)))
    pc.set_band(0.02)
    mv = BoxMotionValidator(pc, [0.05] * r.dof)
    stream = torch.cuda.Stream()
    sets, outs = {}, {}
    for name, E, seed in (("direct", n_direct, 1), ("captured", n_captured, 2)):
        sets[name] = _edges(r, E, seed)
        outs[name] = [torch.zeros(E, dtype=t, device="cuda") for t in (torch.uint8, torch.int32)]
    torch.cuda.synchronize()

    def call(name):
        (a, b), (v, n) = sets[name], outs[name]
        E = v.numel()
        mv._dev_check_motions(a.data_ptr(), b.data_ptr(), E, E, v.data_ptr(), n.data_ptr(), stream.cuda_stream)

    def result(name):
        stream.synchronize()
        return (mv.last_recheck_count(),) + tuple(x.cpu().numpy().tobytes() for x in outs[name])

    alone = {}
    for name in ("direct", "captured", "direct"):  # buffers and widths are in place before the capture
        call(name)
        alone[name] = result(name)
        assert alone[name][0] > 0
    assert alone["direct"][0] != alone["captured"][0]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        call("captured")
    ms = []
    for step in ("replay", "direct", "direct", "replay", "replay", "direct", "replay", "direct", "direct", "direct"):
        name = "direct" if step == "direct" else "captured"
        for x in outs[name]:
            x.fill_(7)
        torch.cuda.synchronize()
        if step == "direct":
            call(name)
        else:
            with torch.cuda.stream(stream):
                g.replay()
        assert result(name) == alone[name], step
        if step == "direct":
            ms.append(mv._dev_edge_kernel_ms(stream.cuda_stream))
    # the span of one launch, not of what ran between two (2 ms is ten times the longest here)
    assert all(0 < t < 2 for t in ms), ms
