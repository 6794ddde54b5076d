"""TwoTierPlan.digests(side=...) against work queued on `side` after the call:
the next bytes land in the hashed wires without a host wait, and the digests are
those of the first bytes -- eager and as graph replays."""
import pytest

from provekv_amd import synth
from provekv_amd.pool import TwoTierPlan

pytestmark = pytest.mark.gpu


def _setup(ctx):
    import torch
    plan = TwoTierPlan(ctx, 2, 8, 64, 200, [40, 24])
    x = [torch.from_numpy(synth.corpus_tokens(s, 2, 8, plan.tokens, 64).reshape(-1)).cuda() for s in (1, 2)]
    bufs, other = plan.alloc(), plan.alloc()
    plan.encode(x[0], bufs)
    plan.encode(x[1], other)
    first = {k: bufs[k].clone() for k in ("pool_wire", "shell_wire")}
    plan.digests(bufs)
    torch.cuda.synchronize()
    return plan, bufs, other, first, plan.digest_report(bufs)


def _spoil(bufs, first):
    import torch
    for k, v in first.items():
        bufs[k].copy_(v)
    for k in bufs:
        if k.endswith("digests"):
            bufs[k].zero_()
    torch.cuda.synchronize()


def _overwrite(bufs, other, side):
    import torch
    with torch.cuda.stream(side):
        for k in ("shell_wire", "pool_wire"):
            bufs[k].copy_(other[k])


@pytest.mark.parametrize("explicit", [False, True])
def test_side_work_after_the_call(ctx, explicit):
    import torch
    plan, bufs, other, first, want = _setup(ctx)
    side, own = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(3):
        _spoil(bufs, first)
        main = own if explicit else torch.cuda.current_stream()
        with torch.cuda.stream(main):
            torch.cuda._sleep(2_000_000)   # the digests start late
        plan.digests(bufs, stream=main if explicit else None, side=side)
        _overwrite(bufs, other, side)
        torch.cuda.synchronize()
        assert torch.equal(bufs["shell_wire"], other["shell_wire"])
        assert plan.digest_report(bufs) == want


def test_side_work_after_the_call_in_a_graph():
    import torch
    from provekv_amd.device import Context
    ctx = Context(0)   # its tables stay as captured
    plan, bufs, other, first, want = _setup(ctx)
    side, cap = torch.cuda.Stream(), torch.cuda.Stream()
    plan.digests(bufs, stream=cap, side=side)   # the table is on the device before the capture
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=cap):
        plan.digests(bufs, side=side)
        _overwrite(bufs, other, side)
        torch.cuda.current_stream().wait_stream(side)
    for _ in range(3):
        _spoil(bufs, first)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(bufs["shell_wire"], other["shell_wire"])
        assert plan.digest_report(bufs) == want
        plan.digests(bufs, side=side)   # the program's own eager work between replays
        torch.cuda.synchronize()
        assert plan.digest_report(bufs) != want
