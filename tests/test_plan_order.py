"""The order TwoTierPlan's calls leave between the calling stream and a `side`
stream, on the CPU: streams and events that only record what each queued
operation comes after."""
import contextlib

import pytest
import torch

from provekv_amd.pool import DeviceKVCache, TwoTierPlan


class Event:
    after = frozenset()

    def record(self, stream):
        self.after = stream.after


class Stream:
    """A queue whose operations come after everything in `after`."""

    def __init__(self, capturing=False, idle=False):
        self.after, self.capturing, self.idle = frozenset(), capturing, idle

    def run(self, name):
        before, self.after = self.after, self.after | {name}
        return before

    def record_event(self):
        ev = Event()
        ev.record(self)
        return ev

    def wait_event(self, event):
        self.after = self.after | event.after

    def wait_stream(self, other):
        self.wait_event(other.record_event())

    def query(self):
        assert not self.capturing, "a query invalidates a capture"
        return self.idle


class Profile:
    def __init__(self, ctx, name):
        self.ctx, self.name = ctx, name

    def payload_len(self, radii=0):
        return 12

    def _run(self, op, stream, status, status_cleared):
        before = self.ctx.log[f"{self.name} {op}"] = stream.run(f"{self.name} {op}")
        if status is None:
            assert not status_cleared
        elif status_cleared:
            assert self.ctx.cleared[status.data_ptr()] in before
        else:
            self.ctx.log["clear", status.data_ptr()] = before

    def encode_segments(self, *a, stream=None, status=None, status_cleared=False, **kw):
        self._run("encode", stream, status, status_cleared)

    def decode_segments(self, *a, stream=None, status=None, status_cleared=False, **kw):
        self._run("decode", stream, status, status_cleared)


class Context:
    def __init__(self):
        self.log, self.cleared = {}, {}

    def clear_status(self, buffers, stream=None):
        name = f"clear {len(self.log)}"
        before = stream.run(name)
        for status, _ in buffers:
            self.cleared[status.data_ptr()] = name
            self.log["clear", status.data_ptr()] = before

    def fib_profile(self, *a):
        return Profile(self, "pool")

    def turbo_profile(self, *a):
        return Profile(self, "shells")

    def build_digests(self, tiers, layers, stream):
        self.log["digests"] = stream.run("digests")


@pytest.fixture
def plan(monkeypatch):
    current = [Stream()]

    @contextlib.contextmanager
    def use(stream):
        current.append(stream)
        yield
        current.pop()

    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "stream", use)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: current[-1])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: current[-1].capturing)
    return TwoTierPlan(Context(), 2, 3, 64, 20, [3, 2])


@pytest.mark.parametrize("idle", [False, True])
@pytest.mark.parametrize("capturing", [False, True])
def test_digests_come_between_the_side_streams_work(plan, idle, capturing):
    """What was queued on `side` before the call comes before the digests, what
    is queued there afterwards (the next encode into the hashed wire) after."""
    bufs = plan.alloc("cpu")
    main, side = torch.cuda.current_stream(), Stream(idle=idle)
    main.capturing = capturing
    if not idle:
        side.run("encode before")
    plan.digests(bufs, side=side)
    assert idle or "encode before" in plan.ctx.log["digests"]
    assert "digests" in side.run("encode after")
    assert "digests" in main.run("next call")


@pytest.mark.parametrize("joined", [False, True])
def test_digests_on_an_explicit_capturing_stream(plan, joined):
    """The calling stream, not the current one, decides whether the call is part
    of a capture: `side` is then forked from it and never queried."""
    bufs = plan.alloc("cpu")
    main, side = Stream(capturing=True), Stream(capturing=joined)
    main.run("capture begins")
    waited = []
    side.wait_stream = lambda other: (waited.append(other), Stream.wait_stream(side, other))
    plan.digests(bufs, stream=main, side=side)
    assert waited == [main, main]   # the fork, then the order after the digests
    assert "capture begins" in side.after and "digests" in side.after


@pytest.mark.parametrize("two_streams", [False, True])
def test_step_clears_status_words_after_their_readers(plan, two_streams):
    """The words of a tier are cleared on the stream its rehydrate runs on: what
    that stream had queued (a read of the last step's words) comes before."""
    bufs, cache = plan.alloc("cpu"), DeviceKVCache(2, 3, plan.tokens, 64, device="cpu")
    main, side = torch.cuda.current_stream(), Stream() if two_streams else None
    readers = {"pool_cstatus": main, "shell_cstatus": side or main, "pool_status": main, "shell_status": main}
    for step in range(2):
        plan.build_and_rehydrate(None, bufs, cache, side=side)
        for name, stream in readers.items():
            if step:
                assert f"read {name}" in plan.ctx.log["clear", bufs[name].data_ptr()]
            stream.run(f"read {name}")


@pytest.mark.parametrize("two_streams", [False, True])
def test_calls_without_status_words(plan, two_streams):
    """Buffers whose status entries are None: every call checks itself (it raises
    the first failure), and nothing is cleared for it."""
    bufs, cache = plan.alloc("cpu"), DeviceKVCache(2, 3, plan.tokens, 64, device="cpu")
    bufs.update({f"{tier}_{s}": None for tier in ("pool", "shell") for s in ("status", "dstatus", "cstatus")})
    side = Stream() if two_streams else None
    main = torch.cuda.current_stream()
    plan.encode(None, bufs, stream=main)
    plan.decode(bufs, stream=main)
    plan.rehydrate(bufs, cache, stream=main)
    plan.build_and_rehydrate(None, bufs, cache, side=side)
    assert {"pool encode", "shells encode", "pool decode", "shells decode"} <= set(plan.ctx.log)
    assert not plan.ctx.cleared
