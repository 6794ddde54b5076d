"""Status words cleared once for a step: failures of each of the step's calls are
reported at the vector and segment they happened, on a second step over stale
words too, on one stream and two, and the entry point refuses what it must."""
import ctypes as C

import numpy as np
import pytest

from provekv_amd import _lib as L
from provekv_amd import synth
from provekv_amd.pool import DeviceKVCache, TwoTierPlan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("two_streams", [False, True])
def test_step_reports_after_one_clear(ctx, two_streams):
    import torch
    layers, heads, prefix, agents = 2, 3, 9, [4, 1]
    plan = TwoTierPlan(ctx, layers, heads, 64, prefix, agents)
    bufs = plan.alloc()
    cache = DeviceKVCache(layers, heads, plan.tokens, 64)
    side = torch.cuda.Stream() if two_streams else None
    good = synth.corpus_tokens(7, layers, heads, plan.tokens, 64)
    names = ("pool_status", "shell_status", "pool_cstatus", "shell_cstatus")

    def step(x):
        plan.build_and_rehydrate(torch.from_numpy(x.reshape(-1).copy()).cuda(), bufs, cache, side=side)
        torch.cuda.synchronize()
        return {k: bufs[k].cpu().numpy().view(np.uint32).reshape(-1, 2) for k in names}

    for k, v in step(good).items():
        assert (v == 0xFFFFFFFF).all(), k
    bad = good.copy()
    bad[3, 1, 2, 0, 5] = np.nan              # pool: token 3, layer 1, head 2, K
    bad[prefix + 4, 0, 1, 1, 0] = np.inf     # agent 1's only token, layer 0, head 1, V
    st = step(bad)
    assert (st["pool_status"] != 0xFFFFFFFF).any(1).tolist() == [False, False, True, False]
    assert st["pool_status"][2, 0] >> 4 == 3 * heads + 2
    want = [False] * 8
    want[4 + 1] = True                       # agent 1, layer 0, V
    assert (st["shell_status"] != 0xFFFFFFFF).any(1).tolist() == want
    assert st["shell_status"][5].min() >> 4 == 1
    with pytest.raises(L.PkvError):
        plan.check(bufs, decode=False)
    for k, v in step(good).items():          # stale words are cleared again
        assert (v == 0xFFFFFFFF).all(), k


@pytest.mark.parametrize("two_streams", [False, True])
def test_step_without_status_words_raises(ctx, two_streams):
    """Status entries that are None: each call reports its own failure."""
    import torch
    plan = TwoTierPlan(ctx, 2, 3, 64, 9, [4, 1])
    bufs, cache = plan.alloc(), DeviceKVCache(2, 3, plan.tokens, 64)
    bufs.update({f"{tier}_{s}": None for tier in ("pool", "shell") for s in ("status", "dstatus", "cstatus")})
    side = torch.cuda.Stream() if two_streams else None
    good = torch.from_numpy(synth.corpus_tokens(7, 2, 3, plan.tokens, 64)).cuda()
    plan.build_and_rehydrate(good.view(-1), bufs, cache, side=side)
    plan.encode(good.view(-1), bufs)
    plan.decode(bufs)
    for token in (3, 9):   # the pool's, then a shell's
        bad = good.clone()
        bad[token, 1, 2, 0, 5] = float("nan")
        torch.cuda.synchronize()
        with pytest.raises(L.PkvError):
            plan.build_and_rehydrate(bad.view(-1), bufs, cache, side=side)
        with pytest.raises(L.PkvError):
            plan.encode(bad.view(-1), bufs)


def test_clear_and_run_refusals(ctx):
    import torch
    prof = ctx.turbo_profile(64, 4, 32, 42)
    st = torch.zeros(2, dtype=torch.int32, device="cuda")
    with pytest.raises(L.PkvError):
        ctx.clear_status([(st, 1)] * 9)
    ctx.clear_status([(st, 1)] * 8)
    assert (st.cpu() == -1).all()
    x = torch.ones(64, device="cuda")
    wire = torch.zeros(prof.blob_len(1), dtype=torch.uint8, device="cuda")
    from provekv_amd.device import contiguous_segment, segments
    segs = segments([contiguous_segment(0, 1, 64, 0)])
    with pytest.raises(ValueError):
        prof.encode_segments(x, segs, wire, status_cleared=True)

    def run(flags, status, reserved=0):
        op = L.SegmentsOp(1, 0, L.DT_F32, flags, x.data_ptr(), 64, segs.ctypes.data, wire.data_ptr(), wire.numel(),
                          0, 1, 1, 0, reserved, status)
        return L.lib().pkv_run_segments(ctx.ptr, prof.ptr, C.byref(op), None)
    assert run(2, st.data_ptr()) == run(1, None) == run(0, st.data_ptr(), 1)
    assert run(2, st.data_ptr()) != 0
    assert run(0, st.data_ptr()) == 0 and run(1, st.data_ptr()) == 0 and run(0, None) == 0
    torch.cuda.synchronize()


def test_blob_order_and_overlap(ctx):
    """Blobs may lie in any order in the wire; overlapping ones are refused, in
    table order or out of it."""
    import torch
    from oracle import oracle as O
    from provekv_amd.device import segments
    prof = ctx.turbo_profile(64, 4, 32, 42)
    n, blob = 3, prof.blob_len(3)
    x = torch.from_numpy(np.random.RandomState(3).randn(4 * n, 64).astype(np.float32)).cuda()
    wire = torch.zeros(5 * blob, dtype=torch.uint8, device="cuda")

    def encode(offsets):
        segs = segments([(k * n * 64, 0, 64, o, n, n) for k, o in enumerate(offsets)])
        prof.encode_segments(x.view(-1), segs, wire)
    for offsets in ([0, blob, 2 * blob, 3 * blob], [3 * blob + 1, 0, 2 * blob + 1, blob],
                    [7, 3 * blob, blob + 9, 4 * blob]):
        encode(offsets)
        w = wire.cpu().numpy()
        for k, o in enumerate(offsets):
            assert w[o:o + blob].tobytes() == O.turbo_encode_batch(x[k * n:(k + 1) * n].cpu().numpy(), 42)
    for offsets in ([0, blob - 1, 2 * blob, 3 * blob], [3 * blob, 0, 2 * blob, 2 * blob + 1], [0, blob, 0, 2 * blob]):
        with pytest.raises(L.PkvError):
            encode(offsets)


@pytest.mark.parametrize("dim,bits", [(64, 4), (64, 2), (128, 4), (128, 8)])
@pytest.mark.parametrize("radii", [0, 1])
@pytest.mark.parametrize("sizes,cap", [([1, 64, 3], 0), ([64, 2, 65], 0), ([128, 5, 1], 0), ([129, 2, 3], 0),
                                       ([2, 70, 1], 0), ([3, 128, 2, 64], 3)])
def test_words_stored_by_the_owning_workgroup(ctx, dim, bits, radii, sizes, cap):
    """Calls whose segments each fall to one workgroup store the words themselves,
    over stale ones; a call after an explicit clear marks them in memory.  Both report
    the same failures, at the first and last vectors and in the header."""
    import torch
    from provekv_amd.device import segments
    prof = ctx.turbo_profile(dim, bits, 32, 42)
    rows, off, elem = [], 0, 0
    for n in sizes:
        rows.append((elem, 0, dim, off, n, max(n, 1)))
        off += prof.blob_len(n, radii) + 3
        elem += n * dim
    segs = segments(rows)
    nseg = len(sizes)
    x = np.random.RandomState(dim).randn(elem).astype(np.float32)
    bad = x.copy()
    bad[rows[0][0] + (sizes[0] - 1) * dim + dim - 1] = np.nan          # last vector of the first segment
    bad[rows[-1][0]] = np.inf                                          # first of the last segment
    wire = torch.zeros(off, dtype=torch.uint8, device="cuda")
    out = torch.zeros(elem, device="cuda")

    def both(call):
        own = torch.zeros(2 * nseg, dtype=torch.int32, device="cuda")  # stale: a failure at vector 0
        ref = torch.zeros_like(own)
        call(own, False)
        ctx.clear_status([(ref, nseg)])
        call(ref, True)
        own, ref = (s.cpu().numpy().view(np.uint32).reshape(-1, 2) for s in (own, ref))
        assert np.array_equal(own, ref)
        return own

    def encode(v):
        t = torch.from_numpy(v).cuda()
        return both(lambda st, cl: prof.encode_segments(t, segs, wire, radii=radii, status=st, status_cleared=cl))

    def decode(w):
        return both(lambda st, cl: prof.decode_segments(w, segs, out, radii=radii, status=st, status_cleared=cl,
                                                        max_workgroups=cap))
    st = encode(bad)
    assert (st[0, 1] >> 4, st[-1, 1] >> 4) == (sizes[0] - 1, 0)
    assert (st[1:-1] == 0xFFFFFFFF).all() and (st[:, 0] == 0xFFFFFFFF).all()
    assert (encode(x) == 0xFFFFFFFF).all()
    assert (decode(wire) == 0xFFFFFFFF).all()
    w = wire.clone()
    w[rows[-1][3]] ^= 1                                                # header of the last segment
    plen = (prof.blob_len(2, radii) - prof.blob_len(1, radii))
    rw = dim // 2 if radii else 0                                      # the first radius, or the radii's minimum
    at = rows[0][3] + 38 + (sizes[0] - 1) * plen + rw
    w[at:at + 4] = torch.tensor([0, 0, 0xC0, 0x7F], dtype=torch.uint8, device="cuda")   # NaN
    st = decode(w)
    assert st[-1, 0] >> 4 == 0 and st[-1, 0] != 0xFFFFFFFF
    assert st[0, 1] >> 4 == sizes[0] - 1 and st[0, 0] == 0xFFFFFFFF
