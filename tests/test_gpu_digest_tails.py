"""Digests at the edges of the four-lane leaf pass and of the fused last pass:
ranges ending at every byte of a 16-byte piece, block and chunk, at every
alignment, counts of chunks around the 16-chunk tiles and the 64-value merge,
and tiers whose layers mix ranges that end in different passes."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("align", [0, 1, 2, 3])
def test_range_tails(ctx, align):
    import torch
    rng = np.random.RandomState(align)
    lens = (list(range(0, 130)) + [1007, 1008, 1009, 1023, 1024, 1025, 1039, 1040, 1041, 2047, 2048, 2049] +
            [16 * 1024 + d for d in (-17, -1, 0, 1, 15, 16, 17)] + [17 * 1024 + 33, 64 * 1024 - 1, 64 * 1024,
                                                                    64 * 1024 + 1, 80 * 1024 + 5])
    rg, off = [], align
    for n in lens:
        rg.append((off, n))
        off += n + (4 - n) % 4       # every range at this alignment
    buf = rng.randint(0, 256, off).astype(np.uint8)
    rg = np.array(rg, np.uint64)
    # the buffer ends with the last range's last byte
    buf = buf[:int(rg[-1].sum())]
    got = ctx.blake3_ranges(torch.from_numpy(buf).cuda(), rg).cpu().numpy()
    assert np.array_equal(got, O.blake3_ranges(buf, rg))


@pytest.mark.parametrize("layers", [1, 3, 11])
@pytest.mark.parametrize("big", [False, True], ids=["one_or_two_passes", "three_passes"])
def test_tier_layer_digests(ctx, layers, big):
    import torch
    rng = np.random.RandomState(layers)
    kib = [0, 1, 15, 16, 17, 30, 100, 255, 256, 257, 1000, 1024] + ([4096, 5000] if big else [])
    lens = [1024 * k + d for k in kib for d in (0, 7)]
    rng.shuffle(lens)
    rg, off = [], 3
    for n in lens:
        rg.append((off, n))
        off += n + 1
    buf = rng.randint(0, 256, off).astype(np.uint8)
    rg = np.array(rg, np.uint64)
    n = len(rg) // 2
    dbuf = torch.from_numpy(buf).cuda()
    blob = torch.zeros((n, 2, 32), dtype=torch.uint8, device="cuda")
    lay = torch.zeros((n, 32), dtype=torch.uint8, device="cuda")
    ref = O.blake3_ranges(buf, rg)
    for _ in range(2):   # the second call reuses the table and the scratch
        ctx.tier_digests(dbuf, rg, layers, blob, lay)
        assert np.array_equal(blob.cpu().numpy().reshape(-1, 32), ref)
        want = [O.layer_digest(i % layers, ref[2 * i].tobytes(), ref[2 * i + 1].tobytes()) for i in range(n)]
        assert [bytes(r) for r in lay.cpu().numpy()] == want
        blob.zero_()
        lay.zero_()
    # layer indexes of several digits, from digests alone
    kv = torch.from_numpy(np.tile(ref[:2], (1234, 1)).copy()).cuda()
    got = ctx.layer_digests(kv.view(1234, 2, 32), 100000).cpu().numpy()
    for i in (0, 9, 10, 99, 100, 999, 1000, 1233):
        assert bytes(got[i]) == O.layer_digest(i, ref[0].tobytes(), ref[1].tobytes())


@pytest.mark.parametrize("na,nb", [(4, 0), (0, 3), (5, 7), (1, 200)])
@pytest.mark.parametrize("side", [False, True])
def test_build_digests_two_buffers(ctx, na, nb, side):
    """Both tiers of a build by one launch sequence, from two buffers of their own,
    repeated on other bytes and after work queued on a side stream."""
    import torch
    rng = np.random.RandomState(na + nb)
    bufs, tiers, refs = [], [], []
    for n, size in ((na, 70000), (nb, 20000)):
        rg = np.array([(k * size + k % 3, int(rng.randint(0, size - 3))) for k in range(2 * n)],
                      np.uint64).reshape(-1, 2)
        bufs.append(torch.zeros(2 * n * size + 8, dtype=torch.uint8, device="cuda"))
        tiers.append((bufs[-1], rg, torch.zeros((n, 2, 32), dtype=torch.uint8, device="cuda"),
                      torch.zeros((n, 32), dtype=torch.uint8, device="cuda")))
    other = torch.cuda.Stream()
    for rep in range(3):
        new = [torch.from_numpy(rng.randint(0, 256, b.numel()).astype(np.uint8)).cuda() for b in bufs]
        torch.cuda.synchronize()
        if side:
            with torch.cuda.stream(other):
                torch.cuda._sleep(2_000_000)
                for b, x in zip(bufs, new):
                    b.copy_(x)
            torch.cuda.current_stream().wait_stream(other)
        else:
            for b, x in zip(bufs, new):
                b.copy_(x)
        ctx.build_digests(tiers, 3)
        for x, (_, rg, blob, lay) in zip(new, tiers):
            ref = O.blake3_ranges(x.cpu().numpy(), rg) if len(rg) else np.zeros((0, 32), np.uint8)
            assert np.array_equal(blob.cpu().numpy().reshape(-1, 32), ref), rep
            want = [O.layer_digest(i % 3, ref[2 * i].tobytes(), ref[2 * i + 1].tobytes()) for i in range(len(rg) // 2)]
            assert [bytes(r) for r in lay.cpu().numpy()] == want, rep


def test_build_digests_refuses_a_reserved_field(ctx):
    import ctypes as C
    import torch
    from provekv_amd import _lib as L
    buf, rg = torch.zeros(64, dtype=torch.uint8, device="cuda"), np.array([(0, 8), (8, 8)], np.uint64)
    blob, lay = (torch.zeros(n, dtype=torch.uint8, device="cuda") for n in (64, 32))
    for n in (0, 1):
        for reserved, ok in ((0, True), (1, False)):
            t = L.DigestTier(buf.data_ptr(), 64, rg.ctypes.data, blob.data_ptr(), lay.data_ptr(), n, reserved)
            rc = L.lib().pkv_blake3_build_digests(ctx.ptr, C.byref(t), 1, 3, None)
            assert (rc == 0) == ok
    torch.cuda.synchronize()


@pytest.mark.parametrize("chunks", [48 * 1024 - 1, 48 * 1024], ids=["four_lanes", "one_lane"])
def test_build_digests_at_the_first_pass_line(ctx, chunks):
    """The chunks of both tiers together decide the form of the first pass."""
    import torch
    rng = np.random.RandomState(5)
    data = rng.randint(0, 256, (28 << 20) + 8).astype(np.uint8)
    tiers, refs = [], []
    for k, n, total in ((0, 7, 28 * 1024), (1, 30, chunks - 28 * 1024)):
        cuts = np.linspace(0, total, 2 * n + 1).astype(np.int64)   # whole chunks, less 5 bytes at each end
        rg = np.stack([1024 * cuts[:-1] + k, 1024 * np.diff(cuts) - 5], 1).astype(np.uint64)
        refs.append(O.blake3_ranges(data, rg))
        tiers.append((torch.from_numpy(data).cuda(), rg, torch.zeros((n, 2, 32), dtype=torch.uint8, device="cuda"),
                      torch.zeros((n, 32), dtype=torch.uint8, device="cuda")))
    assert sum(-(-int(ln) // 1024) for _, rg, _, _ in tiers for _, ln in rg) == chunks
    ctx.build_digests(tiers, 3)
    for (_, rg, blob, lay), ref in zip(tiers, refs):
        assert np.array_equal(blob.cpu().numpy().reshape(-1, 32), ref)
        want = [O.layer_digest(i % 3, ref[2 * i].tobytes(), ref[2 * i + 1].tobytes()) for i in range(len(rg) // 2)]
        assert [bytes(r) for r in lay.cpu().numpy()] == want


def test_plan_digests_follow_the_side_stream(ctx):
    """TwoTierPlan.digests(side=...) hashes what the side stream had queued."""
    import torch
    from provekv_amd import synth
    from provekv_amd.pool import TwoTierPlan
    plan = TwoTierPlan(ctx, 2, 3, 64, 20, [3, 2])
    bufs = plan.alloc()
    side = torch.cuda.Stream()
    x = [torch.from_numpy(synth.corpus_tokens(s, 2, 3, plan.tokens, 64).reshape(-1)).cuda() for s in (1, 2)]
    torch.cuda.synchronize()

    def host():
        torch.cuda.synchronize()
        return plan.digest_report(bufs)
    want = []
    for v in x:
        plan.encode(v, bufs)
        plan.digests(bufs)
        want.append(host())
    assert want[0] != want[1]
    for k in (0, 1, 0):
        with torch.cuda.stream(side):
            torch.cuda._sleep(2_000_000)
        plan.encode(x[k], bufs, stream=side)
        plan.digests(bufs, side=side)
        assert host() == want[k]
