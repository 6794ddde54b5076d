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
