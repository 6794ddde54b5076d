"""The fib matrix-core decode across its dispatch: with and without the table of
partial sums (decided by output bytes per value), direct and staged stores, one
half-tile per workgroup and a bounded grid that walks them; blobs of every size
around the 16-, 32- and 128-vector groups, at every byte alignment, with uniform
random indices (any table row) and with a rejected norm, into three layouts.
Bit for bit against the oracle; rows that must not be written stay."""
import numpy as np
import pytest

from oracle import oracle as O
from provekv_amd.device import SEG_DTYPE

pytestmark = pytest.mark.gpu

SEED = 42
SIZES = [1, 0, 15, 16, 17, 33, 64, 127, 128, 129, 160, 257, 300]


def _blob(rng, n, bad=None):
    """A valid FB2 blob of n vectors with uniform random indices and norms."""
    pay = rng.randint(0, 256, (n, 12)).astype(np.uint8)
    pay[:, :2] = np.exp(rng.randn(n)).astype(np.float16).view(np.uint8).reshape(n, 2)
    if bad is not None:
        pay[bad, :2] = 0
    hdr = bytearray(O.fib_encode_batch(np.ones((1, 64), np.float32), *_constants())[:19])
    hdr[10:14] = int(n).to_bytes(4, "little")
    return bytes(hdr) + pay.tobytes()


def _constants():
    return O.fib_constants(SEED)


@pytest.mark.parametrize("dtype,fanout", [("f32", 1), ("f32", 2), ("f32", 3), ("f32", 4), ("bf16", 1), ("bf16", 6),
                                          ("bf16", 7), ("f16", 2)])
@pytest.mark.parametrize("heads", [0, 5, 32], ids=["rows", "heads5", "heads32"])
@pytest.mark.parametrize("cap", [0, 3])
def test_fib_decode_rules(ctx, dtype, fanout, heads, cap):
    import torch
    rng = np.random.RandomState(fanout + heads)
    cb, rot = _constants()
    prof = ctx.fib_profile(64, 4, 32, SEED)
    wire, rows, refs, off, elem = bytearray(), [], [], 0, 0
    for k, n in enumerate(SIZES):
        bad = 5 if n == 17 else None
        b = _blob(rng, n, bad)
        wire += bytes(k % 5) + b
        off = len(wire) - len(b)
        T = -(-n // heads) if heads else 0
        # rows back to back, or vector t * heads + h to head h, token t
        rows.append((elem, 64, T * 64, off, n, heads) if heads else (elem, 0, 64, off, n, max(n, 1)))
        ref = np.full((n, 64), 9.0, np.float32)
        good = [i for i in range(n) if i != bad]
        if good:
            keep = _rows(b, good)
            ref[good] = O.fib_decode_batch(keep, cb, rot)
        refs.append((elem, T, ref))
        elem += 64 * (heads * T if heads else n)
    segs = np.array(rows, dtype=SEG_DTYPE)
    tdt = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[dtype]
    stride = elem + 64
    out = torch.full((fanout * stride,), 9.0, dtype=tdt, device="cuda")
    status = torch.zeros(2 * len(segs), dtype=torch.int32, device="cuda")
    prof.decode_segments(torch.from_numpy(np.frombuffer(bytes(wire), np.uint8).copy()).cuda(), segs, out,
                         status=status, fanout=fanout, fanout_stride=stride, max_workgroups=cap)
    st = status.cpu().numpy().view(np.uint32).reshape(-1, 2)
    for k, n in enumerate(SIZES):
        want = (0xFFFFFFFF, (5 << 4) | st[k, 1] & 15) if n == 17 else (0xFFFFFFFF, 0xFFFFFFFF)
        assert tuple(st[k]) == want, (n, st[k])
    want = np.full(stride, 9.0, np.float32)
    for e, T, ref in refs:
        for i, row in enumerate(ref):
            o = e + (i // heads * 64 + i % heads * T * 64 if heads else i * 64)
            want[o:o + 64] = row
    want = torch.from_numpy(want).to(tdt)
    got = out.cpu().view(fanout, stride)
    bits = torch.int32 if dtype == "f32" else torch.int16
    for c in range(fanout):
        assert torch.equal(got[c].view(bits), want.view(bits)), c


def test_handles_of_equal_constants(ctx):
    """They share the table of partial sums, and the one that is left keeps it."""
    import torch
    cb, rot = _constants()
    blob = _blob(np.random.RandomState(3), 100)
    wire = torch.from_numpy(np.frombuffer(blob, np.uint8).copy()).cuda()
    segs = np.array([(0, 0, 64, 0, 100, 100)], dtype=SEG_DTYPE)
    want = O.fib_decode_batch(blob, cb, rot).view(np.uint32)
    profs = [ctx.fib_profile_with_constants(cb, rot) for _ in range(3)]
    for p in profs:
        out = torch.zeros(100 * 64, device="cuda")
        p.decode_segments(wire, segs, out)
        assert np.array_equal(out.cpu().numpy().view(np.uint32).reshape(100, 64), want)
        p.close()


def _rows(blob, idx):
    """The blob of the vectors `idx` of `blob`."""
    hdr = bytearray(blob[:19])
    hdr[10:14] = len(idx).to_bytes(4, "little")
    pay = np.frombuffer(blob[19:], np.uint8).reshape(-1, 12)[idx]
    return bytes(hdr) + pay.tobytes()
