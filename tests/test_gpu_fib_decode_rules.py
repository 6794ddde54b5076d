"""The fib matrix-core decode across its dispatch: with and without the table of
partial sums (decided by output bytes per value), direct and staged stores, one
half-tile per workgroup and a bounded grid that walks them; blobs of every size
around the 16-, 32- and 128-vector groups, at every byte alignment, with uniform
random indices (any table row) and with a rejected norm, into three layouts.
Bit for bit against the oracle; rows that must not be written stay.  The kinds of
a rejected vector, the bf16 stores at every exponent, and handles that share the
table."""
import numpy as np
import pytest

from oracle import oracle as O
from provekv_amd.device import SEG_DTYPE

pytestmark = pytest.mark.gpu

SEED = 42
CORRUPT, DECODE_NONFINITE = 5, 7   # status kinds
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
        want = (0xFFFFFFFF, (5 << 4) | CORRUPT) if n == 17 else (0xFFFFFFFF, 0xFFFFFFFF)
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


@pytest.mark.parametrize("fanout", [1, 2, 4])
def test_rejected_norm_and_overflowing_product(ctx, fanout):
    """A norm that is zero, negative or not finite is corrupt; a valid one whose
    products leave f32 is a decode that is not finite; the first one is reported."""
    import torch
    cb = (np.arange(1, 129, dtype=np.float32) * np.float32(1e36)).reshape(32, 4)
    prof = ctx.fib_profile_with_constants(cb, np.eye(64))
    blob = _blob(np.random.RandomState(9), 140)
    segs = np.array([(0, 0, 64, 0, 140, 140)], dtype=SEG_DTYPE)
    big, ok = 6e4, 1.0
    for at, norm, kind in ((3, 0.0, CORRUPT), (130, -1.0, CORRUPT), (17, np.inf, CORRUPT), (64, np.nan, CORRUPT),
                           (0, big, DECODE_NONFINITE), (139, big, DECODE_NONFINITE), (0, ok, None)):
        norms = np.ones(140, np.float16)
        norms[at] = norm
        for later in range(at + 1, 140, 7):   # failures after the first, of the other kind
            norms[later] = norm if kind is None else big if kind == CORRUPT else 0.0
        wire = np.frombuffer(blob, np.uint8).copy()
        wire[19:].reshape(-1, 12)[:, :2] = norms.view(np.uint8).reshape(-1, 2)
        out = torch.zeros(fanout * 140 * 64, device="cuda")
        status = torch.zeros(2, dtype=torch.int32, device="cuda")
        prof.decode_segments(torch.from_numpy(wire).cuda(), segs, out, status=status, fanout=fanout,
                             fanout_stride=140 * 64)
        st = status.cpu().numpy().view(np.uint32).tolist()
        assert st == [0xFFFFFFFF, 0xFFFFFFFF if kind is None else (at << 4) | kind], (at, norm)


def test_bf16_stores_at_every_exponent(ctx):
    """The bf16 conversion against torch's (round to nearest even): ties, their
    neighbours and carries into the exponent at every exponent from the f32
    subnormals (bf16 subnormals among them) to the overflow to infinity.  With an
    identity rotation a decode is a codebook entry times the power-of-two norm."""
    import torch
    rng = np.random.RandomState(2)
    low = [0, 1, 0x7FFF, 0x8000, 0x8001, 0xFFFF]
    mant = [(hi << 16) | lo for hi in (0, 1, 0x3E, 0x7E, 0x7F) for lo in low] + list(rng.randint(0, 1 << 23, 34))
    mant = np.array(mant, np.uint32)
    norms = (2.0 ** np.arange(-24, 16)).astype(np.float16)
    idx = [sum(((16 * half + b) % 32) << (5 * b) for b in range(16)).to_bytes(10, "little") for half in (0, 1)]
    pay = b"".join(v.tobytes() + i for v in norms for i in idx)
    n = 2 * len(norms)
    hdr = bytearray(_blob(rng, 1)[:19])
    hdr[10:14] = n.to_bytes(4, "little")
    blob = bytes(hdr) + pay
    wire = torch.from_numpy(np.frombuffer(blob, np.uint8).copy()).cuda()
    segs = np.array([(0, 0, 64, 0, n, n)], dtype=SEG_DTYPE)
    seen = set()
    for e in (-126, -100, -60, -20, 20, 60, 100, 112):
        pos = (np.uint32(e + 127) << np.uint32(23) | mant).view(np.float32)
        cb = np.concatenate([pos, -pos]).reshape(32, 4)
        want = O.fib_decode_batch(blob, cb, np.eye(64))
        seen |= set((want.view(np.uint32) >> 23 & 0xFF).reshape(-1).tolist())
        prof = ctx.fib_profile_with_constants(cb, np.eye(64))
        for fanout in (1, 2):
            out = torch.zeros(fanout * n * 64, dtype=torch.bfloat16, device="cuda")
            prof.decode_segments(wire, segs, out, fanout=fanout, fanout_stride=n * 64)
            ref = torch.from_numpy(want).reshape(-1).to(torch.bfloat16).view(torch.int16)
            assert torch.equal(out.cpu().view(fanout, -1).view(torch.int16), ref.expand(fanout, -1)), e
    assert seen == set(range(255))


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
