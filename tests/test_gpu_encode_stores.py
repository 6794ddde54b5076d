"""Payload stores of the encodes: blobs of every small size at every byte
alignment, guard bytes on both sides left alone, bytes equal to the oracle's."""
import numpy as np
import pytest

from oracle import oracle as O
from provekv_amd.device import segments

pytestmark = pytest.mark.gpu

SEED = 42
SIZES = [1, 2, 3, 5, 15, 16, 17, 31, 32, 33, 63, 64, 65, 128, 129, 257]


@pytest.mark.parametrize("codec,dim,bits,proj,mode,radii", [
    ("fib", 64, 0, 0, 0, 0), ("turbo", 64, 4, 32, 1, 0), ("turbo", 64, 4, 32, 1, 1), ("turbo", 128, 4, 32, 1, 0),
    ("turbo", 128, 4, 64, 1, 1), ("turbo", 64, 2, 32, 1, 1), ("turbo", 64, 1, 32, 0, 1), ("turbo", 128, 8, 32, 1, 0)])
@pytest.mark.parametrize("align", [0, 1, 2, 3])
def test_blob_bytes_and_guards(ctx, codec, dim, bits, proj, mode, radii, align):
    import torch
    rng = np.random.RandomState(dim + bits + align)
    if codec == "fib":
        prof, (cb, rot) = ctx.fib_profile(64, 4, 32, SEED), O.fib_constants(SEED)
        ref = lambda x: O.fib_encode_batch(x, cb, rot)                                       # noqa: E731
    else:
        prof = ctx.turbo_profile(dim, bits, proj, SEED, mode)
        ref = lambda x: O.turbo_encode_batch(x, SEED, bits=bits, proj=proj, mode=mode, radii_codec=radii)  # noqa: E731
    rows, off, elem = [], 16 + align, 0
    for n in SIZES:
        rows.append((elem, 0, dim, off, n, n))
        off += prof.blob_len(n, radii) + 5
        off += (align - off) % 4
        elem += n * dim
    x = rng.randn(elem // dim, dim).astype(np.float32)
    wire = torch.full((off + 16,), 0xA5, dtype=torch.uint8, device="cuda")
    prof.encode_segments(torch.from_numpy(x.reshape(-1)).cuda(), segments(rows), wire, radii=radii)
    got = wire.cpu().numpy()
    want = np.full(off + 16, 0xA5, np.uint8)
    for e, _, _, o, n, _ in rows:
        b = ref(x[e // dim:e // dim + n])
        want[o:o + len(b)] = np.frombuffer(b, np.uint8)
    assert np.array_equal(got, want)
