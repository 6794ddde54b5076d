"""Radii and angle bins of the encodes at the edges of their fast path: pairs on
octant lines, zero pairs and vectors, squares that underflow or overflow with and
without the rotation's scale, beside ordinary vectors in the same wave."""
import numpy as np
import pytest

from oracle import oracle as O
from provekv_amd.device import contiguous_segment, segments

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,bits", [(64, 4), (128, 4), (64, 3), (128, 2)])
@pytest.mark.parametrize("radii", [0, 1])
def test_edges_of_the_fast_path(ctx, dim, bits, radii):
    import torch
    rng = np.random.RandomState(dim + bits)
    rows = [np.zeros(dim), np.ones(dim)]
    one = np.zeros(dim)
    one[5] = 3.0
    rows += [one, -one, np.arange(dim) % 2]
    for e in (-149, -140, -126, -100, -60, -48, -47, -46, -33, -32, -31, -30, -29, -28, -27, -16, 16, 40, 58, 59, 60,
              61):
        rows.append(rng.randn(dim) * 2.0 ** e)
        rows.append(rng.choice([-1.0, 1.0, 2.0], dim) * 2.0 ** e)
    rows += list(rng.randn(40, dim))
    with np.errstate(over="ignore"):
        x = np.array(rows, np.float32)
    assert np.isfinite(x).all()
    prof = ctx.turbo_profile(dim, bits, 32, 42)
    for n in (len(x), 33, 1):
        wire = torch.zeros(prof.blob_len(n, radii), dtype=torch.uint8, device="cuda")
        prof.encode_segments(torch.from_numpy(x[:n].reshape(-1).copy()).cuda(),
                             segments([contiguous_segment(0, n, dim, 0)]), wire, radii=radii)
        assert wire.cpu().numpy().tobytes() == O.turbo_encode_batch(x[:n], 42, bits=bits, proj=32, radii_codec=radii)
