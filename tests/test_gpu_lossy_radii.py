"""BlockLogU8 decode at the border of its short expf: the decode kernels take
the fused form while every vector of a wave has |mn|, |mx| <= 32 and the
general form otherwise, so waves wholly inside, wholly outside and mixed are
compared bit for bit with the oracle, at counts around the waves' groups."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SEED = 42


def _vectors(n, dim, scales):
    rng = np.random.RandomState(n * dim + len(scales))
    x = rng.randn(n, dim).astype(np.float64)
    return (x * np.exp(np.resize(np.asarray(scales, np.float64), n))[:, None]).astype(np.float32)


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("scales", [
    [0.0, 1.0, -3.0],                                   # inside
    [31.0, 31.9, 32.0, 32.1, 33.0, 0.0],                # the upper border, mixed with ordinary vectors
    [-26.0, -28.0, -29.5, -31.0, 0.0],                  # the lower border (small radii fall below the scale)
    [41.0, -50.0, -80.0],                               # outside
], ids=["inside", "upper", "lower", "outside"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 200, 513])
def test_lossy_decode_bits(dim, scales, n):
    from oracle import oracle as O
    from provekv_amd.codec import RadiiCompression, TurboQuantAdapter
    x = _vectors(n, dim, scales)
    ad = TurboQuantAdapter(dim, 4, 32, RadiiCompression.Lossy)
    blob = ad.encode_batch_compact(x, SEED)
    assert blob == O.turbo_encode_batch(x, SEED, radii_codec=1)
    ref = O.turbo_decode_batch(blob, dim, SEED)
    assert np.array_equal(ad.decode_batch_compact(blob, SEED).view(np.uint32), ref.view(np.uint32))
