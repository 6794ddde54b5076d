"""Scores at the edges of the table kernel: query counts around its groups of
four, two and one, blob sizes around its waves and staging rounds, every byte
alignment of a blob, and radii on both sides of the short expf's bound; bit for
bit against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from provekv_amd.device import segments

pytestmark = pytest.mark.gpu

SEED = 42


@pytest.mark.parametrize("dim,bits,proj,mode", [(64, 4, 32, 1), (128, 4, 32, 1), (64, 5, 32, 1), (128, 5, 32, 1),
                                                (64, 3, 32, 0), (128, 4, 32, 0)])
@pytest.mark.parametrize("lossy", [False, True])
@pytest.mark.parametrize("nq", [1, 2, 3, 4, 5, 6, 7, 9])
def test_score_groups(ctx, dim, bits, proj, mode, lossy, nq):
    import torch
    rng = np.random.RandomState(nq * dim + bits)
    prof = ctx.turbo_profile(dim, bits, proj, SEED, mode)
    blobs, rows, off, col = [], [], 0, 0
    for k, n in enumerate([1, 31, 33, 64, 65, 300]):
        x = rng.randn(n, dim).astype(np.float32)
        if k in (1, 5):          # some vectors past e^32, so that waves of both forms and mixed ones occur
            x[::7] *= np.float32(np.exp(36.0 if k == 5 else -36.0))
        b = O.turbo_encode_batch(x, SEED, bits=bits, proj=proj, mode=mode, radii_codec=int(lossy))
        off += k                 # every alignment of a blob
        rows.append((col, 1, 1, off, n, 1))
        blobs.append((off, b))
        off += len(b)
        col += n
    wire = np.zeros(off, np.uint8)
    for o, b in blobs:
        wire[o:o + len(b)] = np.frombuffer(b, np.uint8)
    segs = segments(rows)
    q = rng.randn(len(rows) * nq, dim).astype(np.float32)
    prep = prof.prepare_queries(torch.from_numpy(q).cuda())
    scores = torch.full((nq * col,), 7.0, dtype=torch.float32, device="cuda")
    status = torch.zeros(2 * len(rows), dtype=torch.int32, device="cuda")
    prof.score_segments(torch.from_numpy(wire).cuda(), segs, prep, scores, col, radii=int(lossy), status=status,
                        nq=nq, query_stride=nq)
    assert prof.score_status_error(status.cpu().numpy().view(np.uint32)) is None
    got = scores.cpu().numpy().reshape(nq, col)
    pref = O.turbo_prepare_queries(q, SEED, proj=proj, mode=mode)
    for k, (o, b) in enumerate(blobs):
        c, n = int(segs[k]["elem_offset"]), int(segs[k]["n_vectors"])
        ref = O.turbo_score(b, pref[k * nq:(k + 1) * nq], dim, SEED, bits=bits, proj=proj, mode=mode)
        assert np.array_equal(np.ascontiguousarray(got[:, c:c + n]).view(np.uint32),
                              np.ascontiguousarray(ref, np.float32).view(np.uint32)), (k, n)
