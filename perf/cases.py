"""The work a program hands this framework, as cases that can be timed and
compared: building a two-tier KV pool and rehydrating it, its encodes and
decodes one by one, long-context KV at head_dim 128, attention scores on
compressed keys, the digests of a build, and the codec adapters on host
buffers.

listed() are the cases, draw() one more of the same ranges, prepare() what the
program has in hand before the call, run() one pass, work() what a pass cannot
do without, exact() the same results in 64 bits.  Outputs are wire bytes,
digests and decodes whose bits the formats fix, so every case is compared
exactly.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from provekv_amd import _lib as L
from provekv_amd.codec import FibQuantAdapter, RadiiCompression, TurboQuantAdapter
from provekv_amd.device import SEG_DTYPE, contiguous_segment, default_context, segments
from provekv_amd.pool import DeviceKVCache, TwoTierPlan

SEED = 42                 # profile seed (constants), not the inputs'
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def listed():
    return [
        # one new token of every layer appended to one agent's hot shell: the
        # smallest call of a serving loop
        dict(name="token_append", kind="shell_encode", layers=24, heads=32, agents=1, tokens=1, lossy=False),
        # one layer's keys of a shared prefix through the fib adapter on host
        # buffers, there and back: the reference's own call
        dict(name="adapter_layer", kind="adapter", codec="fib", dim=64, n=25600, lossy=False),
        # a small pool on few layers and heads, ragged agents, bf16 cache, one
        # stream: a short conversation
        dict(name="step_small", kind="step", layers=6, heads=5, prefix=37, agents=3, tokens=11, ragged=True,
             lossy=True, cache="bf16", copies=1, side=False),
        # the headline workload: the SmolLM2-1.7B-shape pool of 8 agents built
        # and rehydrated into every agent's f32 cache
        dict(name="step_n8", kind="step", layers=24, heads=32, prefix=800, agents=8, tokens=28, ragged=False,
             lossy=False, cache="f32", copies=8, side=True),
        # the shared prefix alone: encode, and decode to one f32 copy
        dict(name="pool_encode", kind="pool_encode", layers=24, heads=32, tokens=800),
        dict(name="pool_decode", kind="pool_decode", layers=24, heads=32, tokens=800),
        # all agents' shells alone: lossless encode, and a lossy decode into
        # one bf16 cache from an odd number of tokens
        dict(name="shell_encode", kind="shell_encode", layers=24, heads=32, agents=8, tokens=28, lossy=False),
        dict(name="shell_decode", kind="shell_decode", layers=24, heads=32, agents=8, tokens=29, lossy=True,
             cache="bf16", copies=1),
        # long-context KV at head_dim 128 (Llama-3-8B's KV heads and context, a
        # quarter of its layers): bf16 in, log-quantized radii
        dict(name="long_encode", kind="kv_encode", dim=128, layers=8, heads=8, tokens=32768, input="bf16", lossy=True),
        dict(name="long_decode", kind="kv_decode", dim=128, layers=8, heads=8, tokens=32768, input="bf16", lossy=True),
        # attention logits of one decode step over the same keys, four query
        # heads to a KV head
        dict(name="long_scores", kind="scores", dim=128, blobs=64, tokens=32768, group=4, lossy=True),
        # the payload and layer digests of the headline build
        dict(name="digests_n8", kind="digests", layers=24, heads=32, prefix=800, agents=8, tokens=28, ragged=False,
             lossy=False),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "pool_encode", "pool_decode", "shell_encode", "shell_decode", "kv_encode", "kv_decode",
                       "scores", "digests", "adapter"])
    lossy = rng.random() < 0.5
    if kind in ("step", "digests"):
        c = dict(kind=kind, layers=rng.randint(2, 24), heads=rng.randint(2, 32), prefix=_log(rng, 4, 800),
                 agents=rng.randint(1, 8), tokens=_log(rng, 1, 64), ragged=rng.random() < 0.5, lossy=lossy)
        if kind == "step":
            c.update(cache=rng.choice(["f32", "bf16", "f16"]), copies=rng.randint(1, 8), side=rng.random() < 0.5)
        c["prefix"] = min(c["prefix"], 1024 - c["agents"] * c["tokens"])
        return c
    if kind in ("pool_encode", "pool_decode"):
        return dict(kind=kind, layers=rng.randint(1, 24), heads=rng.randint(1, 32), tokens=_log(rng, 5, 800))
    if kind in ("shell_encode", "shell_decode"):
        c = dict(kind=kind, layers=rng.randint(1, 24), heads=rng.randint(1, 32), agents=rng.randint(1, 8),
                 tokens=_log(rng, 1, 64), lossy=lossy)
        if kind == "shell_decode":
            c.update(cache=rng.choice(["f32", "bf16", "f16"]), copies=rng.randint(1, 4))
        return c
    if kind in ("kv_encode", "kv_decode"):
        dim = rng.choice([64, 128])
        layers, heads = rng.randint(1, 8), rng.randint(1, 8)
        return dict(kind=kind, dim=dim, layers=layers, heads=heads, tokens=_log(rng, 16, 32768),
                    input=rng.choice(["f32", "bf16"]), lossy=lossy)
    if kind == "scores":
        return dict(kind=kind, dim=rng.choice([64, 128]), blobs=rng.randint(1, 64), tokens=_log(rng, 16, 32768),
                    group=rng.randint(1, 8) if rng.random() < 0.5 else 4, lossy=lossy)
    codec = rng.choice(["fib", "turbo"])
    return dict(kind="adapter", codec=codec, dim=64 if codec == "fib" else rng.choice([64, 128]),
                n=_log(rng, 1, 32768), lossy=lossy and codec == "turbo")


# ---------------------------------------------------------------- inputs
def _gen(seed, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _kv(seed, lead, dim, device="cuda"):
    """K and V rows with per-channel key scales and outlier channels, values
    Gaussian: f32 [lead..., 2 (K|V), dim]; the scales belong to the trailing
    head of `lead`."""
    g = _gen(seed, device)
    x = torch.randn((*lead, 2, dim), generator=g, device=device)
    scale = torch.exp(0.5 * torch.randn((lead[-1], dim), generator=g, device=device))
    out = torch.rand((lead[-1], dim), generator=g, device=device).argsort(dim=-1) < max(2, dim // 32)
    x[..., 0, :] *= torch.where(out, scale * 8.0, scale)
    x[..., 1, :] *= 0.5
    return x


def _corpus(c, seed, tokens):
    """proveKV's per-token vectors, [tokens][layers][heads][K|V][64]."""
    return _kv(seed, (tokens, c["layers"], c["heads"]), 64).reshape(-1)


def _agent_tokens(c):
    """New tokens of each agent; ragged: unlike numbers around `tokens`."""
    if not c["ragged"]:
        return [c["tokens"]] * c["agents"]
    return [max(1, c["tokens"] + (a % 3 - 1) * (c["tokens"] // 3)) for a in range(c["agents"])]


def _plan(c, prefix, agents):
    return TwoTierPlan(default_context(), c["layers"], c["heads"], 64, prefix, agents, seed=SEED,
                       lossy=bool(c.get("lossy")))


def _status(segs):
    return torch.empty(2 * len(segs), dtype=torch.int32, device="cuda")


def _kv_plan(c):
    """One blob per (layer, K|V) over contiguous [layers][K|V][heads][tokens][dim]."""
    prof = default_context().turbo_profile(c["dim"], 4, 32, SEED)
    radii = L.RADII_LOG_U8 if c["lossy"] else L.RADII_F32
    n, nb = c["heads"] * c["tokens"], 2 * c["layers"]
    blob = prof.blob_len(n, radii)
    segs = segments([contiguous_segment(b * n * c["dim"], n, c["dim"], b * blob) for b in range(nb)])
    return prof, radii, n, nb, blob, segs


def _kv_input(c, seed):
    x = torch.randn((c["layers"], 2, c["heads"], c["tokens"], c["dim"]), generator=_gen(seed), device="cuda")
    g = _gen(seed + (1 << 32))
    shape = (c["layers"], c["heads"], 1, c["dim"])
    scale = torch.exp(0.7 * torch.randn(shape, generator=g, device="cuda"))
    out = torch.rand(shape, generator=g, device="cuda").argsort(dim=-1) < 4
    x[:, 0] *= torch.where(out, scale * 10.0, scale)
    return x.to(DTYPES[c["input"]]).view(-1)


def prepare(case, seed):
    c, kind = case, case["kind"]
    s = {"case": c}
    if kind == "step":
        agents = _agent_tokens(c)
        plan = s["plan"] = _plan(c, c["prefix"], agents)
        s["bufs"] = plan.alloc()
        s["cache"] = DeviceKVCache(c["layers"], c["heads"], plan.tokens, 64, dtype=DTYPES[c["cache"]],
                                   copies=c["copies"])
        s["corpus"] = _corpus(c, seed, plan.tokens)
        s["side"] = torch.cuda.Stream() if c["side"] else None
    elif kind == "digests":
        plan = s["plan"] = _plan(c, c["prefix"], _agent_tokens(c))
        s["bufs"] = plan.alloc()
        s["side"] = torch.cuda.Stream()
        plan.encode(_corpus(c, seed, plan.tokens), s["bufs"])
    elif kind in ("pool_encode", "pool_decode"):
        plan = s["plan"] = _plan(c, c["tokens"], [])
        s["corpus"] = _corpus(c, seed, c["tokens"])
        s["wire"] = torch.empty(plan.pool.wire_bytes, dtype=torch.uint8, device="cuda")
        s["status"] = _status(plan.pool.enc)
        if kind == "pool_decode":
            plan.fib.encode_segments(s.pop("corpus"), plan.pool.enc, s["wire"], status=s["status"])
            s["out"] = torch.empty(plan.pool.out_elems, dtype=torch.float32, device="cuda")
    elif kind in ("shell_encode", "shell_decode"):
        agents = [c["tokens"]] * c["agents"]
        plan = s["plan"] = _plan(c, 0, agents)
        s["corpus"] = _corpus(c, seed, sum(agents))
        s["wire"] = torch.empty(plan.shells.wire_bytes, dtype=torch.uint8, device="cuda")
        s["status"] = _status(plan.shells.enc)
        if kind == "shell_decode":
            plan.turbo.encode_segments(s.pop("corpus"), plan.shells.enc, s["wire"], radii=plan.radii,
                                       status=s["status"])
            cache = s["cache"] = DeviceKVCache(c["layers"], c["heads"], sum(agents), 64, dtype=DTYPES[c["cache"]],
                                               copies=c["copies"])
            s["segs"] = cache.segments_for(plan.shells, [a * c["tokens"] for a in range(c["agents"])])
    elif kind in ("kv_encode", "kv_decode"):
        prof, radii, n, nb, blob, segs = _kv_plan(c)
        s.update(prof=prof, radii=radii, segs=segs, x=_kv_input(c, seed), status=_status(segs),
                 wire=torch.empty(nb * blob, dtype=torch.uint8, device="cuda"))
        if kind == "kv_decode":
            prof.encode_segments(s.pop("x"), segs, s["wire"], radii=radii, status=s["status"])
            s["out"] = torch.empty(nb * n * c["dim"], dtype=torch.float32, device="cuda")
    elif kind == "scores":
        prof = s["prof"] = default_context().turbo_profile(c["dim"], 4, 32, SEED)
        radii = s["radii"] = L.RADII_LOG_U8 if c["lossy"] else L.RADII_F32
        b, t, d = c["blobs"], c["tokens"], c["dim"]
        blob = prof.blob_len(t, radii)
        enc = segments([contiguous_segment(i * t * d, t, d, i * blob) for i in range(b)])
        x = torch.randn((b, t, d), generator=_gen(seed), device="cuda")
        x *= torch.exp(0.7 * torch.randn((b, 1, d), generator=_gen(seed + (1 << 32)), device="cuda"))
        s["wire"] = torch.empty(b * blob, dtype=torch.uint8, device="cuda")
        s["status"] = _status(enc)
        prof.encode_segments(x.view(-1), enc, s["wire"], radii=radii, status=s["status"])
        s["segs"] = np.array([(i * t, 1, 1, i * blob, t, 1) for i in range(b)], dtype=SEG_DTYPE)
        s["queries"] = torch.randn((b * c["group"], d), generator=_gen(seed + (2 << 32)), device="cuda")
        s["prepared"] = torch.empty((b * c["group"], prof.prepared_len()), dtype=torch.float32, device="cuda")
        s["scores"] = torch.empty(c["group"] * b * t, dtype=torch.float32, device="cuda")
        s["qstatus"] = torch.empty(2, dtype=torch.int32, device="cuda")
    else:
        if c["codec"] == "fib":
            s["codec"] = FibQuantAdapter(64, 4, 32)
        else:
            s["codec"] = TurboQuantAdapter(c["dim"], 4, 32, RadiiCompression.Lossy if c["lossy"] else
                                           RadiiCompression.Lossless)
        s["x"] = np.ascontiguousarray(_kv(seed, (c["n"], 1), c["dim"], "cpu")[:, 0, 0].numpy())
    return s


# ---------------------------------------------------------------- one pass
def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "step":
        s["plan"].build_and_rehydrate(s["corpus"], s["bufs"], s["cache"], side=s["side"])
        return {"pool_wire": s["bufs"]["pool_wire"], "shell_wire": s["bufs"]["shell_wire"], "cache": s["cache"].buf}
    if kind == "digests":
        s["plan"].digests(s["bufs"], side=s["side"])
        return [s["bufs"][k] for k in ("pool_digests", "shell_digests", "pool_layer_digests", "shell_layer_digests")]
    if kind == "pool_encode":
        s["plan"].fib.encode_segments(s["corpus"], s["plan"].pool.enc, s["wire"], status=s["status"])
        return [s["wire"], s["status"]]
    if kind == "pool_decode":
        s["plan"].fib.decode_segments(s["wire"], s["plan"].pool.dec, s["out"], status=s["status"])
        return [s["out"], s["status"]]
    if kind == "shell_encode":
        s["plan"].turbo.encode_segments(s["corpus"], s["plan"].shells.enc, s["wire"], radii=s["plan"].radii,
                                        status=s["status"])
        return [s["wire"], s["status"]]
    if kind == "shell_decode":
        cache = s["cache"]
        s["plan"].turbo.decode_segments(s["wire"], s["segs"], cache.buf.view(-1), radii=s["plan"].radii,
                                        status=s["status"], fanout=cache.copies, fanout_stride=cache.copy_stride)
        return [cache.buf, s["status"]]
    if kind == "kv_encode":
        s["prof"].encode_segments(s["x"], s["segs"], s["wire"], radii=s["radii"], status=s["status"])
        return [s["wire"], s["status"]]
    if kind == "kv_decode":
        s["prof"].decode_segments(s["wire"], s["segs"], s["out"], radii=s["radii"], status=s["status"])
        return [s["out"], s["status"]]
    if kind == "scores":
        s["prof"].prepare_queries(s["queries"], s["prepared"], status=s["qstatus"])
        s["prof"].score_segments(s["wire"], s["segs"], s["prepared"], s["scores"], c["blobs"] * c["tokens"],
                                 radii=s["radii"], post_scale=1.0 / math.sqrt(c["dim"]), status=s["status"],
                                 nq=c["group"], query_stride=c["group"])
        return [s["scores"], s["prepared"], s["status"]]
    blob = s["codec"].encode_batch_compact(s["x"], SEED)
    return [np.frombuffer(blob, dtype=np.uint8), s["codec"].decode_batch_compact(blob, SEED)]


# ---------------------------------------------------------------- what a pass cannot do without
def _turbo_len(dim, lossy):
    return (dim // 2 + 8 if lossy else 2 * dim) + dim // 2 * 3 // 8 + 4


def work(case):
    c, kind = case, case["kind"]
    # operations per vector: the rotation (dense for fib, butterflies for
    # turbo), the 16 x 32 distances of a fib encode, the turbo encode's second
    # rotation and 32 sketch dots
    fib_enc, fib_dec = 2 * 64 * 64 + 16 * 32 * 8, 2 * 64 * 64

    def turbo_enc(d):
        return 2 * d * (int(math.log2(d)) + 1) + 4 * d + 64 * d

    def turbo_dec(d):
        return d * (int(math.log2(d)) + 3)
    if kind in ("step", "digests"):
        per = 2 * c["layers"] * c["heads"]
        n_pool, n_shell = per * c["prefix"], per * sum(_agent_tokens(c))
        wire = n_pool * 12 + n_shell * _turbo_len(64, c["lossy"])
        if kind == "digests":
            return {"bytes": wire, "flops": 0}
        size = 4 if c["cache"] == "f32" else 2
        return {"bytes": (n_pool + n_shell) * 64 * (4 + size * c["copies"]) + wire,
                "flops": n_pool * (fib_enc + fib_dec) + n_shell * (turbo_enc(64) + turbo_dec(64))}
    if kind in ("pool_encode", "pool_decode"):
        n = 2 * c["layers"] * c["heads"] * c["tokens"]
        return {"bytes": n * 268, "flops": n * (fib_enc if kind == "pool_encode" else fib_dec)}
    if kind in ("shell_encode", "shell_decode"):
        n = 2 * c["layers"] * c["heads"] * c["tokens"] * c["agents"]
        if kind == "shell_encode":
            return {"bytes": n * (256 + _turbo_len(64, c["lossy"])), "flops": n * turbo_enc(64)}
        size = 64 * (4 if c["cache"] == "f32" else 2) * c["copies"]
        return {"bytes": n * (size + _turbo_len(64, c["lossy"])), "flops": n * turbo_dec(64)}
    if kind in ("kv_encode", "kv_decode"):
        d = c["dim"]
        n = 2 * c["layers"] * c["heads"] * c["tokens"]
        if kind == "kv_encode":
            return {"bytes": n * (d * (4 if c["input"] == "f32" else 2) + _turbo_len(d, c["lossy"])),
                    "flops": n * turbo_enc(d)}
        return {"bytes": n * (4 * d + _turbo_len(d, c["lossy"])), "flops": n * turbo_dec(d)}
    if kind == "scores":
        n, d = c["blobs"] * c["tokens"], c["dim"]
        return {"bytes": n * (_turbo_len(d, c["lossy"]) + 4 * c["group"]), "flops": n * c["group"] * (3 * d + 64)}
    d, n = c["dim"], c["n"]
    plen = 12 if c["codec"] == "fib" else _turbo_len(d, c["lossy"])
    return {"bytes": 2 * n * (4 * d + plen),
            "flops": n * ((fib_enc + fib_dec) if c["codec"] == "fib" else (turbo_enc(d) + turbo_dec(d)))}


def tolerance(case):
    # wire bytes and digests are the format's; decodes and scores are fixed
    # sequences of f32 roundings, the same for every implementation of it
    return "exact"


# ---------------------------------------------------------------- the same in 64 bits
def _hadamard(d, device):
    h = torch.ones((1, 1), dtype=torch.float64, device=device)
    while h.shape[0] < d:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(d)


def _cos_sin(bins):
    th = bins.double() / 8.0 * (2.0 * math.pi) - math.pi
    return torch.cos(th), torch.sin(th)


def _bins(raw, count, bits):
    """`count` LSB-first fields of `bits` bits from byte rows."""
    b = ((raw.unsqueeze(-1) >> torch.arange(8, device=raw.device, dtype=torch.uint8)) & 1).flatten(-2)
    b = b[..., :count * bits].reshape(*b.shape[:-1], count, bits).to(torch.int64)
    return (b << torch.arange(bits, device=raw.device)).sum(-1)


def _turbo_fields(pay, d, lossy):
    """Radii (f64), angle bins and sketch signs (+-1) of payload rows."""
    p = d // 2
    if lossy:
        lo = pay[:, p:p + 4].contiguous().view(torch.float32).double()
        hi = pay[:, p + 4:p + 8].contiguous().view(torch.float32).double()
        r, at = torch.exp(lo + (hi - lo) * (pay[:, :p].double() / 255.0)), p + 8
    else:
        r, at = pay[:, :4 * p].contiguous().view(torch.float32).double(), 4 * p
    na = p * 3 // 8
    return r, _bins(pay[:, at:at + na], p, 3), _bins(pay[:, at + na:at + na + 4], 32, 1).double() * 2.0 - 1.0


def _turbo_rows(r, bins, signs):
    d = signs.numel()
    co, si = _cos_sin(bins)
    y = torch.stack([r * co, r * si], dim=-1).flatten(-2)
    return (y @ _hadamard(d, y.device)) * signs


def _turbo_decode(pay, d, lossy, signs):
    r, bins, _ = _turbo_fields(pay, d, lossy)
    return _turbo_rows(r, bins, signs)


def _turbo_through(x, lossy, signs):
    """Encode and decode of f64 rows."""
    y = (x * signs) @ _hadamard(x.shape[-1], x.device)
    a, b = y[..., 0::2], y[..., 1::2]
    r = torch.sqrt(a * a + b * b)
    bins = torch.floor((torch.atan2(b, a) + math.pi) / (2.0 * math.pi) * 8.0).long() % 8
    if lossy:
        lg = torch.log(r.clamp_min(2.0 ** -126))
        lo, hi = lg.amin(-1, keepdim=True).float().double(), lg.amax(-1, keepdim=True).float().double()
        code = torch.floor((lg - lo) / (hi - lo).clamp_min(2.0 ** -23) * 255.0 + 0.5).clamp(0, 255)
        r = torch.exp(lo + (hi - lo) * (code / 255.0))
    return _turbo_rows(r, bins, signs)


def _fib_rows(idx, norm, cb, rot):
    return (cb[idx].flatten(-2) @ rot) * norm[:, None]


def _fib_decode(pay, cb, rot):
    return _fib_rows(_bins(pay[:, 2:], 16, 5), pay[:, :2].contiguous().view(torch.float16).double()[:, 0], cb, rot)


def _fib_through(x, cb, rot):
    nrm = x.norm(dim=-1)
    rho = ((x / nrm[:, None]) @ rot.t()).reshape(-1, 16, 4)
    dist = (cb * cb).sum(-1) - 2.0 * (rho @ cb.t())
    return _fib_rows(dist.argmin(-1), nrm.float().half().double(), cb, rot)


def _fib_constants(prof, device="cuda"):
    cb, rot = prof.constants()
    return (torch.from_numpy(cb.reshape(32, 4)).double().to(device),
            torch.from_numpy(rot.reshape(prof.dim, prof.dim)).to(device))


def _turbo_signs(prof, device="cuda"):
    return torch.from_numpy(prof.constants()[0]).double().to(device)


def _payloads(wire, segs, hdr, plen):
    for g in segs:
        o, n = int(g["wire_offset"]) + hdr, int(g["n_vectors"])
        yield g, wire[o:o + n * plen].view(n, plen)


def exact(case, seed):
    c, kind = case, case["kind"]
    s = prepare(case, seed)
    if kind in ("pool_encode", "shell_encode", "kv_encode", "digests"):
        return None                       # bytes
    if kind == "pool_decode":
        plan = s["plan"]
        cb, rot = _fib_constants(plan.fib)
        return [torch.cat([_fib_decode(p, cb, rot) for _, p in _payloads(s["wire"], plan.pool.dec, 19, 12)]).view(-1),
                None]
    if kind == "shell_decode":
        plan, cache = s["plan"], s["cache"]
        signs = _turbo_signs(plan.turbo)
        out = torch.zeros(cache.buf.shape, dtype=torch.float64, device="cuda")
        for (name, layer, side, _, _), (_, p) in zip(plan.shells.blob_offsets,
                                                     _payloads(s["wire"], plan.shells.enc, 38,
                                                               _turbo_len(64, c["lossy"]))):
            rows = _turbo_decode(p, 64, c["lossy"], signs).view(c["tokens"], c["heads"], 64)
            t0 = int(name[5:]) * c["tokens"]
            out[:, layer, side, :, t0:t0 + c["tokens"]] = rows.transpose(0, 1)
        return [out, None]
    if kind == "kv_decode":
        signs = _turbo_signs(s["prof"])
        out = torch.empty(s["out"].shape, dtype=torch.float64, device="cuda")
        for g, p in _payloads(s["wire"], s["segs"], 38, _turbo_len(c["dim"], c["lossy"])):
            e = int(g["elem_offset"])
            out[e:e + p.shape[0] * c["dim"]] = _turbo_decode(p, c["dim"], c["lossy"], signs).view(-1)
        return [out, None]
    if kind == "scores":
        d, b, t, m = c["dim"], c["blobs"], c["tokens"], c["group"]
        signs, G = s["prof"].constants()
        signs = torch.from_numpy(signs).double().cuda()
        G = torch.from_numpy(G.reshape(32, d)).double().cuda()
        q = s["queries"].double()
        rq, gq = (q * signs) @ _hadamard(d, q.device), q @ G.t()
        out = torch.empty((m, b, t), dtype=torch.float64, device="cuda")
        for i, (_, p) in enumerate(_payloads(s["wire"], s["segs"], 38, _turbo_len(d, c["lossy"]))):
            r, bins, sg = _turbo_fields(p, d, c["lossy"])
            co, si = _cos_sin(bins)
            y = torch.stack([r * co, r * si], dim=-1).flatten(-2)
            k = slice(i * m, (i + 1) * m)
            out[:, i] = (rq[k] @ y.t() + math.sqrt(math.pi / 2.0) / 32.0 * (gq[k] @ sg.t())) / math.sqrt(d)
        return [out.view(-1), torch.cat([rq, gq], dim=1), None]
    if kind == "step":
        plan, cache = s["plan"], s["cache"]
        cb, rot = _fib_constants(plan.fib)
        signs = _turbo_signs(plan.turbo)
        x = s["corpus"].view(plan.tokens, c["layers"], c["heads"], 2, 64)
        out = torch.zeros(cache.buf.shape[1:], dtype=torch.float64, device="cuda")
        for layer in range(c["layers"]):
            for side in (0, 1):
                y = x[:, layer, :, side].double().reshape(-1, 64)
                cut = plan.prefix * c["heads"]
                rows = torch.cat([_fib_through(y[:cut], cb, rot), _turbo_through(y[cut:], c["lossy"], signs)])
                out[layer, side] = rows.view(plan.tokens, c["heads"], 64).transpose(0, 1)
        return {"pool_wire": None, "shell_wire": None, "cache": out.expand(cache.buf.shape)}
    x = torch.from_numpy(s["x"]).double()
    if c["codec"] == "fib":
        cb, rot = _fib_constants(s["codec"].build_quantizer(SEED), "cpu")
        return [None, _fib_through(x, cb, rot)]
    prof = default_context().turbo_profile(c["dim"], 4, 32, SEED)
    return [None, _turbo_through(x, c["lossy"], _turbo_signs(prof, "cpu"))]
