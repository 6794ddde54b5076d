// pkv_capi.cpp -- host half of libpkv_hip.so: the C ABI declared in
// include/pkv_codec.h.  Owns contexts, profiles (constants resident on the
// device), segment-table validation and upload, kernel launches, and the
// host-buffer drop-ins for the adapters' encode_batch_compact /
// decode_batch_compact (proveKV/src/codec.rs:248-326, 513-569).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <memory>
#include <mutex>
#include <new>
#include <vector>

#include "pkv_blake3.h"
#include "pkv_internal.h"
#include "pkv_math.h"

using namespace pkv;

namespace {

constexpr int kSlots = 32;   // table slots per context (allocated on first use)

int hip_status(hipError_t e) {
    if (e == hipSuccess) return PKV_OK;
    if (e == hipErrorOutOfMemory) return PKV_ERR_OOM;
    return PKV_ERR_DEVICE;
}

#define HIP_TRY(expr)                          \
    do {                                       \
        hipError_t _e = (expr);                \
        if (_e != hipSuccess) return hip_status(_e); \
    } while (0)


// Streams that have launched work on a buffer since it was last known idle.
// No event is recorded per launch: when the buffer must be rewritten the
// library records an event on each of these streams at that moment (it
// follows all their earlier work) and the host waits on it.  Past kMaxUsers
// streams the device is synchronised instead.
constexpr int kMaxUsers = 4;
struct Users {
    hipStream_t s[kMaxUsers] = {};
    int n = 0;
    bool overflow = false;
    void add(hipStream_t st) {
        for (int i = 0; i < n; ++i)
            if (s[i] == st) return;
        if (n < kMaxUsers) s[n++] = st; else overflow = true;
    }
    // host waits until every recorded user is done
    int drain_host(hipEvent_t ev) {
        if (overflow) HIP_TRY(hipDeviceSynchronize());
        else
            for (int i = 0; i < n; ++i) {
                HIP_TRY(hipEventRecord(ev, s[i]));
                HIP_TRY(hipEventSynchronize(ev));
            }
        n = 0;
        overflow = false;
        return PKV_OK;
    }
};

struct Slot {
    void* dev = nullptr;         // segs | tile_start | status
    void* host = nullptr;        // pinned staging (keeps the uploaded table)
    size_t cap = 0;
    hipEvent_t ev = nullptr;     // drain helper
    hipEvent_t up_ev = nullptr;  // recorded on the uploading stream right after the table copy
    hipStream_t up_stream = nullptr;
    bool up_done = true;         // the host has seen up_ev complete
    Users users;                 // streams that read (or wrote status into) the slot
    hipEvent_t done_ev = nullptr;  // private slot: recorded after the launches of the call that took it
    bool done_recorded = false;
    bool shared = false;         // table only (no status words): reusable by equal tables
    bool digest = false;         // a table of digest ranges (+ its chaining-value scratch), and its plan:
    std::vector<uint32_t> b3_tiles;   // tiles per pass
    bool b3_quad = false;             // pass 0 on four lanes per chunk
    uint64_t b3_end[2] = {0, 0};      // last byte (exclusive) the ranges need of each buffer
    uint64_t b3_split = 0;
    uint32_t nseg = 0;
    uint64_t hash = 0;
};

struct NoallocScratch;   // pkv_decode_segments_noalloc's per-device scratch (below)

// A fib decode's table of partial sums, shared by the profiles of a device with
// the same constants; the last of them frees it.
struct FibPrefix {
    int device = 0;
    std::vector<float> key;   // what the sums are formed from: rows of f32(Pi), then the codebook
    float* d = nullptr;
    FibPrefix() = default;
    FibPrefix(const FibPrefix&) = delete;
    FibPrefix& operator=(const FibPrefix&) = delete;
    ~FibPrefix() {
        if (d) (void)hipFree(d);
    }
};

}  // namespace

struct pkv_ctx {
    int device = 0;
    std::mutex mu;
    Slot slots[kSlots];
    int next = 0;
    hipStream_t own_stream = nullptr;   // for the host-buffer entry points
    void* io_buf = nullptr;             // host-buffer entry points: in + out (device memory)
    size_t io_buf_cap = 0;
    NoallocScratch* noalloc = nullptr;  // this device's `scratch` (pkv_decode_segments_noalloc)
};

struct pkv_profile {
    pkv_ctx* ctx = nullptr;
    int kind = 0;
    uint32_t dim = 0;
    // the adapter parameters the profile was built from (the JSON codes'
    // checks need them); json_ok = 0 when unknown (fib with caller
    // constants) or when the adapter's bits - 1 angle width does not apply
    pkv_codec_params params{};
    int json_ok = 0;
    // turbo
    uint32_t bits = 0, pbits = 0, proj = 0, mode = 0;
    uint64_t seed = 0;
    std::vector<float> signs, qjl, cs, qb;
    std::vector<uint32_t> qa;
    float* d_signs = nullptr;
    float* d_qjl = nullptr;
    float* d_cs = nullptr;
    uint32_t* d_qa = nullptr;
    float* d_qb = nullptr;
    // fib
    uint32_t k = 0, n = 0, wbits = 0;
    std::vector<float> codebook, rot32t, rot32;
    std::vector<uint32_t> mf;
    std::vector<double> rot, rot_t, cb64;
    float* d_cb = nullptr;
    double* d_cb64 = nullptr;
    double* d_rot_t = nullptr;
    double* d_rot64 = nullptr;   // row-major f64 rotation (encode's exact redo)
    float* d_rot32t = nullptr;
    float* d_rot32 = nullptr;
    std::shared_ptr<FibPrefix> prefix;   // decode partial sums (matrix-core decode only), or none
    int mfma_decode = 0;
    uint32_t* d_mf = nullptr;
    float thr = 0.0f;
};

// ---- fixed scratch of pkv_decode_segments_noalloc: [segment table | tile
// prefix] of one call, for at most PKV_NOALLOC_MAX_SEGMENTS segments.  A
// file-scope device array: every GPU the library runs on holds its own copy,
// at its own address, from module load to process end.  In host code
// `scratch` names a host-side stand-in, never the device memory: host code
// uses only the address hipGetSymbolAddress returns for the current device.
namespace {
constexpr size_t pad256c(size_t v) { return (v + 255) & ~static_cast<size_t>(255); }
constexpr size_t kNaTileOff = pad256c(sizeof(pkv_seg) * PKV_NOALLOC_MAX_SEGMENTS);
constexpr size_t kNaBytes = kNaTileOff + sizeof(uint32_t) * (PKV_NOALLOC_MAX_SEGMENTS + 1);
}  // namespace

static __device__ __align__(256) uint8_t scratch[kNaBytes];

namespace {

constexpr int kMaxDevices = 64;

// One device's scratch: its address, and the event that orders the calls
// sharing it.  Every call waits on the device for the event (the previous
// call's kernel, on whatever stream and context it ran) before it rewrites
// the table, and records the event after its own launch; `mu` makes that
// wait / rewrite / launch / record sequence atomic among host threads.
struct NoallocScratch {
    uint8_t* ptr = nullptr;
    hipEvent_t ev = nullptr;
    std::mutex mu;
};
std::mutex g_scratch_mu;
NoallocScratch g_scratch[kMaxDevices];

// Set-up, once per device with that device current (the caller has made it
// current): the device address of `scratch` and the ordering event.
int noalloc_scratch(int device, NoallocScratch** out) {
    if (device < 0 || device >= kMaxDevices) return PKV_ERR_DEVICE;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    NoallocScratch& s = g_scratch[device];
    if (!s.ptr) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_status(e);
        if (!p) return PKV_ERR_DEVICE;
        hipEvent_t ev = nullptr;
        HIP_TRY(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
        s.ev = ev;
        s.ptr = static_cast<uint8_t*>(p);
    }
    *out = &s;
    return PKV_OK;
}

std::mutex g_logb_mu;
bool g_logb_done[kMaxDevices] = {};

// Once per device (the caller has made it current), before the first
// context there returns: measure the cheap-log bound table of the BlockLogU8
// encodes, check that the f16 matrix cores keep subnormal operands (the QJL
// acceptance bound counts on it) and that the encodes' short sqrt fix-up
// agrees with the correctly rounded sqrt on every input it is used on; a
// device that fails either check is refused.
int device_checks_once(int device, hipStream_t st) {
    std::lock_guard<std::mutex> lock(g_logb_mu);
    if (device >= 0 && device < kMaxDevices && g_logb_done[device]) return PKV_OK;
    float* d = nullptr;
    HIP_TRY(hipMalloc(&d, 4 * sizeof(float)));
    float got[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    hipError_t e = static_cast<hipError_t>(launch_logf_bound(st));
    if (e == hipSuccess) e = static_cast<hipError_t>(launch_f16_subnormal_probe(d, st));
    if (e == hipSuccess) e = static_cast<hipError_t>(launch_sqrt_check(reinterpret_cast<uint32_t*>(d + 2), st));
    if (e == hipSuccess) e = hipMemcpyAsync(got, d, sizeof got, hipMemcpyDeviceToHost, st);
    const hipError_t se = hipStreamSynchronize(st);   // queued work ends before `d` is freed
    if (e == hipSuccess) e = se;
    (void)hipFree(d);
    if (e != hipSuccess) return hip_status(e);
    if (got[0] != 0x1p-10f + 0x1p-14f || got[1] != 0x1p-10f) return PKV_ERR_UNSUPPORTED;
    if (f2u(got[2]) != 0u) return PKV_ERR_UNSUPPORTED;
    if (device >= 0 && device < kMaxDevices) g_logb_done[device] = true;
    return PKV_OK;
}

template <typename T>
int upload(T** dptr, const std::vector<T>& v) {
    size_t bytes = std::max<size_t>(v.size() * sizeof(T), sizeof(T));
    HIP_TRY(hipMalloc(reinterpret_cast<void**>(dptr), bytes));
    if (!v.empty()) HIP_TRY(hipMemcpy(*dptr, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return PKV_OK;
}

uint32_t turbo_plen(const pkv_profile* p, int radii) {
    uint32_t pairs = p->dim / 2;
    uint32_t rad = radii == PKV_RADII_LOG_U8 ? pairs + 8 : 4 * pairs;
    uint32_t ang = (pairs * p->pbits + 7) / 8;
    uint32_t sig = p->mode ? (p->proj + 7) / 8 : 0;
    return rad + ang + sig;
}

uint32_t fib_plen(const pkv_profile* p) { return 2 + ((p->dim / p->k) * p->wbits + 7) / 8; }

uint32_t hdr_len(const pkv_profile* p) { return p->kind == PKV_CODEC_TURBO ? 38u : 19u; }

bool mul_add_ok(uint64_t a, uint64_t b, uint64_t c, uint64_t* out) {
    uint64_t t;
    if (__builtin_mul_overflow(a, b, &t)) return false;
    if (__builtin_add_overflow(t, c, out)) return false;
    return true;
}

// Highest element index (exclusive) a segment touches in the f32 tensor.
bool seg_extent(const pkv_seg& s, uint32_t dim, uint64_t* end) {
    uint64_t n = s.n_vectors;
    if (n == 0) { *end = 0; return true; }
    uint64_t q = (n - 1) / s.group;
    uint64_t r = std::min<uint64_t>(s.group - 1, n - 1);
    uint64_t a, b;
    if (!mul_add_ok(q, s.stride_outer, 0, &a)) return false;
    if (!mul_add_ok(r, s.stride_inner, a, &b)) return false;
    if (__builtin_add_overflow(b, s.elem_offset, &b)) return false;
    if (__builtin_add_overflow(b, dim, &b)) return false;
    *end = b;
    return true;
}

// Checks a segment table against the tensor and wire extents and writes the
// prefix of workgroup tiles per segment into tile_start[0 .. nseg].
int validate_segments(const pkv_profile* p, int radii, bool encode, int dtype, const void* d_f32,
                      uint64_t f32_elems, const pkv_seg* segs, uint32_t nseg, const void* d_wire,
                      uint64_t wire_bytes, uint32_t* tile_start, uint32_t fanout = 1,
                      uint64_t fanout_stride = 0) {
    if (!segs || nseg == 0) return PKV_ERR_INVALID_ARG;
    if (!d_f32 || !d_wire) return PKV_ERR_INVALID_ARG;
    if (fanout == 0 || fanout_stride % 4 != 0) return PKV_ERR_INVALID_ARG;
    // encode reads 16 B (8 bf16 / 4 f32) per access; decode writes 4 values per access
    const uint32_t align = encode && dtype == PKV_BF16 ? 8u : 4u;
    uint64_t fan_extra;
    if (__builtin_mul_overflow(static_cast<uint64_t>(fanout - 1), fanout_stride, &fan_extra))
        return PKV_ERR_DIM_MISMATCH;
    if (reinterpret_cast<uintptr_t>(d_f32) % 16 != 0) return PKV_ERR_INVALID_ARG;
    const uint32_t plen = p->kind == PKV_CODEC_TURBO ? turbo_plen(p, radii) : fib_plen(p);
    const uint32_t hdr = hdr_len(p);
    uint64_t total = 0, prev_end = 0;
    bool in_order = true;   // every blob starts at or after the end of the one before it
    for (uint32_t i = 0; i < nseg; ++i) {
        const pkv_seg& s = segs[i];
        if (s.group == 0) return PKV_ERR_INVALID_ARG;
        if (s.n_vectors > MAX_SEG_VECTORS) return PKV_ERR_INVALID_ARG;
        if (encode && s.n_vectors == 0) return PKV_ERR_EMPTY_BATCH;
        if (s.elem_offset % align || s.stride_outer % align || s.stride_inner % align) return PKV_ERR_INVALID_ARG;
        uint64_t end;
        if (!seg_extent(s, p->dim, &end) || __builtin_add_overflow(end, fan_extra, &end) || end > f32_elems)
            return PKV_ERR_DIM_MISMATCH;
        uint64_t blob_end;
        if (!mul_add_ok(s.n_vectors, plen, hdr, &blob_end) ||
            __builtin_add_overflow(blob_end, s.wire_offset, &blob_end) || blob_end > wire_bytes)
            return PKV_ERR_CAPACITY;
        in_order &= s.wire_offset >= prev_end;
        prev_end = blob_end;
        uint64_t tiles = (static_cast<uint64_t>(s.n_vectors) + TILE - 1) / TILE;
        if (tiles == 0) tiles = 1;   // an empty blob still gets its header checked
        tile_start[i] = static_cast<uint32_t>(total);
        total += tiles;
        if (total > 0x7fffffffull) return PKV_ERR_INVALID_ARG;
    }
    tile_start[nseg] = static_cast<uint32_t>(total);
    if (encode && !in_order) {   // encoded blobs are written by different workgroups: no overlap
        std::vector<std::pair<uint64_t, uint64_t>> blobs(nseg);
        for (uint32_t i = 0; i < nseg; ++i)
            blobs[i] = {segs[i].wire_offset,
                        segs[i].wire_offset + hdr + static_cast<uint64_t>(segs[i].n_vectors) * plen};
        std::sort(blobs.begin(), blobs.end());
        for (size_t i = 1; i < blobs.size(); ++i)
            if (blobs[i].first < blobs[i - 1].second) return PKV_ERR_INVALID_ARG;
    }
    return PKV_OK;
}

// Hash of a table of 8-byte words (n a multiple of 8), four words a step: the
// byte-wise hash before it was most of a call's host time at a few hundred
// segments.  Equal hashes are confirmed by a comparison of the tables.
uint64_t table_hash(const void* p, size_t n) {
    constexpr uint64_t kMul = 0x9e3779b97f4a7c15ull;
    const auto* b = static_cast<const uint8_t*>(p);
    uint64_t h[4] = {n, 1, 2, 3};
    size_t i = 0;
    for (; i + 32 <= n; i += 32)
        for (int k = 0; k < 4; ++k) {
            uint64_t w;
            std::memcpy(&w, b + i + 8 * k, 8);
            h[k] = (h[k] ^ w) * kMul;
            h[k] ^= h[k] >> 29;
        }
    for (; i + 8 <= n; i += 8) {
        uint64_t w;
        std::memcpy(&w, b + i, 8);
        h[0] = (h[0] ^ w) * kMul;
        h[0] ^= h[0] >> 29;
    }
    return ((h[0] * kMul ^ h[1]) * kMul ^ h[2]) * kMul ^ h[3];
}

// Takes the next ring slot for `total` bytes (device table + pinned staging),
// waiting first for every stream that still uses it and growing it when
// needed.  The slot comes back private (not reusable as a shared table).
int acquire_slot(pkv_ctx* ctx, size_t total, Slot** out) {
    Slot& sl = ctx->slots[ctx->next];
    ctx->next = (ctx->next + 1) % kSlots;
    if (!sl.ev) HIP_TRY(hipEventCreateWithFlags(&sl.ev, hipEventDisableTiming));
    if (!sl.up_ev) HIP_TRY(hipEventCreateWithFlags(&sl.up_ev, hipEventDisableTiming));
    // the pinned copy and the device table are about to be rewritten: wait
    // for the slot's last use (a private slot's own event), or for all work
    // its streams had queued by now (a shared slot's users)
    if (sl.done_recorded && sl.users.n == 1 && !sl.users.overflow) {
        HIP_TRY(hipEventSynchronize(sl.done_ev));
        sl.users.n = 0;
    } else if (sl.users.n || sl.users.overflow) {
        int rc = sl.users.drain_host(sl.ev);
        if (rc) return rc;
    }
    sl.done_recorded = false;
    sl.shared = false;
    sl.digest = false;
    if (sl.cap < total) {
        if (sl.dev) HIP_TRY(hipFree(sl.dev));
        if (sl.host) HIP_TRY(hipHostFree(sl.host));
        sl.dev = sl.host = nullptr;
        sl.cap = 0;
        size_t cap = std::max<size_t>(total, 64 * 1024);
        HIP_TRY(hipMalloc(&sl.dev, cap));
        HIP_TRY(hipHostMalloc(&sl.host, cap, hipHostMallocDefault));
        sl.cap = cap;
    }
    *out = &sl;
    return PKV_OK;
}

// Stage the segment table + tile prefix (+ status words when the caller gave
// none) into a ring slot and copy it to the device on `stream`.  A table the
// device already holds in a table-only slot is reused as is: the kernels only
// read it, so a launch in flight on it does not matter, and repeated calls
// over the same segments (every step of a serving loop) upload nothing.  A
// caller on another stream than the one that uploaded the table waits (on the
// device) for that upload unless the host has already seen it complete.
// Tables up to this many tiles also get a per-tile segment map (one scalar
// load per workgroup instead of a binary search of the tile prefix).
constexpr uint64_t kMaxMapTiles = 1u << 20;

int stage_table(pkv_ctx* ctx, const pkv_seg* segs, uint32_t nseg, const std::vector<uint32_t>& tiles,
                bool need_status, hipStream_t stream, Slot** out_slot, SegDev** d_segs, uint32_t** d_tiles,
                uint32_t** d_status, uint32_t** d_map) {
    const size_t seg_bytes = sizeof(pkv_seg) * nseg;
    const size_t tile_bytes = sizeof(uint32_t) * (nseg + 1);
    const uint64_t ntiles = tiles[nseg];
    const bool with_map = ntiles <= kMaxMapTiles;
    const size_t tile_off = (seg_bytes + 255) & ~static_cast<size_t>(255);
    const size_t map_off = (tile_off + tile_bytes + 255) & ~static_cast<size_t>(255);
    const size_t map_bytes = with_map ? sizeof(uint32_t) * ntiles : 0;
    const size_t stat_off = (map_off + map_bytes + 255) & ~static_cast<size_t>(255);
    const size_t total = stat_off + (need_status ? sizeof(uint32_t) * 2 * nseg : 0) + 256;
    const uint64_t hash = table_hash(segs, seg_bytes);
    if (!need_status) {
        for (Slot& c : ctx->slots) {
            if (c.shared && c.nseg == nseg && c.hash == hash && std::memcmp(c.host, segs, seg_bytes) == 0) {
                if (!c.up_done && c.up_stream != stream) {
                    const hipError_t q = hipEventQuery(c.up_ev);
                    if (q == hipSuccess) c.up_done = true;
                    else if (q == hipErrorNotReady) HIP_TRY(hipStreamWaitEvent(stream, c.up_ev, 0));
                    else return hip_status(q);
                }
                auto* d = static_cast<uint8_t*>(c.dev);
                *d_segs = reinterpret_cast<SegDev*>(d);
                *d_tiles = reinterpret_cast<uint32_t*>(d + tile_off);
                *d_map = with_map ? reinterpret_cast<uint32_t*>(d + map_off) : nullptr;
                *d_status = nullptr;
                *out_slot = &c;
                return PKV_OK;
            }
        }
    }
    Slot* slp;
    int rc = acquire_slot(ctx, total, &slp);
    if (rc) return rc;
    Slot& sl = *slp;
    auto* h = static_cast<uint8_t*>(sl.host);
    std::memcpy(h, segs, seg_bytes);
    std::memcpy(h + tile_off, tiles.data(), tile_bytes);
    if (with_map) {
        auto* m = reinterpret_cast<uint32_t*>(h + map_off);
        for (uint32_t i = 0; i < nseg; ++i) std::fill(m + tiles[i], m + tiles[i + 1], i);
    }
    HIP_TRY(hipMemcpyAsync(sl.dev, sl.host, stat_off, hipMemcpyHostToDevice, stream));
    HIP_TRY(hipEventRecord(sl.up_ev, stream));
    sl.up_stream = stream;
    sl.up_done = false;
    sl.shared = !need_status;
    sl.nseg = nseg;
    sl.hash = hash;
    auto* d = static_cast<uint8_t*>(sl.dev);
    *d_segs = reinterpret_cast<SegDev*>(d);
    *d_tiles = reinterpret_cast<uint32_t*>(d + tile_off);
    *d_map = with_map ? reinterpret_cast<uint32_t*>(d + map_off) : nullptr;
    *d_status = need_status ? reinterpret_cast<uint32_t*>(d + stat_off) : nullptr;
    *out_slot = &sl;
    return PKV_OK;
}

// After the last launch of a call that read the slot.  A private slot (this
// call's status words or scratch) gets an event, so that taking it again
// waits for this call only, not for everything queued after it.
int finish_slot(Slot* sl, hipStream_t stream) {
    sl->users.add(stream);
    if (sl->shared) return PKV_OK;
    if (!sl->done_ev) HIP_TRY(hipEventCreateWithFlags(&sl->done_ev, hipEventDisableTiming));
    HIP_TRY(hipEventRecord(sl->done_ev, stream));
    sl->done_recorded = true;
    return PKV_OK;
}

TurboDev turbo_dev(const pkv_profile* p) {
    TurboDev t;
    t.signs = p->d_signs;
    t.qjl = p->d_qjl;
    t.cs = p->d_cs;
    t.qa = p->d_qa;
    t.qb = p->d_qb;
    t.seed = p->seed;
    t.dim = p->dim;
    t.pbits = p->pbits;
    t.proj = p->proj;
    t.mode = p->mode;
    return t;
}

FibDev fib_dev(const pkv_profile* p) {
    FibDev f;
    f.codebook = p->d_cb;
    f.codebook64 = p->d_cb64;
    f.rot_t = p->d_rot_t;
    f.rot64 = p->d_rot64;
    f.rot32t = p->d_rot32t;
    f.rot32 = p->d_rot32;
    f.prefix = p->prefix ? p->prefix->d : nullptr;
    f.mfma_decode = p->mfma_decode;
    f.mf = p->d_mf;
    f.thr = p->thr;
    f.dim = p->dim;
    f.k = p->k;
    f.n = p->n;
    f.bits = p->wbits;
    return f;
}

// Clears the status words (unless the caller has, or each workgroup stores its
// segment's) and launches the encode or decode kernel of the
// profile over a device-resident segment table (dsegs, dtiles: nseg + 1 tile
// prefix, nblocks tiles in all; segs: the host's copy).  Returns a hipError_t as int.
int launch_segments(const pkv_profile* prof, int radii, bool encode, int dtype, const void* d_f32,
                    const uint8_t* d_wire, const pkv_seg* segs, const SegDev* dsegs, const uint32_t* dtiles,
                    uint32_t nseg, uint32_t nblocks, uint32_t* status, bool per_vector, uint32_t fanout,
                    uint64_t fanout_stride, uint32_t grid_cap, hipStream_t stream, float* diag = nullptr,
                    const uint32_t* dmap = nullptr, bool cleared = false) {
    LaunchCommon lc;
    lc.segs = dsegs;
    lc.tile_start = dtiles;
    lc.tile_seg = dmap;
    lc.nseg = nseg;
    lc.status = status;
    lc.radii = static_cast<uint32_t>(radii);
    lc.plen = prof->kind == PKV_CODEC_TURBO ? turbo_plen(prof, radii) : fib_plen(prof);
    lc.in_bf16 = encode && dtype == PKV_BF16 ? 1u : 0u;
    lc.per_vector = per_vector ? 1u : 0u;
    lc.out_dtype = encode ? static_cast<uint32_t>(PKV_F32) : static_cast<uint32_t>(dtype);
    lc.fanout = fanout;
    lc.fanout_stride = fanout_stride;
    lc.grid_cap = grid_cap;
    lc.diag = diag;
    if (!cleared && prof->kind == PKV_CODEC_TURBO && nblocks == nseg) {   // as many tiles as segments
        const uint32_t most = turbo_own_vectors(lc, turbo_dev(prof), encode, nblocks);
        uint32_t i = 0;
        while (i < nseg && segs[i].n_vectors - 1u < most) ++i;   // 1 .. most vectors
        lc.own_status = i == nseg ? 1u : 0u;
    }
    if (!cleared && !lc.own_status) {
        const int e = launch_fill_u32(status, STATUS_NONE, 2ull * nseg, stream);
        if (e) return e;
    }
    if (prof->kind == PKV_CODEC_TURBO)
        return encode ? launch_turbo_encode(lc, turbo_dev(prof), d_f32, const_cast<uint8_t*>(d_wire), nblocks, stream)
                      : launch_turbo_decode(lc, turbo_dev(prof), d_wire, const_cast<void*>(d_f32), nblocks, stream);
    return encode ? launch_fib_encode(lc, fib_dev(prof), d_f32, const_cast<uint8_t*>(d_wire), nblocks, stream)
                  : launch_fib_decode(lc, fib_dev(prof), d_wire, const_cast<void*>(d_f32), nblocks, stream);
}

// Caller holds ctx->mu.
int copy_back(hipStream_t st, void* h1, const void* d1, size_t n1, void* h2, const void* d2, size_t n2);
int resolve_status(const pkv_profile* p, const uint32_t* st, uint32_t nseg, const pkv_seg* segs, pkv_error* err,
                   bool per_vector);

int run_segments_locked(pkv_ctx* ctx, const pkv_profile* prof, int radii, bool encode, int dtype,
                        const void* d_f32, uint64_t f32_elems, const pkv_seg* segs, uint32_t nseg,
                        const uint8_t* d_wire, uint64_t wire_bytes, uint32_t* d_status, hipStream_t stream,
                        bool per_vector = false, uint32_t fanout = 1, uint64_t fanout_stride = 0,
                        uint32_t grid_cap = 0, float* diag = nullptr, bool cleared = false) {
    if (!ctx || !prof) return PKV_ERR_INVALID_ARG;
    if (prof->kind == PKV_CODEC_TURBO && radii != PKV_RADII_F32 && radii != PKV_RADII_LOG_U8)
        return PKV_ERR_INVALID_ARG;
    if (prof->kind == PKV_CODEC_FIB) radii = PKV_RADII_F32;
    // dtype: encode input (f32 / bf16) or decode output (f32 / bf16 / f16)
    if (dtype != PKV_F32 && dtype != PKV_BF16 && (encode || dtype != PKV_F16)) return PKV_ERR_INVALID_ARG;
    if (encode && fanout != 1) return PKV_ERR_INVALID_ARG;
    std::vector<uint32_t> tiles(static_cast<size_t>(nseg) + 1);
    int rc = validate_segments(prof, radii, encode, dtype, d_f32, f32_elems, segs, nseg, d_wire, wire_bytes,
                               tiles.data(), fanout, fanout_stride);
    if (rc) return rc;
    HIP_TRY(hipSetDevice(ctx->device));
    if (!d_status) {
        // Without the caller's status words the call reports a rejected input
        // or blob itself (the reference's encode / decode return the error),
        // so it waits for its kernels; that wait cannot be captured.
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        HIP_TRY(hipStreamIsCapturing(stream, &cap));
        if (cap != hipStreamCaptureStatusNone) return PKV_ERR_UNSUPPORTED;
    }
    Slot* sl;
    SegDev* dsegs;
    uint32_t *dtiles, *dstat, *dmap;
    rc = stage_table(ctx, segs, nseg, tiles, d_status == nullptr, stream, &sl, &dsegs, &dtiles, &dstat, &dmap);
    if (rc) return rc;
    uint32_t* status = d_status ? d_status : dstat;
    const int e = launch_segments(prof, radii, encode, dtype, d_f32, d_wire, segs, dsegs, dtiles, nseg, tiles[nseg],
                                  status, per_vector, fanout, fanout_stride, grid_cap, stream, diag, dmap, cleared);
    int rc2 = finish_slot(sl, stream);
    if (e) return hip_status(static_cast<hipError_t>(e));
    if (rc2 || d_status) return rc2;
    // the private status words, read back into the slot's pinned mirror
    uint32_t* host_status = reinterpret_cast<uint32_t*>(static_cast<uint8_t*>(sl->host) +
                                                        (reinterpret_cast<uint8_t*>(dstat) -
                                                         static_cast<uint8_t*>(sl->dev)));
    rc = copy_back(stream, host_status, dstat, sizeof(uint32_t) * 2 * nseg, nullptr, nullptr, 0);
    if (rc) return rc;
    return resolve_status(prof, host_status, nseg, segs, nullptr, per_vector);
}

int run_segments(pkv_ctx* ctx, const pkv_profile* prof, int radii, bool encode, int dtype, const void* d_f32,
                 uint64_t f32_elems, const pkv_seg* segs, uint32_t nseg, const uint8_t* d_wire,
                 uint64_t wire_bytes, uint32_t* d_status, hipStream_t stream) {
    if (!ctx) return PKV_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(ctx->mu);
    return run_segments_locked(ctx, prof, radii, encode, dtype, d_f32, f32_elems, segs, nseg, d_wire, wire_bytes,
                               d_status, stream);
}

// Two device-to-host copies on `st`, then a wait for them and for all work
// queued before: the wait happens also when the second copy fails to enqueue,
// so no queued copy outlives the caller's (or this frame's) host buffers.
int copy_back(hipStream_t st, void* h1, const void* d1, size_t n1, void* h2, const void* d2, size_t n2) {
    hipError_t e = hipMemcpyAsync(h1, d1, n1, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess && n2) e = hipMemcpyAsync(h2, d2, n2, hipMemcpyDeviceToHost, st);
    const hipError_t se = hipStreamSynchronize(st);
    if (e == hipSuccess) e = se;
    return e == hipSuccess ? PKV_OK : hip_status(e);
}

int ensure_io_buf(pkv_ctx* ctx, size_t bytes) {
    if (ctx->io_buf_cap >= bytes) return PKV_OK;
    if (ctx->io_buf) HIP_TRY(hipFree(ctx->io_buf));
    ctx->io_buf = nullptr;
    ctx->io_buf_cap = 0;
    size_t cap = std::max<size_t>(bytes, 1 << 20);
    HIP_TRY(hipMalloc(&ctx->io_buf, cap));
    ctx->io_buf_cap = cap;
    return PKV_OK;
}

int resolve_status(const pkv_profile* p, const uint32_t* st, uint32_t nseg, const pkv_seg* segs, pkv_error* err,
                   bool per_vector = false) {
    for (uint32_t s = 0; s < nseg; ++s) {
        uint32_t w0 = st[2 * s], w1 = st[2 * s + 1];
        if (w0 == STATUS_NONE && w1 == STATUS_NONE) continue;
        // Fib batches of >= 4 vectors validate every input before encoding any
        // norm (codec.rs:592-610 precede 694-704); smaller ones and per-vector
        // calls fail at the first failing vector.  Without a segment table
        // (pkv_segments_status) a fib segment counts as a batch of >= 4.
        uint32_t pick;
        if (p->kind == PKV_CODEC_FIB && !per_vector && (!segs || segs[s].n_vectors >= 4))
            pick = w0 != STATUS_NONE ? w0 : w1;   // batch validation precedes norm encoding
        else
            pick = std::min(w0, w1);              // per-vector order
        uint32_t kind = pick & 15u;
        int code;
        switch (kind) {
            case KIND_NONFINITE_INPUT: code = PKV_ERR_NONFINITE_INPUT; break;
            case KIND_ZERO_NORM: code = PKV_ERR_ZERO_NORM; break;
            case KIND_NORM16: code = PKV_ERR_NORM_UNREPRESENTABLE; break;
            case KIND_NONFINITE_RADIUS:
            case KIND_NONFINITE_RESIDUAL: code = PKV_ERR_NONFINITE_CODE; break;
            default: code = PKV_ERR_CORRUPT_PAYLOAD; break;
        }
        if (err) {
            err->status = code;
            err->segment = static_cast<int32_t>(s);
            err->index = pick >> 4;
        }
        return code;
    }
    if (err) { err->status = PKV_OK; err->segment = -1; err->index = 0; }
    return PKV_OK;
}

uint16_t rd16(const uint8_t* b) { return static_cast<uint16_t>(b[0] | (b[1] << 8)); }
uint32_t rd32(const uint8_t* b) {
    return static_cast<uint32_t>(b[0]) | (static_cast<uint32_t>(b[1]) << 8) | (static_cast<uint32_t>(b[2]) << 16) |
           (static_cast<uint32_t>(b[3]) << 24);
}
uint64_t rd64(const uint8_t* b) { return rd32(b) | (static_cast<uint64_t>(rd32(b + 4)) << 32); }

// ---- legacy per-vector records: TQW1 (turbo-quant/src/wire.rs:44-98) and
// compact FB1 (fib-quant/src/codec.rs:81-92).  Every header field is fixed by
// the profile, so a record is a constant header followed by the payload the
// batched path writes (TQW1 always carries f32 radii).
uint32_t record_hdr_len(const pkv_profile* p) { return p->kind == PKV_CODEC_TURBO ? 46u : 11u; }

uint32_t record_plen(const pkv_profile* p) {
    return p->kind == PKV_CODEC_TURBO ? turbo_plen(p, PKV_RADII_F32) : fib_plen(p);
}

struct ByteWriter {
    HdrBytes h{};
    void put(uint32_t i, uint32_t v) { h.w[i >> 2] |= (v & 0xffu) << (8 * (i & 3)); }
    void put16(uint32_t i, uint32_t v) { put(i, v); put(i + 1, v >> 8); }
    void put32(uint32_t i, uint32_t v) { for (uint32_t k = 0; k < 4; ++k) put(i + k, v >> (8 * k)); }
    void put64(uint32_t i, uint64_t v) { put32(i, static_cast<uint32_t>(v)); put32(i + 4, static_cast<uint32_t>(v >> 32)); }
};

HdrBytes record_header(const pkv_profile* p) {
    ByteWriter b;
    if (p->kind == PKV_CODEC_TURBO) {
        b.put(0, 'T'); b.put(1, 'Q'); b.put(2, 'W'); b.put(3, '1');
        b.put16(4, 1);                       // VERSION
        b.put16(6, 1);                       // rotation flag: FastHadamard (power-of-two dims)
        b.put(8, 1);                         // VARIANT_TURBO_CODE
        b.put32(10, p->dim);
        b.put(14, p->pbits);
        b.put32(18, p->proj);                // profile.projections(), also without QJL
        b.put64(22, p->seed);
        b.put32(30, p->dim / 2);             // polar block count
        b.put32(34, p->mode ? p->proj : 0);  // QJL sign count
        b.put64(38, turbo_plen(p, PKV_RADII_F32));
    } else {
        b.put(0, 'F'); b.put(1, 'B'); b.put(2, '1');
        b.put(3, 1);                         // COMPACT_VERSION
        b.put(4, p->wbits);
        b.put32(5, p->dim / p->k);           // block_count
        b.put16(9, 2);                       // fp16 norm length
    }
    return b.h;
}

// Header of an n-vector batched blob (TQB1, wire.rs:267-346; FB2,
// codec.rs:195-320); the records are reshaped into blobs with f32 radii.
HdrBytes blob_header(const pkv_profile* p, uint64_t n, int radii = PKV_RADII_F32) {
    ByteWriter b;
    if (p->kind == PKV_CODEC_TURBO) {
        b.put(0, 'T'); b.put(1, 'Q'); b.put(2, 'B'); b.put(3, '1');
        b.put16(4, 1);
        b.put16(6, 1);
        b.put(8, 2);
        b.put32(10, p->dim);
        b.put(14, p->pbits);
        b.put(15, radii == PKV_RADII_LOG_U8 ? 1u : 0u);
        b.put32(18, p->proj);
        b.put64(22, p->seed);
        b.put32(30, static_cast<uint32_t>(n));
        b.put32(34, turbo_plen(p, radii));
    } else {
        b.put(0, 'F'); b.put(1, 'B'); b.put(2, '2');
        b.put(3, 1);
        b.put(4, p->wbits);
        b.put32(6, p->dim / p->k);
        b.put32(10, static_cast<uint32_t>(n));
        b.put16(15, 2);
        b.put16(17, fib_plen(p) - 2);
    }
    return b.h;
}

uint64_t pad256(uint64_t v) { return (v + 255) & ~static_cast<uint64_t>(255); }

}  // namespace

// =====================================================================
extern "C" {

const char* pkv_status_string(int status) {
    switch (status) {
        case PKV_OK: return "ok";
        case PKV_ERR_INVALID_ARG: return "invalid argument";
        case PKV_ERR_DIM_MISMATCH: return "dimension mismatch";
        case PKV_ERR_OOM: return "out of device memory";
        case PKV_ERR_DEVICE: return "HIP runtime error";
        case PKV_ERR_CORRUPT_PAYLOAD: return "corrupt payload";
        case PKV_ERR_UNSUPPORTED: return "unsupported profile";
        case PKV_ERR_NONFINITE_INPUT: return "non-finite input";
        case PKV_ERR_ZERO_NORM: return "zero norm";
        case PKV_ERR_NORM_UNREPRESENTABLE: return "norm cannot be represented as finite positive fp16";
        case PKV_ERR_EMPTY_BATCH: return "empty batch";
        case PKV_ERR_CAPACITY: return "buffer too small";
        case PKV_ERR_NONFINITE_CODE: return "non-finite radius or residual";
        case PKV_ERR_SCRATCH_LIMIT: return "more segments than the no-allocation scratch holds";
        default: return "unknown status";
    }
}

int pkv_device_available(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return 0;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, 0) != hipSuccess) return 0;
    return std::strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? 1 : 0;
}

int pkv_ctx_create(int device, pkv_ctx** out) {
    if (!out) return PKV_ERR_INVALID_ARG;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || device < 0 || device >= n) return PKV_ERR_DEVICE;
    hipDeviceProp_t prop;
    HIP_TRY(hipGetDeviceProperties(&prop, device));
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) return PKV_ERR_UNSUPPORTED;
    HIP_TRY(hipSetDevice(device));
    pkv_ctx* c = new (std::nothrow) pkv_ctx();
    if (!c) return PKV_ERR_OOM;
    c->device = device;
    hipError_t e = hipStreamCreateWithFlags(&c->own_stream, hipStreamNonBlocking);
    if (e != hipSuccess) { delete c; return hip_status(e); }
    int rc = noalloc_scratch(device, &c->noalloc);   // device is current
    if (!rc) rc = device_checks_once(device, c->own_stream);
    if (rc) { (void)hipStreamDestroy(c->own_stream); delete c; return rc; }
    *out = c;
    return PKV_OK;
}

void pkv_ctx_destroy(pkv_ctx* ctx) {
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    for (Slot& s : ctx->slots) {
        if (s.users.n || s.users.overflow) (void)s.users.drain_host(s.ev);
        if (s.ev) (void)hipEventDestroy(s.ev);
        if (s.up_ev) (void)hipEventDestroy(s.up_ev);
        if (s.done_ev) (void)hipEventDestroy(s.done_ev);
        if (s.dev) (void)hipFree(s.dev);
        if (s.host) (void)hipHostFree(s.host);
    }
    if (ctx->own_stream) {
        (void)hipStreamSynchronize(ctx->own_stream);
        (void)hipStreamDestroy(ctx->own_stream);
    }
    if (ctx->io_buf) (void)hipFree(ctx->io_buf);
    delete ctx;
}

// Operands of the QJL matrix-core path: each dot is three products on the f16
// matrix cores, Gh xh + Gh xl + Gl xh, with G = Gh + Gl + eG split here
// (round to nearest even: Gh = f16(G), Gl = f16(G - Gh)) and the scaled
// residual x = xh + xl + ex split in the kernel.  Per tile t (16 projections
// on v_mfma_f32_16x16x32_f16 at head_dim 128, 32 on v_mfma_f32_32x32x16_f16 at
// head_dim 64), K step s and half (0: Gh, 1: Gl):
//   qa[((t * 4 + s) * 2 + half) * 64 + lane] (4 words: 8 f16, j = 0..7) =
//       G[16t + lane % 16][16 B(lane / 16) + 64 (s / 2) + 8 (s % 2) + j]
//           (head_dim 128; B = (0, 2, 1, 3): the encode's residual layout)
//       G[32t + lane % 32][32 (lane / 32) + 8s + j]      (head_dim 64)
//   qb[((t * nb + r) * 64 + lane) * 2 + {0, 1}] = (a_j, b_j) of the projection
//       j in accumulator register r: 16t + 4 (lane / 16) + r (128),
//       32t + 8 (r / 4) + 4 (lane / 32) + r % 4 (64);
// a sign is kept when |acc| > a_j xn + b_j, xn >= |x| (derivation at
// turbo_encode_qjl_kernel):
//   a_j = ((7.1 d + 30) u |g_j| + 1.001 * 2^-25 sqrt(d)) (1 + 2^-10),
//   b_j = (1.002 * 2^-24 sqrt(d) |g_j| + d 2^-49) (1 + 2^-10), u = 2^-24,
// each rounded up to f32.
static void turbo_qjl_mfma_constants(pkv_profile* p) {
    const uint32_t dim = p->dim;
    const bool wide = dim == 128;
    const uint32_t tp = wide ? 16 : 32;                 // projections per tile
    const uint32_t tiles = p->proj / tp, nb = wide ? 4 : 16;
    p->qa.assign(static_cast<size_t>(tiles) * 4 * 2 * 64 * 4, 0u);
    p->qb.assign(static_cast<size_t>(tiles) * nb * 64 * 2, 0.0f);
    const double u = std::ldexp(1.0, -24), d = static_cast<double>(dim), sd = std::sqrt(d);
    auto up = [](double v) {
        float f = static_cast<float>(v);
        if (static_cast<double>(f) < v) f = std::nextafter(f, std::numeric_limits<float>::infinity());
        return f;
    };
    for (uint32_t t = 0; t < tiles; ++t)
        for (uint32_t lane = 0; lane < 64; ++lane) {
            const uint32_t row = wide ? 16 * t + lane % 16 : 32 * t + lane % 32;
            const uint32_t rq = lane / 16, blk = ((rq & 1) << 1) | (rq >> 1);
            for (uint32_t st = 0; st < 4; ++st)
                for (uint32_t j = 0; j < 8; ++j) {
                    const uint32_t col = wide ? 16 * blk + 64 * (st / 2) + 8 * (st % 2) + j : 32 * (lane / 32) + 8 * st + j;
                    const float g = p->qjl[static_cast<size_t>(row) * dim + col];
                    const uint16_t gh = f32_to_f16(g);
                    const uint16_t gl = f32_to_f16(g - f16_to_f32(gh));   // g - gh is exact in f32
                    const size_t w0 = (((t * 4 + st) * 2 + 0) * 64 + lane) * 4 + j / 2;
                    const size_t w1 = (((t * 4 + st) * 2 + 1) * 64 + lane) * 4 + j / 2;
                    p->qa[w0] |= static_cast<uint32_t>(gh) << (16 * (j & 1));
                    p->qa[w1] |= static_cast<uint32_t>(gl) << (16 * (j & 1));
                }
            for (uint32_t r = 0; r < nb; ++r) {
                const uint32_t j = wide ? 16 * t + 4 * (lane / 16) + r : 32 * t + 8 * (r / 4) + 4 * (lane / 32) + r % 4;
                double g2 = 0.0;
                for (uint32_t c = 0; c < dim; ++c) {
                    const double g = p->qjl[static_cast<size_t>(j) * dim + c];
                    g2 += g * g;
                }
                const double gn = std::sqrt(g2) * (1.0 + std::ldexp(1.0, -40));   // >= |g_j|
                const double safety = 1.0 + std::ldexp(1.0, -10);
                const double aj = ((7.1 * d + 30.0) * u * gn + 1.001 * std::ldexp(sd, -25)) * safety;
                const double bj = (1.002 * std::ldexp(sd, -24) * gn + d * std::ldexp(1.0, -49)) * safety;
                p->qb[((t * nb + r) * 64 + lane) * 2 + 0] = up(aj);
                p->qb[((t * nb + r) * 64 + lane) * 2 + 1] = up(bj);
            }
        }
}

static int turbo_profile_common(pkv_ctx* ctx, uint32_t dim, uint32_t bits, uint32_t proj, uint64_t seed, int mode,
                                const float* signs, const float* qjl, pkv_profile** out) {
    if (!ctx || !out) return PKV_ERR_INVALID_ARG;
    *out = nullptr;
    // reference validity (turbo-quant/src/turbo.rs:148-164)
    if (dim == 0 || dim % 2 != 0) return PKV_ERR_INVALID_ARG;
    if (mode != PKV_TURBO_POLAR_ONLY && mode != PKV_TURBO_POLAR_WITH_QJL) return PKV_ERR_INVALID_ARG;
    if (mode == PKV_TURBO_POLAR_WITH_QJL ? (bits < 2 || bits > 16) : (bits < 1 || bits > 16))
        return PKV_ERR_INVALID_ARG;
    if (mode == PKV_TURBO_POLAR_WITH_QJL && proj == 0) return PKV_ERR_INVALID_ARG;
    // what the kernels implement
    const uint32_t pbits = mode == PKV_TURBO_POLAR_WITH_QJL ? bits - 1 : bits;
    if (dim != 64 && dim != 128) return PKV_ERR_UNSUPPORTED;
    if (pbits > 8) return PKV_ERR_UNSUPPORTED;
    if (mode == PKV_TURBO_POLAR_WITH_QJL && proj != 32 && proj != 64) return PKV_ERR_UNSUPPORTED;
    pkv_profile* p = new (std::nothrow) pkv_profile();
    if (!p) return PKV_ERR_OOM;
    p->ctx = ctx;
    p->kind = PKV_CODEC_TURBO;
    p->dim = dim;
    p->bits = bits;
    p->pbits = pbits;
    p->proj = proj;   // written to TQB1 bytes 18..21 in every mode (wire.rs:311, 343)
    p->mode = static_cast<uint32_t>(mode);
    p->seed = seed;
    p->params.kind = PKV_CODEC_TURBO;
    p->params.dim = dim;
    p->params.bits = bits;
    p->params.projections = proj;
    p->params.seed = seed;
    p->json_ok = mode == PKV_TURBO_POLAR_WITH_QJL;   // TurboQuantAdapter::decode: PolarQuantizer(bits - 1)
    const uint32_t qrows = mode == PKV_TURBO_POLAR_WITH_QJL ? proj : 0;
    if (signs) {
        p->signs.assign(signs, signs + dim);
        if (qrows) p->qjl.assign(qjl, qjl + static_cast<size_t>(qrows) * dim);
    } else {
        make_turbo_constants(dim, qrows, seed, p->signs, p->qjl);
    }
    // (cos, sin) of every dequantized angle, host libm (polar.rs:91-95, 312-313)
    const uint32_t levels = 1u << pbits;
    p->cs.resize(2 * levels);
    const float PI = 3.14159265358979323846f;
    for (uint32_t i = 0; i < levels; ++i) {
        float th = (static_cast<float>(i) / static_cast<float>(levels)) * (2.0f * PI) - PI;
        p->cs[2 * i] = std::cos(th);
        p->cs[2 * i + 1] = std::sin(th);
    }
    int rc = hip_status(hipSetDevice(ctx->device));
    if (!rc) rc = upload(&p->d_signs, p->signs);
    if (!rc) rc = upload(&p->d_qjl, p->qjl);
    if (!rc) rc = upload(&p->d_cs, p->cs);
    if (!rc && (dim == 64 || dim == 128) && qrows) {
        turbo_qjl_mfma_constants(p);
        rc = upload(&p->d_qa, p->qa);
        if (!rc) rc = upload(&p->d_qb, p->qb);
    }
    if (rc) { pkv_profile_destroy(p); return rc; }
    *out = p;
    return PKV_OK;
}

int pkv_turbo_profile_create(pkv_ctx* ctx, uint32_t dim, uint32_t bits, uint32_t projections, uint64_t seed,
                             int mode, pkv_profile** out) {
    return turbo_profile_common(ctx, dim, bits, projections, seed, mode, nullptr, nullptr, out);
}

int pkv_turbo_profile_create_with_constants(pkv_ctx* ctx, uint32_t dim, uint32_t bits, uint32_t projections,
                                            uint64_t seed, int mode, const float* signs, const float* qjl,
                                            pkv_profile** out) {
    if (!signs || (mode == PKV_TURBO_POLAR_WITH_QJL && !qjl)) return PKV_ERR_INVALID_ARG;
    return turbo_profile_common(ctx, dim, bits, projections, seed, mode, signs, qjl, out);
}

// f16 halves of v: hi = f16(v), lo = f16(v - hi), both round-to-nearest-even.
static void f16_split(double v, uint16_t* hi, uint16_t* lo) {
    const _Float16 h = static_cast<_Float16>(v);
    const _Float16 l = static_cast<_Float16>(v - static_cast<double>(h));
    std::memcpy(hi, &h, 2);
    std::memcpy(lo, &l, 2);
}

// Operands of the fib encode MFMA path and the acceptance margin `thr` of its
// approximate argmin.  u = 2^-24; f16 splits: RNE on the host (|v - hi - lo|
// <= 2^-22 |v| + 2^-25), round-toward-zero in the kernel (<= 2^-20 |v| +
// 2^-24).  Per rotated component, against the reference's
// rho = f32(sum_c Pi[j][c] f64(f32(x_c / |x|))) (sequential f64), with unit
// rows and a unit x_hat (sum_c |Pi[j][c] x_c| <= 1, sum_c |Pi[j][c]| <= 8,
// sum_c |x_c| <= 8):
//   x_hat' = x * f32(1 / |x|)                        2.01u
//   kernel split of x_hat' (2^-20 + 8 * 2^-24)       24u
//   host split of Pi (2^-22 + 8 * 2^-25)              8u
//   dropped Pi_lo * x_lo                              8u
//   f32 accumulation: the 128 small cross products first (< 1u), then 64
//     hi * hi products, counted as 128 roundings of at most u (twice the
//     sequential round-to-nearest count: truncating adders are covered)   128u
//   the reference's own x_hat and rho roundings       2u
//     (under FibQuantizer::encode semantics, codec.rs:479-483, x_hat stays
//     f64 and only rho's cast to f32 rounds: at most 1u + 2^-50)
// so |rho' - rho| <= eps_rho = 175u for both semantics.  A key is the scoring MFMA's
// f32(|c|^2 + off - 2 c . rho') (16 products of f16 halves, C = 0: 32u S,
// S the largest sum of |terms|; kernel split of rho' 2 l1 17u; host splits
// of -2c and of |c|^2 + off (8 l1 + 2 + 4 kmax)u; dropped lo * lo 16 l1 u)
// with its 5 low bits replaced by the index (31 ulp).  Against the
// reference's f32 distance (shifted by |rho_b|^2, common to all codewords)
// a key is off by at most
//   E = e_score + 2 l1max eps_rho + 8u (cmax + 1)^2 + 31 ulp(kmax),
// so a gap > 2E between the two smallest keys fixes the reference's argmin;
// thr = 2E (1 + 2^-10) (the factor covers thr's own rounding to f32).  Keys
// must stay positive (off - 2 cmax > 0) for the unsigned
// order to be the float order; otherwise thr = inf and every block is redone.
static void fib_mfma_constants(pkv_profile* p) {
    const uint32_t n = p->n, k = p->k, dim = p->dim;
    const double off = 1.25;
    double cmax = 0.0, l1max = 0.0;
    std::vector<double> sq(n);
    for (uint32_t w = 0; w < n; ++w) {
        double q = 0.0, l1 = 0.0;
        for (uint32_t t = 0; t < k; ++t) {
            const double c = p->codebook[w * k + t];
            q += c * c;
            l1 += std::fabs(c);
        }
        sq[w] = q;
        cmax = std::max(cmax, std::sqrt(q));
        l1max = std::max(l1max, l1);
    }
    p->mf.assign(MF_WORDS, 0u);
    auto pack = [](uint16_t a, uint16_t b) { return static_cast<uint32_t>(a) | static_cast<uint32_t>(b) << 16; };
    for (uint32_t t = 0; t < 2; ++t)
        for (uint32_t q = 0; q < 4; ++q)
            for (uint32_t lane = 0; lane < 64; ++lane)
                for (uint32_t i = 0; i < 4; ++i) {
                    const uint32_t row = fib_mfma_row(t, lane % 32);
                    const uint32_t col = 32 * (lane / 32) + 8 * q + 2 * i;
                    uint16_t h0, l0, h1, l1;
                    f16_split(p->rot[row * dim + col], &h0, &l0);
                    f16_split(p->rot[row * dim + col + 1], &h1, &l1);
                    p->mf[MF_ROT + (((t * 4 + q) * 2 + 0) * 64 + lane) * 4 + i] = pack(h0, h1);
                    p->mf[MF_ROT + (((t * 4 + q) * 2 + 1) * 64 + lane) * 4 + i] = pack(l0, l1);
                }
    for (uint32_t lane = 0; lane < 64; ++lane) {
        const uint32_t w = lane % 32, h = lane / 32;
        uint16_t ah, al, bh, bl, kh = 0, kl = 0;
        f16_split(-2.0 * static_cast<double>(p->codebook[w * k + h]), &ah, &al);
        f16_split(-2.0 * static_cast<double>(p->codebook[w * k + 2 + h]), &bh, &bl);
        if (h == 0) f16_split(static_cast<double>(static_cast<float>(sq[w] + off)), &kh, &kl);
        uint32_t* m = &p->mf[MF_SCA + lane * 4];
        m[0] = pack(ah, bh);
        m[1] = pack(ah, bh);
        m[2] = pack(al, bl);
        m[3] = pack(kh, kl);
    }
    const double u = std::ldexp(1.0, -24);
    const double eps_rho = 175.0 * u;
    const double kmax = off + cmax * cmax + 2.0 * cmax * (1.0 + eps_rho);
    const double S = off + cmax * cmax + 2.0 * l1max * (1.0 + eps_rho);
    int ex;
    (void)std::frexp(kmax, &ex);   // kmax in [2^(ex-1), 2^ex)
    const double ulp = std::ldexp(1.0, ex - 24);
    const double e_score = 32.0 * u * S + 2.0 * l1max * 17.0 * u + (8.0 * l1max + 2.0 + 4.0 * kmax) * u +
                           16.0 * l1max * u;
    const double e = e_score + 2.0 * l1max * eps_rho + 8.0 * u * (cmax + 1.0) * (cmax + 1.0) + 31.0 * ulp;
    const bool positive = off - 2.0 * cmax * (1.0 + eps_rho) > 0.25;
    p->thr = positive ? static_cast<float>(2.0 * e * (1.0 + std::ldexp(1.0, -10)))
                      : std::numeric_limits<float>::infinity();
}

// The matrix-core decode is used only if every product it can form equals
// f32 multiplication for this profile's rotation and codebook.
static int fib_verify_mfma_products(pkv_ctx* ctx, pkv_profile* p) {
    uint32_t* d_bad = nullptr;
    HIP_TRY(hipMalloc(&d_bad, sizeof(uint32_t)));
    uint32_t bad = 1;
    hipError_t e = hipMemsetAsync(d_bad, 0, sizeof(uint32_t), ctx->own_stream);
    if (e == hipSuccess) e = static_cast<hipError_t>(launch_fib_product_check(p->d_rot32, p->d_cb, d_bad, ctx->own_stream));
    if (e == hipSuccess) e = hipMemcpyAsync(&bad, d_bad, sizeof(uint32_t), hipMemcpyDeviceToHost, ctx->own_stream);
    const hipError_t se = hipStreamSynchronize(ctx->own_stream);   // queued work ends before `d_bad` is freed
    if (e == hipSuccess) e = se;
    (void)hipFree(d_bad);
    if (e != hipSuccess) return hip_status(e);
    p->mfma_decode = bad == 0 ? 1 : 0;
    return PKV_OK;
}

// The tables in use (a table leaves with its last profile).
static std::mutex g_prefix_mu;
static std::vector<std::weak_ptr<FibPrefix>> g_prefix;

// The matrix-core decode's table of partial sums: that of a profile with the same
// constants, or a new one, complete when this returns.  Without memory for it the
// profile decodes by the kernel that forms every sum.
static int fib_build_prefix(pkv_ctx* ctx, pkv_profile* p) {
    if (!p->mfma_decode) return PKV_OK;
    std::vector<float> key(p->rot32.begin(), p->rot32.begin() + FIB_PREFIX_BLOCKS * p->k * p->dim);
    key.insert(key.end(), p->codebook.begin(), p->codebook.end());
    std::lock_guard<std::mutex> lock(g_prefix_mu);
    g_prefix.erase(std::remove_if(g_prefix.begin(), g_prefix.end(), [](auto& w) { return w.expired(); }),
                   g_prefix.end());
    for (const auto& w : g_prefix) {
        std::shared_ptr<FibPrefix> t = w.lock();
        if (t && t->device == ctx->device && t->key.size() == key.size() &&
            std::memcmp(t->key.data(), key.data(), sizeof(float) * key.size()) == 0) {
            p->prefix = std::move(t);
            return PKV_OK;
        }
    }
    auto t = std::make_shared<FibPrefix>();
    t->device = ctx->device;
    t->key = std::move(key);
    const hipError_t me =
        hipMalloc(reinterpret_cast<void**>(&t->d), (sizeof(float) * p->dim) << (5 * FIB_PREFIX_BLOCKS));
    if (me != hipSuccess) {
        t->d = nullptr;
        (void)hipGetLastError();   // the next launch check must not see it
        return me == hipErrorOutOfMemory ? PKV_OK : hip_status(me);
    }
    const hipError_t e = static_cast<hipError_t>(launch_fib_prefix(p->d_rot32, p->d_cb, t->d, ctx->own_stream));
    const hipError_t se = hipStreamSynchronize(ctx->own_stream);
    if (e != hipSuccess || se != hipSuccess) return hip_status(e == hipSuccess ? se : e);
    g_prefix.push_back(t);
    p->prefix = std::move(t);
    return PKV_OK;
}

static int fib_profile_common(pkv_ctx* ctx, uint32_t dim, uint32_t k, uint32_t n, std::vector<float> cb,
                              std::vector<double> rot, pkv_profile** out) {
    pkv_profile* p = new (std::nothrow) pkv_profile();
    if (!p) return PKV_ERR_OOM;
    p->ctx = ctx;
    p->kind = PKV_CODEC_FIB;
    p->dim = dim;
    p->k = k;
    p->n = n;
    p->wbits = 5;
    p->codebook = std::move(cb);
    p->rot = std::move(rot);
    p->rot32t.resize(static_cast<size_t>(dim) * dim);
    p->rot_t.resize(static_cast<size_t>(dim) * dim);
    p->rot32.resize(static_cast<size_t>(dim) * dim);
    for (uint32_t r = 0; r < dim; ++r)
        for (uint32_t c = 0; c < dim; ++c) {
            const float v = static_cast<float>(p->rot[static_cast<size_t>(r) * dim + c]);
            p->rot32t[static_cast<size_t>(c) * dim + r] = v;
            p->rot32[static_cast<size_t>(r) * dim + c] = v;
            p->rot_t[static_cast<size_t>(c) * dim + r] = p->rot[static_cast<size_t>(r) * dim + c];
        }
    fib_mfma_constants(p);
    p->cb64.assign(p->codebook.begin(), p->codebook.end());   // f64::from(f32), codebook.rs:118-131
    int rc = hip_status(hipSetDevice(ctx->device));
    if (!rc) rc = upload(&p->d_cb, p->codebook);
    if (!rc) rc = upload(&p->d_cb64, p->cb64);
    if (!rc) rc = upload(&p->d_rot_t, p->rot_t);
    if (!rc) rc = upload(&p->d_rot64, p->rot);
    if (!rc) rc = upload(&p->d_rot32t, p->rot32t);
    if (!rc) rc = upload(&p->d_mf, p->mf);
    if (!rc) rc = upload(&p->d_rot32, p->rot32);
    if (!rc) rc = fib_verify_mfma_products(ctx, p);
    if (!rc) rc = fib_build_prefix(ctx, p);
    if (rc) { pkv_profile_destroy(p); return rc; }
    *out = p;
    return PKV_OK;
}

// FibQuantProfileV1's shape checks (fib-quant/src/profile.rs:281-318, and the
// rotation / codebook size limits the profile applies before allocating them):
// invalid shapes first, then the one shape the kernels implement.
static int fib_check(uint32_t dim, uint32_t k, uint32_t n) {
    if (dim == 0 || k == 0 || k >= dim || dim % k != 0) return PKV_ERR_INVALID_ARG;
    if (dim > 16384 || k > 256 || n < 2 || n > (1u << 20)) return PKV_ERR_INVALID_ARG;
    if (static_cast<uint64_t>(dim) * dim > 16777216ull) return PKV_ERR_INVALID_ARG;    // rotation matrix values
    if (static_cast<uint64_t>(n) * k > 67108864ull) return PKV_ERR_INVALID_ARG;       // codebook values
    if (dim != 64 || k != 4 || n != 32) return PKV_ERR_UNSUPPORTED;      // fib_k4_n32 at head_dim 64
    return PKV_OK;
}

// ---- Lloyd refinement on the context's device (pkv_lloyd.hip)
namespace {

int lloyd_shape_ok(uint32_t ns, uint32_t k, uint32_t n, uint32_t restarts) {
    if (k == 0 || n < 2 || k > LLOYD_MAX_K || n > LLOYD_MAX_N || n * k > LLOYD_MAX_NK) return PKV_ERR_UNSUPPORTED;
    if (ns == 0 || restarts == 0 || restarts > 4096) return PKV_ERR_INVALID_ARG;
    return PKV_OK;
}

// Caller holds ctx->mu.  Host buffers in and out; the device work runs on
// the context's own stream, which the call waits for.
int lloyd_on_device_locked(pkv_ctx* ctx, const double* samples, uint32_t ns, uint32_t k, uint32_t n,
                           const double* starts, uint32_t restarts, uint32_t iterations, double* out_cb,
                           double* out_mse, double* init_mse) {
    int rc = lloyd_shape_ok(ns, k, n, restarts);
    if (rc) return rc;
    HIP_TRY(hipSetDevice(ctx->device));
    const size_t s_bytes = sizeof(double) * ns * k, st_bytes = sizeof(double) * restarts * n * k;
    auto pad = [](size_t b) { return (b + 255) & ~static_cast<size_t>(255); };
    const size_t o_st = pad(s_bytes), o_cb = o_st + pad(st_bytes), o_mse = o_cb + pad(st_bytes),
                 o_init = o_mse + pad(sizeof(double) * restarts), o_stat = o_init + 256,
                 o_bd = o_stat + pad(sizeof(uint32_t) * restarts), o_asg = o_bd + pad(sizeof(double) * ns * restarts),
                 total = o_asg + pad(static_cast<size_t>(ns) * restarts);
    uint8_t* d = nullptr;
    HIP_TRY(hipMalloc(&d, total));
    hipStream_t st = ctx->own_stream;
    std::vector<uint32_t> status(restarts, 1u);
    hipError_t e = hipMemcpyAsync(d, samples, s_bytes, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipMemcpyAsync(d + o_st, starts, st_bytes, hipMemcpyHostToDevice, st);
    if (e == hipSuccess)
        e = static_cast<hipError_t>(launch_lloyd(
            reinterpret_cast<const double*>(d), ns, k, n, reinterpret_cast<const double*>(d + o_st), restarts,
            iterations, reinterpret_cast<double*>(d + o_cb), reinterpret_cast<double*>(d + o_mse),
            reinterpret_cast<double*>(d + o_init), reinterpret_cast<uint32_t*>(d + o_stat),
            reinterpret_cast<double*>(d + o_bd), d + o_asg, st));
    if (e == hipSuccess) e = hipMemcpyAsync(out_cb, d + o_cb, st_bytes, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipMemcpyAsync(out_mse, d + o_mse, sizeof(double) * restarts, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipMemcpyAsync(init_mse, d + o_init, sizeof(double), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess)
        e = hipMemcpyAsync(status.data(), d + o_stat, sizeof(uint32_t) * restarts, hipMemcpyDeviceToHost, st);
    // whatever was queued finishes before the scratch and `status` go away
    const hipError_t se = hipStreamSynchronize(st);
    if (e == hipSuccess) e = se;
    (void)hipFree(d);
    if (e != hipSuccess) return hip_status(e);
    for (uint32_t v : status)
        if (v) return PKV_ERR_INVALID_ARG;   // an empty cell with no donor (EmptyCellRepairFailed)
    return PKV_OK;
}

struct CtxLloyd final : LloydDevice {
    pkv_ctx* ctx;
    explicit CtxLloyd(pkv_ctx* c) : ctx(c) {}
    int refine(const std::vector<double>& samples, uint32_t ns, uint32_t k, uint32_t n,
               const std::vector<double>& starts, uint32_t restarts, uint32_t iterations, std::vector<double>& out,
               std::vector<double>& mse, double* init_mse) const override {
        out.assign(static_cast<size_t>(restarts) * n * k, 0.0);
        mse.assign(restarts, 0.0);
        std::lock_guard<std::mutex> lock(ctx->mu);
        return lloyd_on_device_locked(ctx, samples.data(), ns, k, n, starts.data(), restarts, iterations, out.data(),
                                      mse.data(), init_mse);
    }
};

}  // namespace

int pkv_lloyd_refine(pkv_ctx* ctx, const double* samples, uint32_t ns, uint32_t k, uint32_t n, const double* starts,
                     uint32_t restarts, uint32_t iterations, double* out_codebooks, double* out_mse,
                     double* init_mse) {
    if (!ctx || !samples || !starts || !out_codebooks || !out_mse || !init_mse) return PKV_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(ctx->mu);
    return lloyd_on_device_locked(ctx, samples, ns, k, n, starts, restarts, iterations, out_codebooks, out_mse,
                                  init_mse);
}

int pkv_fib_profile_create(pkv_ctx* ctx, uint32_t dim, uint32_t k, uint32_t n, uint64_t seed,
                           uint32_t training_samples, uint32_t lloyd_restarts, uint32_t lloyd_iterations,
                           pkv_profile** out) {
    if (!ctx || !out) return PKV_ERR_INVALID_ARG;
    *out = nullptr;
    int rc = fib_check(dim, k, n);
    if (rc) return rc;
    // FibQuantProfileV1::validate (fib-quant/src/profile.rs:176-263)
    if (lloyd_restarts == 0 || lloyd_restarts > 1024) return PKV_ERR_INVALID_ARG;
    if (lloyd_iterations == 0 || lloyd_iterations > 100000) return PKV_ERR_INVALID_ARG;
    if (training_samples < n || training_samples > 10000000) return PKV_ERR_INVALID_ARG;
    std::vector<float> cb;
    std::vector<double> rot, rot_t;
    // a codebook not built yet in this process is refined on the context's device
    const CtxLloyd dev(ctx);
    rc = make_fib_codebook(dim, k, n, seed, training_samples, lloyd_restarts, lloyd_iterations, cb, nullptr, nullptr,
                           &dev);
    if (rc) return rc;
    rc = make_fib_rotation(dim, seed, rot);
    if (rc) return rc;
    rc = fib_profile_common(ctx, dim, k, n, std::move(cb), std::move(rot), out);
    if (rc) return rc;
    pkv_codec_params& pp = (*out)->params;
    pp.kind = PKV_CODEC_FIB;
    pp.dim = dim;
    pp.k = k;
    pp.n = n;
    pp.seed = seed;
    pp.training_samples = training_samples;
    pp.lloyd_restarts = lloyd_restarts;
    pp.lloyd_iterations = lloyd_iterations;
    (*out)->json_ok = 1;
    return PKV_OK;
}

int pkv_fib_profile_create_with_constants(pkv_ctx* ctx, uint32_t dim, uint32_t k, uint32_t n, const float* codebook,
                                          const double* rotation, pkv_profile** out) {
    if (!ctx || !out || !codebook || !rotation) return PKV_ERR_INVALID_ARG;
    *out = nullptr;
    int rc = fib_check(dim, k, n);
    if (rc) return rc;
    for (uint32_t i = 0; i < n * k; ++i)
        if (!std::isfinite(codebook[i])) return PKV_ERR_INVALID_ARG;   // FibCodebookV1::validate
    std::vector<float> cb(codebook, codebook + n * k);
    std::vector<double> rot(rotation, rotation + static_cast<size_t>(dim) * dim);
    return fib_profile_common(ctx, dim, k, n, std::move(cb), std::move(rot), out);
}

void pkv_profile_destroy(pkv_profile* p) {
    if (!p) return;
    if (p->ctx) (void)hipSetDevice(p->ctx->device);
    (void)hipDeviceSynchronize();
    for (void* d : {static_cast<void*>(p->d_signs), static_cast<void*>(p->d_qjl), static_cast<void*>(p->d_cs),
                    static_cast<void*>(p->d_qa), static_cast<void*>(p->d_qb),
                    static_cast<void*>(p->d_cb), static_cast<void*>(p->d_rot_t), static_cast<void*>(p->d_rot64),
                    static_cast<void*>(p->d_rot32t),
                    static_cast<void*>(p->d_mf), static_cast<void*>(p->d_rot32), static_cast<void*>(p->d_cb64)})
        if (d) (void)hipFree(d);
    delete p;   // with the table of partial sums when no other profile holds it
}

int pkv_fib_decode_path(const pkv_profile* p) {
    if (!p || p->kind != PKV_CODEC_FIB) return -1;
    return p->mfma_decode ? 1 : 0;
}

int pkv_profile_constants(const pkv_profile* p, void* a, size_t a_bytes, void* b, size_t b_bytes) {
    if (!p) return PKV_ERR_INVALID_ARG;
    if (p->kind == PKV_CODEC_TURBO) {
        size_t na = p->signs.size() * sizeof(float), nb = p->qjl.size() * sizeof(float);
        if ((a && a_bytes < na) || (b && b_bytes < nb)) return PKV_ERR_CAPACITY;
        if (a) std::memcpy(a, p->signs.data(), na);
        if (b && nb) std::memcpy(b, p->qjl.data(), nb);
    } else {
        size_t na = p->codebook.size() * sizeof(float), nb = p->rot.size() * sizeof(double);
        if ((a && a_bytes < na) || (b && b_bytes < nb)) return PKV_ERR_CAPACITY;
        if (a) std::memcpy(a, p->codebook.data(), na);
        if (b) std::memcpy(b, p->rot.data(), nb);
    }
    return PKV_OK;
}

uint32_t pkv_payload_len(const pkv_profile* p, int radii_codec) {
    if (!p) return 0;
    return p->kind == PKV_CODEC_TURBO ? turbo_plen(p, radii_codec) : fib_plen(p);
}

uint32_t pkv_header_len(const pkv_profile* p) { return p ? hdr_len(p) : 0; }

uint64_t pkv_blob_len(const pkv_profile* p, int radii_codec, uint64_t n) {
    if (!p) return 0;
    return hdr_len(p) + n * pkv_payload_len(p, radii_codec);
}

int pkv_write_header(const pkv_profile* p, int radii_codec, uint64_t n_vectors, uint8_t* out, uint64_t cap) {
    if (!p || !out) return PKV_ERR_INVALID_ARG;
    int radii = radii_codec;
    if (p->kind == PKV_CODEC_FIB) radii = PKV_RADII_F32;
    else if (radii != PKV_RADII_F32 && radii != PKV_RADII_LOG_U8) return PKV_ERR_INVALID_ARG;
    if (n_vectors == 0) return PKV_ERR_EMPTY_BATCH;   // encode_batch rejects an empty batch
    if (n_vectors > 0xFFFFFFFFull) return PKV_ERR_INVALID_ARG;   // n is a u32 field
    const uint32_t len = hdr_len(p);
    if (cap < len) return PKV_ERR_CAPACITY;
    const HdrBytes h = blob_header(p, n_vectors, radii);
    for (uint32_t i = 0; i < len; ++i) out[i] = static_cast<uint8_t>(h.w[i >> 2] >> (8 * (i & 3)));
    return PKV_OK;
}

int pkv_segments_status(const pkv_profile* prof, const uint32_t* host_status, uint32_t nseg, pkv_error* err) {
    if (!prof || (!host_status && nseg)) return PKV_ERR_INVALID_ARG;
    return resolve_status(prof, host_status, nseg, nullptr, err);
}

int pkv_encode_segments(pkv_ctx* ctx, const pkv_profile* prof, int radii_codec, int in_dtype, const void* d_in,
                        uint64_t in_elems, const pkv_seg* segs, uint32_t nseg, uint8_t* d_wire, uint64_t wire_bytes,
                        uint32_t* d_status, void* stream) {
    return run_segments(ctx, prof, radii_codec, true, in_dtype, d_in, in_elems, segs, nseg, d_wire, wire_bytes,
                        d_status, static_cast<hipStream_t>(stream));
}

int pkv_encode_segments_bounded(pkv_ctx* ctx, const pkv_profile* prof, int radii_codec, int in_dtype,
                                const void* d_in, uint64_t in_elems, const pkv_seg* segs, uint32_t nseg,
                                uint8_t* d_wire, uint64_t wire_bytes, uint32_t max_workgroups, uint32_t* d_status,
                                void* stream) {
    if (!ctx) return PKV_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(ctx->mu);
    return run_segments_locked(ctx, prof, radii_codec, true, in_dtype, d_in, in_elems, segs, nseg, d_wire, wire_bytes,
                               d_status, static_cast<hipStream_t>(stream), false, 1, 0, max_workgroups);
}

int pkv_decode_segments(pkv_ctx* ctx, const pkv_profile* prof, int radii_codec, const uint8_t* d_wire,
                        uint64_t wire_bytes, const pkv_seg* segs, uint32_t nseg, float* d_out, uint64_t out_elems,
                        uint32_t* d_status, void* stream) {
    return run_segments(ctx, prof, radii_codec, false, PKV_F32, d_out, out_elems, segs, nseg, d_wire, wire_bytes,
                        d_status, static_cast<hipStream_t>(stream));
}

int pkv_decode_segments_ex(pkv_ctx* ctx, const pkv_profile* prof, int radii_codec, const uint8_t* d_wire,
                           uint64_t wire_bytes, const pkv_seg* segs, uint32_t nseg, void* d_out, int out_dtype,
                           uint64_t out_elems, uint32_t fanout, uint64_t fanout_stride, uint32_t* d_status,
                           void* stream) {
    if (!ctx) return PKV_ERR_INVALID_ARG;
    if (out_dtype != PKV_F32 && out_dtype != PKV_BF16 && out_dtype != PKV_F16) return PKV_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(ctx->mu);
    return run_segments_locked(ctx, prof, radii_codec, false, out_dtype, d_out, out_elems, segs, nseg, d_wire,
                               wire_bytes, d_status, static_cast<hipStream_t>(stream), false, fanout, fanout_stride);
}

int pkv_decode_segments_bounded(pkv_ctx* ctx, const pkv_profile* prof, int radii_codec, const uint8_t* d_wire,
                                uint64_t wire_bytes, const pkv_seg* segs, uint32_t nseg, void* d_out, int out_dtype,
                                uint64_t out_elems, uint32_t fanout, uint64_t fanout_stride, uint32_t max_workgroups,
                                uint32_t* d_status, void* stream) {
    if (!ctx) return PKV_ERR_INVALID_ARG;
    if (out_dtype != PKV_F32 && out_dtype != PKV_BF16 && out_dtype != PKV_F16) return PKV_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(ctx->mu);
    return run_segments_locked(ctx, prof, radii_codec, false, out_dtype, d_out, out_elems, segs, nseg, d_wire,
                               wire_bytes, d_status, static_cast<hipStream_t>(stream), false, fanout, fanout_stride,
                               max_workgroups);
}

int pkv_status_clear(pkv_ctx* ctx, uint32_t* const* d_status, const uint32_t* nsegs, uint32_t n, void* stream) {
    if (!ctx || n > PKV_STATUS_BUFFERS_MAX || (n && (!d_status || !nsegs))) return PKV_ERR_INVALID_ARG;
    FillList list{};
    list.count = n;
    for (uint32_t i = 0; i < n; ++i) {
        if (nsegs[i] && (!d_status[i] || reinterpret_cast<uintptr_t>(d_status[i]) % 4)) return PKV_ERR_INVALID_ARG;
        list.p[i] = d_status[i];
        list.n[i] = 2ull * nsegs[i];
    }
    std::lock_guard<std::mutex> lock(ctx->mu);
    HIP_TRY(hipSetDevice(ctx->device));
    return hip_status(static_cast<hipError_t>(launch_fill_list(list, STATUS_NONE, stream)));
}

int pkv_run_segments(pkv_ctx* ctx, const pkv_profile* prof, const pkv_segments_op* op, void* stream) {
    if (!ctx || !op || (op->flags & ~PKV_STATUS_CLEARED) || op->reserved) return PKV_ERR_INVALID_ARG;
    const bool cleared = (op->flags & PKV_STATUS_CLEARED) != 0;
    if (cleared && !op->d_status) return PKV_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(ctx->mu);
    return run_segments_locked(ctx, prof, op->radii_codec, op->encode != 0, op->dtype, op->d_tensor, op->elems,
                               op->segs, op->nseg, op->d_wire, op->wire_bytes, op->d_status,
                               static_cast<hipStream_t>(stream), false, op->fanout, op->fanout_stride,
                               op->max_workgroups, nullptr, cleared);
}

// pkv_decode_segments_ex with the table and its tile prefix in this device's
// `scratch` (address from set-up): no allocating call.  Calls sharing the
// scratch are ordered on the device by its event, whatever their stream or
// context.
int pkv_decode_segments_noalloc(pkv_ctx* ctx, const pkv_profile* prof, int radii_codec, const uint8_t* d_wire,
                                uint64_t wire_bytes, const pkv_seg* segs, uint32_t nseg, void* d_out, int out_dtype,
                                uint64_t out_elems, uint32_t fanout, uint64_t fanout_stride, uint32_t* d_status,
                                void* stream) {
    if (!ctx || !prof) return PKV_ERR_INVALID_ARG;
    // the caller's status words are the only report of a rejected blob (its
    // output is left untouched): without them a decode error would pass silently
    if (!d_status) return PKV_ERR_INVALID_ARG;
    if (nseg > PKV_NOALLOC_MAX_SEGMENTS) return PKV_ERR_SCRATCH_LIMIT;
    if (!ctx->noalloc) return PKV_ERR_DEVICE;
    if (out_dtype != PKV_F32 && out_dtype != PKV_BF16 && out_dtype != PKV_F16) return PKV_ERR_INVALID_ARG;
    int radii = radii_codec;
    if (prof->kind == PKV_CODEC_TURBO && radii != PKV_RADII_F32 && radii != PKV_RADII_LOG_U8)
        return PKV_ERR_INVALID_ARG;
    if (prof->kind == PKV_CODEC_FIB) radii = PKV_RADII_F32;
    uint32_t tiles[PKV_NOALLOC_MAX_SEGMENTS + 1];   // host stack, no heap
    int rc = validate_segments(prof, radii, false, out_dtype, d_out, out_elems, segs, nseg, d_wire, wire_bytes, tiles,
                               fanout, fanout_stride);
    if (rc) return rc;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    std::lock_guard<std::mutex> lock(ctx->mu);
    HIP_TRY(hipSetDevice(ctx->device));
    // the table is copied from host memory on every call, which a captured
    // graph would replay from addresses that no longer hold it
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    HIP_TRY(hipStreamIsCapturing(st, &cap));
    if (cap != hipStreamCaptureStatusNone) return PKV_ERR_UNSUPPORTED;
    NoallocScratch& sc = *ctx->noalloc;
    std::lock_guard<std::mutex> scratch_lock(sc.mu);
    uint8_t* base = sc.ptr;
    // the previous call's kernel (any stream, any context on this device)
    // still reads the table until this event completes
    HIP_TRY(hipStreamWaitEvent(st, sc.ev, 0));
    // pageable host sources: the runtime stages them before returning
    HIP_TRY(hipMemcpyAsync(base, segs, sizeof(pkv_seg) * nseg, hipMemcpyHostToDevice, st));
    HIP_TRY(hipMemcpyAsync(base + kNaTileOff, tiles, sizeof(uint32_t) * (nseg + 1), hipMemcpyHostToDevice, st));
    const int e = launch_segments(prof, radii, false, out_dtype, d_out, d_wire, segs,
                                  reinterpret_cast<const SegDev*>(base),
                                  reinterpret_cast<const uint32_t*>(base + kNaTileOff), nseg, tiles[nseg], d_status,
                                  false, fanout, fanout_stride, 0, st);
    const hipError_t re = hipEventRecord(sc.ev, st);
    if (e) return hip_status(static_cast<hipError_t>(e));
    return re == hipSuccess ? PKV_OK : hip_status(re);
}

int pkv_encode_diagnostics(pkv_ctx* ctx, const pkv_profile* prof, int radii_codec, const float* d_in, uint64_t n,
                           uint8_t* d_wire, uint64_t wire_bytes, float* d_diag, uint64_t diag_elems, float* threshold,
                           uint32_t* d_status, void* stream) {
    if (!ctx || !prof || !d_diag || n == 0 || n > MAX_SEG_VECTORS) return PKV_ERR_INVALID_ARG;
    uint64_t need;
    if (prof->kind == PKV_CODEC_FIB) {
        need = n * 16u * 32u;
        if (threshold) *threshold = prof->thr;
    } else {
        if (!prof->mode || !prof->d_qa || prof->pbits > 4) return PKV_ERR_UNSUPPORTED;   // no matrix-core path
        need = n * prof->proj * 2u;
        if (threshold) *threshold = 0.0f;
    }
    if (diag_elems < need) return PKV_ERR_CAPACITY;
    if (reinterpret_cast<uintptr_t>(d_diag) % 4) return PKV_ERR_INVALID_ARG;
    const pkv_seg seg{0, 0, prof->dim, 0, static_cast<uint32_t>(n), static_cast<uint32_t>(n)};
    std::lock_guard<std::mutex> lock(ctx->mu);
    HIP_TRY(hipSetDevice(ctx->device));
    return run_segments_locked(ctx, prof, radii_codec, true, PKV_F32, d_in, n * prof->dim, &seg, 1, d_wire,
                               wire_bytes, d_status, static_cast<hipStream_t>(stream), false, 1, 0, 0, d_diag);
}

int pkv_radii_log_bound(pkv_ctx* ctx, float* out) {
    if (!ctx || !out) return PKV_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(ctx->mu);
    HIP_TRY(hipSetDevice(ctx->device));
    float* d = nullptr;
    HIP_TRY(hipMalloc(&d, 256 * sizeof(float)));
    hipError_t e = static_cast<hipError_t>(launch_logf_bound_read(d, ctx->own_stream));
    if (e == hipSuccess) e = hipMemcpyAsync(out, d, 256 * sizeof(float), hipMemcpyDeviceToHost, ctx->own_stream);
    const hipError_t se = hipStreamSynchronize(ctx->own_stream);   // queued work ends before `d` is freed
    if (e == hipSuccess) e = se;
    (void)hipFree(d);
    return e == hipSuccess ? PKV_OK : hip_status(e);
}

// ---- BLAKE3 digests of device bytes

namespace {

// Pass tables of one pkv_blake3_ranges call: [ranges | pass 0 | pass 1 | ...],
// each pass nr + 1 B3Pass records (launch sequence in pkv_blake3.hip).
struct B3Plan {
    std::vector<B3Pass> passes;     // passes.size() == npass * (nr + 1)
    std::vector<uint32_t> tiles;    // per pass
    uint64_t cvs = 0;               // chaining values written by passes that do not finish a range
    bool quad = false;              // pass 0 on four lanes per chunk (16-chunk tiles)
    uint64_t end[2] = {0, 0};       // last byte (exclusive) the ranges need of each buffer
};

// Chunks of a call (both tiers of a build together) below which pass 0 puts four
// lanes on a chunk: 16 chunks per wave, ~1.4x the instructions, a quarter of the
// latency; one lane per chunk leaves the GPU with at most a wave per SIMD there.
// Measured, one lane / four, us a call, over 48 ranges | 48 and 384 ranges of two
// tiers | 600 ranges of equal size:
//   16 Ki  58 / 40 | 54 / 34 | 57 / 44      52 Ki  55 / 63 | 52 / 58 | 92 / 66
//   32 Ki  56 / 50 | 52 / 49 | 59 / 55      64 Ki  90 / 70 | 82 / 66 | 93 / 74
//   44 Ki  55 / 51 | 50 / 49 | 90 / 58      80 Ki  89 / 77 | 82 / 73 | 87 / 83
//   48 Ki  54 / 51 | 52 / 57 | 95 / 65      96 Ki  85 / 80 | 78 / 82 | 87 / 91
// Four lanes are ahead in every shape up to 44 Ki; past 48 Ki the count alone does
// not decide (one lane steps up with its second wave per SIMD, 1,024 tiles of 64
// chunks of a range).
constexpr uint64_t kB3QuadBelow = 48ull * 1024;

// Ranges r < split lie in the first buffer, the others in the second.
int plan_blake3(const pkv_range* ranges, uint32_t nr, uint64_t split, const uint64_t (&buf_bytes)[2], B3Plan* plan) {
    std::vector<uint64_t> count(nr), in_base(nr, 0);
    uint64_t total = 0;
    for (uint32_t r = 0; r < nr; ++r) {
        const pkv_range& g = ranges[r];
        const uint64_t bytes = buf_bytes[r < split ? 0 : 1];
        if (g.offset > bytes || g.len > bytes - g.offset) return PKV_ERR_INVALID_ARG;
        uint64_t& end = plan->end[r < split ? 0 : 1];
        end = std::max(end, g.offset + g.len);
        count[r] = b3::chunks_of(g.len);
        if (count[r] > 0xFFFFFFFFull) return PKV_ERR_INVALID_ARG;
        total += count[r];
    }
    plan->quad = total < kB3QuadBelow;
    for (bool more = true; more;) {
        more = false;
        const size_t base = plan->passes.size();
        const uint64_t per_tile = base == 0 && plan->quad ? 16 : 64;   // elements per wave in this pass
        plan->passes.resize(base + nr + 1);
        uint64_t tiles = 0;
        for (uint32_t r = 0; r < nr; ++r) {
            B3Pass& ps = plan->passes[base + r];
            const uint64_t c = count[r], t = (c + per_tile - 1) / per_tile;
            ps.tile_start = static_cast<uint32_t>(tiles);
            ps.count = static_cast<uint32_t>(c);
            ps.in_base = static_cast<uint32_t>(in_base[r]);
            ps.out_base = 0;
            tiles += t;
            if (t > 1) {   // not finished in this pass: t chaining values go on
                ps.out_base = static_cast<uint32_t>(plan->cvs);
                in_base[r] = plan->cvs;
                plan->cvs += t;
                count[r] = t;
                more = true;
            } else {
                count[r] = 0;
            }
            if (tiles > 0xFFFFFFFFull || plan->cvs > 0xFFFFFFFFull) return PKV_ERR_INVALID_ARG;
        }
        plan->passes[base + nr].tile_start = static_cast<uint32_t>(tiles);
        plan->tiles.push_back(static_cast<uint32_t>(tiles));
    }
    return PKV_OK;
}

// Caller holds ctx->mu and has made the device current.  n_layers != 0 (nr =
// 2 n_layers, io.split even): the last pass also forms the layer digests.
int blake3_ranges_locked(pkv_ctx* ctx, const B3Io& io, const uint64_t (&buf_bytes)[2], const pkv_range* ranges,
                         uint32_t nr, hipStream_t stream, uint32_t n_layers = 0, uint32_t layers = 0) {
    const size_t range_bytes = sizeof(pkv_range) * nr;
    const size_t pass_off = (range_bytes + 255) & ~static_cast<size_t>(255);
    const uint64_t hash = table_hash(ranges, range_bytes);
    // The same table again on the same stream (a serving loop's digest of
    // every step) reuses its slot and plan as they are: no upload, and the
    // chaining-value scratch is rewritten only after the previous call, in
    // stream order.
    Slot* sl = nullptr;
    for (Slot& c : ctx->slots)
        if (c.digest && c.nseg == nr && c.hash == hash && c.b3_split == io.split && c.users.n == 1 &&
            !c.users.overflow && c.users.s[0] == stream && c.b3_end[0] <= buf_bytes[0] &&
            c.b3_end[1] <= buf_bytes[1] && std::memcmp(c.host, ranges, range_bytes) == 0) {
            sl = &c;
            break;
        }
    hipError_t cp = hipSuccess;
    if (!sl) {
        B3Plan plan;
        int rc = plan_blake3(ranges, nr, io.split, buf_bytes, &plan);
        if (rc) return rc;
        const size_t pass_bytes = sizeof(B3Pass) * plan.passes.size();
        const size_t cv_off = (pass_off + pass_bytes + 255) & ~static_cast<size_t>(255);
        rc = acquire_slot(ctx, cv_off + 32 * plan.cvs + 256, &sl);
        if (rc) return rc;
        auto* h = static_cast<uint8_t*>(sl->host);
        std::memcpy(h, ranges, range_bytes);
        std::memcpy(h + pass_off, plan.passes.data(), pass_bytes);
        cp = hipMemcpyAsync(sl->dev, sl->host, pass_off + pass_bytes, hipMemcpyHostToDevice, stream);
        // reusable by a later call only once its table is on the way to the device
        sl->digest = cp == hipSuccess;
        sl->nseg = nr;
        sl->hash = hash;
        sl->b3_tiles = std::move(plan.tiles);
        sl->b3_quad = plan.quad;
        sl->b3_end[0] = plan.end[0];
        sl->b3_end[1] = plan.end[1];
        sl->b3_split = io.split;
    }
    const size_t np = sl->b3_tiles.size();
    const size_t cv_off = (pass_off + sizeof(B3Pass) * np * (nr + 1) + 255) & ~static_cast<size_t>(255);
    auto* d = static_cast<uint8_t*>(sl->dev);
    auto* d_ranges = reinterpret_cast<const B3Range*>(d);
    auto* d_cv = reinterpret_cast<uint32_t*>(d + cv_off);
    auto d_pass = [&](size_t p) { return reinterpret_cast<const B3Pass*>(d + pass_off) + p * (nr + 1); };
    int e = cp;
    for (size_t p = 0; p < np && !e; ++p) {
        const uint32_t tiles = sl->b3_tiles[p];
        if (p == 0)
            e = sl->b3_quad ? launch_blake3_quad(io, d_ranges, d_pass(0), nr, tiles, d_cv, stream)
                            : launch_blake3_pass(io, d_ranges, d_pass(0), nr, tiles, d_cv, stream);
        else if (!n_layers || p + 1 < np)
            e = launch_blake3_merge4(io, d_pass(p), nr, tiles, d_cv, d_cv, stream);
    }
    if (n_layers && !e)   // a single pass ended every range itself
        e = launch_blake3_layers(io, np > 1 ? d_pass(np - 1) : nullptr, d_cv, n_layers, layers, stream);
    const int rc2 = finish_slot(sl, stream);
    if (e) return hip_status(static_cast<hipError_t>(e));
    return rc2;
}

// One buffer of nr ranges, its digests at d_out.
B3Io one_buffer(const uint8_t* d_buf, uint64_t nr, uint8_t* d_out) {
    B3Io io{};
    io.buf[0] = d_buf;
    io.out[0] = reinterpret_cast<uint32_t*>(d_out);
    io.split = nr;
    return io;
}

}  // namespace

int pkv_blake3_ranges(pkv_ctx* ctx, const uint8_t* d_buf, uint64_t buf_bytes, const pkv_range* ranges, uint32_t n,
                      uint8_t* d_out, void* stream) {
    if (!ctx) return PKV_ERR_INVALID_ARG;
    if (n == 0) return PKV_OK;
    if (!ranges || !d_out || reinterpret_cast<uintptr_t>(d_out) % 4 || (!d_buf && buf_bytes))
        return PKV_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(ctx->mu);
    HIP_TRY(hipSetDevice(ctx->device));
    return blake3_ranges_locked(ctx, one_buffer(d_buf, n, d_out), {buf_bytes, 0}, ranges, n,
                                static_cast<hipStream_t>(stream));
}

int pkv_blake3_layer_digests(pkv_ctx* ctx, const uint8_t* d_kv_digests, uint32_t n, uint32_t layers, uint8_t* d_out,
                             void* stream) {
    if (!ctx || layers == 0) return PKV_ERR_INVALID_ARG;
    if (n == 0) return PKV_OK;
    if (!d_kv_digests || !d_out || reinterpret_cast<uintptr_t>(d_kv_digests) % 4 ||
        reinterpret_cast<uintptr_t>(d_out) % 4)
        return PKV_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(ctx->mu);
    HIP_TRY(hipSetDevice(ctx->device));
    // no range is left to hash: the payload digests are only read
    B3Io io = one_buffer(nullptr, 2ull * n, const_cast<uint8_t*>(d_kv_digests));
    io.layer[0] = reinterpret_cast<uint32_t*>(d_out);
    const int e = launch_blake3_layers(io, nullptr, nullptr, n, layers, stream);
    return e ? hip_status(static_cast<hipError_t>(e)) : PKV_OK;
}

int pkv_blake3_tier_digests(pkv_ctx* ctx, const uint8_t* d_buf, uint64_t buf_bytes, const pkv_range* ranges,
                            uint32_t n, uint32_t layers, uint8_t* d_blob_digests, uint8_t* d_layer_digests,
                            void* stream) {
    if (!ctx || layers == 0) return PKV_ERR_INVALID_ARG;
    if (n == 0) return PKV_OK;
    const pkv_digest_tier tier{d_buf, buf_bytes, ranges, d_blob_digests, d_layer_digests, n, 0};
    return pkv_blake3_build_digests(ctx, &tier, 1, layers, stream);
}

int pkv_blake3_build_digests(pkv_ctx* ctx, const pkv_digest_tier* tiers, uint32_t n_tiers, uint32_t layers,
                             void* stream) {
    if (!ctx || layers == 0 || n_tiers > 2 || (n_tiers && !tiers)) return PKV_ERR_INVALID_ARG;
    B3Io io{};
    uint64_t bytes[2] = {0, 0}, total = 0;
    const pkv_range* ranges = nullptr;
    uint32_t used = 0;
    for (uint32_t k = 0; k < n_tiers; ++k) {
        const pkv_digest_tier& t = tiers[k];
        if (t.reserved) return PKV_ERR_INVALID_ARG;
        if (t.n == 0) continue;
        if (t.n > 0x7FFFFFFFu || !t.ranges || !t.d_blob_digests || !t.d_layer_digests || (!t.d_buf && t.buf_bytes) ||
            reinterpret_cast<uintptr_t>(t.d_blob_digests) % 4 || reinterpret_cast<uintptr_t>(t.d_layer_digests) % 4)
            return PKV_ERR_INVALID_ARG;
        io.buf[used] = t.d_buf;
        io.out[used] = reinterpret_cast<uint32_t*>(t.d_blob_digests);
        io.layer[used] = reinterpret_cast<uint32_t*>(t.d_layer_digests);
        bytes[used] = t.buf_bytes;
        if (used == 0) io.split = 2ull * t.n;
        ranges = t.ranges;
        total += t.n;
        ++used;
    }
    if (used == 0) return PKV_OK;
    if (total > 0x7FFFFFFFu) return PKV_ERR_INVALID_ARG;
    std::vector<pkv_range> both;
    if (used == 2) {   // the second tier's ranges after the first's
        both.reserve(2 * total);
        both.insert(both.end(), tiers[0].ranges, tiers[0].ranges + 2ull * tiers[0].n);
        both.insert(both.end(), tiers[1].ranges, tiers[1].ranges + 2ull * tiers[1].n);
        ranges = both.data();
    }
    std::lock_guard<std::mutex> lock(ctx->mu);
    HIP_TRY(hipSetDevice(ctx->device));
    return blake3_ranges_locked(ctx, io, bytes, ranges, static_cast<uint32_t>(2 * total),
                                static_cast<hipStream_t>(stream), static_cast<uint32_t>(total), layers);
}

int pkv_blake3(pkv_ctx* ctx, const void* data, uint64_t len, uint8_t out[32]) {
    if (!ctx || !out || (!data && len)) return PKV_ERR_INVALID_ARG;
    const uint64_t in_pad = (len + 255) & ~static_cast<uint64_t>(255);
    std::lock_guard<std::mutex> lock(ctx->mu);   // serialises use of ctx->io_buf
    HIP_TRY(hipSetDevice(ctx->device));
    int rc = ensure_io_buf(ctx, in_pad + 256);
    if (rc) return rc;
    auto* d_in = static_cast<uint8_t*>(ctx->io_buf);
    uint8_t* d_hash = d_in + in_pad;
    hipStream_t st = ctx->own_stream;
    if (len) HIP_TRY(hipMemcpyAsync(d_in, data, len, hipMemcpyHostToDevice, st));
    const pkv_range rg{0, len};
    rc = blake3_ranges_locked(ctx, one_buffer(d_in, 1, d_hash), {len, 0}, &rg, 1, st);
    if (rc) { (void)hipStreamSynchronize(st); return rc; }
    HIP_TRY(hipMemcpyAsync(out, d_hash, 32, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    return PKV_OK;
}

int pkv_fb2_n_blocks(const uint8_t* payload, uint64_t len, uint64_t* n) {
    if (!n || (!payload && len)) return PKV_ERR_INVALID_ARG;
    if (len < 14 || std::memcmp(payload, "FB2", 3) != 0) return PKV_ERR_CORRUPT_PAYLOAD;
    *n = rd32(payload + 10);
    return PKV_OK;
}

int pkv_parse_header(const pkv_profile* p, const uint8_t* b, uint64_t len, uint64_t* n_vectors, int* radii_codec) {
    if (!p || !b) return PKV_ERR_INVALID_ARG;
    if (p->kind == PKV_CODEC_TURBO) {
        // TurboCodeWireV1::decode_batch (turbo-quant/src/wire.rs:401-503, 566)
        if (len < 38) return PKV_ERR_CORRUPT_PAYLOAD;
        if (std::memcmp(b, "TQB1", 4) != 0 || rd16(b + 4) != 1 || rd16(b + 6) != 1 || b[8] != 2)
            return PKV_ERR_CORRUPT_PAYLOAD;
        if (b[15] > 1) return PKV_ERR_CORRUPT_PAYLOAD;
        const int rc = b[15];
        if (rd32(b + 10) != p->dim || rd32(b + 18) != p->proj || rd64(b + 22) != p->seed) return PKV_ERR_CORRUPT_PAYLOAD;
        if (b[14] != p->pbits) return PKV_ERR_CORRUPT_PAYLOAD;
        const uint64_t n = rd32(b + 30);
        if (rd32(b + 34) != turbo_plen(p, rc)) return PKV_ERR_CORRUPT_PAYLOAD;
        // a short buffer is rejected before any vector (wire.rs:489-498); trailing
        // bytes only after every vector (cursor.finish(), wire.rs:566): the
        // host-buffer decode checks them once the kernel has validated the vectors
        if (len < 38 + n * turbo_plen(p, rc)) return PKV_ERR_CORRUPT_PAYLOAD;
        if (n_vectors) *n_vectors = n;
        if (radii_codec) *radii_codec = rc;
        return PKV_OK;
    }
    // FibCodeV1::decode_batch (fib-quant/src/codec.rs:323-402); trailing bytes allowed
    if (len < 19) return PKV_ERR_CORRUPT_PAYLOAD;
    if (std::memcmp(b, "FB2", 3) != 0 || b[3] != 1) return PKV_ERR_CORRUPT_PAYLOAD;
    if (b[4] != p->wbits || rd32(b + 6) != p->dim / p->k) return PKV_ERR_CORRUPT_PAYLOAD;
    const uint64_t n = rd32(b + 10);
    if (b[14] != 0) return PKV_ERR_CORRUPT_PAYLOAD;
    const uint64_t nlen = rd16(b + 15), ilen = rd16(b + 17);
    if (len < 19 + n * (nlen + ilen)) return PKV_ERR_CORRUPT_PAYLOAD;
    if (ilen != fib_plen(p) - 2) return PKV_ERR_CORRUPT_PAYLOAD;
    if (n > 0 && nlen != 2) return PKV_ERR_CORRUPT_PAYLOAD;
    if (n_vectors) *n_vectors = n;
    if (radii_codec) *radii_codec = 0;
    return PKV_OK;
}

int pkv_encode_batch_compact(pkv_ctx* ctx, const pkv_profile* prof, int radii_codec, const float* vectors, uint64_t n,
                             uint8_t* out, uint64_t out_cap, uint64_t* out_len, pkv_error* err) {
    if (err) { err->status = PKV_OK; err->segment = -1; err->index = 0; }
    if (!ctx || !prof || (!vectors && n)) return PKV_ERR_INVALID_ARG;
    if (prof->kind == PKV_CODEC_FIB) radii_codec = PKV_RADII_F32;
    if (radii_codec != PKV_RADII_F32 && radii_codec != PKV_RADII_LOG_U8) return PKV_ERR_INVALID_ARG;
    const uint64_t blob = pkv_blob_len(prof, radii_codec, n);
    if (out_len) *out_len = blob;
    if (n == 0) return PKV_ERR_EMPTY_BATCH;
    if (n > MAX_SEG_VECTORS) return PKV_ERR_INVALID_ARG;
    if (!out || out_cap < blob) return PKV_ERR_CAPACITY;
    const uint64_t in_bytes = n * prof->dim * sizeof(float);
    const uint64_t in_pad = (in_bytes + 255) & ~static_cast<uint64_t>(255);
    std::lock_guard<std::mutex> lock(ctx->mu);   // serialises use of ctx->io_buf
    HIP_TRY(hipSetDevice(ctx->device));
    int rc = ensure_io_buf(ctx, in_pad + blob + 256 + 64);
    if (rc) return rc;
    auto* d_in = static_cast<uint8_t*>(ctx->io_buf);
    uint8_t* d_wire = d_in + in_pad;
    uint32_t* d_stat = reinterpret_cast<uint32_t*>(d_wire + ((blob + 255) & ~static_cast<uint64_t>(255)));
    hipStream_t st = ctx->own_stream;
    HIP_TRY(hipMemcpyAsync(d_in, vectors, in_bytes, hipMemcpyHostToDevice, st));
    pkv_seg seg{0, 0, prof->dim, 0, static_cast<uint32_t>(n), static_cast<uint32_t>(n)};
    rc = run_segments_locked(ctx, prof, radii_codec, true, PKV_F32, d_in, n * prof->dim, &seg, 1, d_wire, blob,
                             d_stat, st);
    if (rc) { (void)hipStreamSynchronize(st); return rc; }
    uint32_t hs[2];
    rc = copy_back(st, hs, d_stat, sizeof hs, out, d_wire, blob);
    if (rc) return rc;
    return resolve_status(prof, hs, 1, &seg, err);
}

int pkv_decode_batch_compact(pkv_ctx* ctx, const pkv_profile* prof, const uint8_t* payload, uint64_t len, float* out,
                             uint64_t out_cap_vectors, uint64_t* n_out, pkv_error* err) {
    if (err) { err->status = PKV_OK; err->segment = -1; err->index = 0; }
    if (!ctx || !prof || !payload) return PKV_ERR_INVALID_ARG;
    if (prof->kind == PKV_CODEC_FIB && !(len >= 3 && std::memcmp(payload, "FB2", 3) == 0)) {
        // FibQuantAdapter::decode_batch_compact's fallback (codec.rs:542-561):
        // the payload is one FB1 record, or else one JSON FibCodeV1, and
        // decode_batch_fast decodes it
        if (n_out) *n_out = 1;
        if (!out || out_cap_vectors < 1) return PKV_ERR_CAPACITY;
        const uint64_t off[2] = {0, len};
        return pkv_decode_vectors(ctx, prof, 0, payload, off, 1, out, out_cap_vectors, err);
    }
    uint64_t n = 0;
    int radii = 0;
    int rc = pkv_parse_header(prof, payload, len, &n, &radii);
    if (rc) { if (err) err->status = rc; return rc; }
    if (n_out) *n_out = n;
    const uint64_t blob = pkv_blob_len(prof, radii, n);
    if (n == 0) {
        if (prof->kind == PKV_CODEC_TURBO && len != blob) {   // cursor.finish(), wire.rs:566
            if (err) err->status = PKV_ERR_CORRUPT_PAYLOAD;
            return PKV_ERR_CORRUPT_PAYLOAD;
        }
        return PKV_OK;
    }
    if (n > MAX_SEG_VECTORS) return PKV_ERR_INVALID_ARG;
    if (!out || out_cap_vectors < n) return PKV_ERR_CAPACITY;
    const uint64_t out_bytes = n * prof->dim * sizeof(float);
    const uint64_t out_pad = (out_bytes + 255) & ~static_cast<uint64_t>(255);
    std::lock_guard<std::mutex> lock(ctx->mu);
    HIP_TRY(hipSetDevice(ctx->device));
    rc = ensure_io_buf(ctx, out_pad + blob + 256 + 64);
    if (rc) return rc;
    auto* d_out = static_cast<uint8_t*>(ctx->io_buf);
    uint8_t* d_wire = d_out + out_pad;
    uint32_t* d_stat = reinterpret_cast<uint32_t*>(d_wire + ((blob + 255) & ~static_cast<uint64_t>(255)));
    hipStream_t st = ctx->own_stream;
    HIP_TRY(hipMemcpyAsync(d_wire, payload, blob, hipMemcpyHostToDevice, st));
    pkv_seg seg{0, 0, prof->dim, 0, static_cast<uint32_t>(n), static_cast<uint32_t>(n)};
    rc = run_segments_locked(ctx, prof, radii, false, PKV_F32, d_out, n * prof->dim, &seg, 1, d_wire, blob, d_stat,
                             st);
    if (rc) { (void)hipStreamSynchronize(st); return rc; }
    uint32_t hs[2];
    rc = copy_back(st, hs, d_stat, sizeof hs, out, d_out, out_bytes);
    if (rc) return rc;
    rc = resolve_status(prof, hs, 1, &seg, err);
    if (rc == PKV_OK && prof->kind == PKV_CODEC_TURBO && len != blob) {   // cursor.finish(), wire.rs:566
        if (err) { err->status = PKV_ERR_CORRUPT_PAYLOAD; err->segment = -1; err->index = 0; }
        return PKV_ERR_CORRUPT_PAYLOAD;
    }
    return rc;
}

// ---- scoring on compressed codes (turbo-quant/src/turbo.rs:322-381)
namespace {

// QJL estimator scale with unit source norm: (PI / 2).sqrt() * 1.0 / m in f32
// (qjl.rs:312-313; PI = std::f32::consts::PI).
float qjl_score_scale(uint32_t proj) {
    const float pi = 3.14159265358979323846f;
    return std::sqrt(pi / 2.0f) * 1.0f / static_cast<float>(proj);
}

// The segment table against a score matrix: segment i's codes land in
// columns col(i) < ld of every query row; blobs lie inside the wire buffer.
int validate_score_segments(const pkv_profile* p, int radii, const pkv_seg* segs, uint32_t nseg, uint32_t nq,
                            uint64_t prepared_rows, uint64_t query_stride, uint64_t ld, uint64_t score_elems,
                            uint64_t wire_bytes, std::vector<uint32_t>& tile_start) {
    if (!segs || nseg == 0) return PKV_ERR_INVALID_ARG;
    uint64_t rows_needed;   // (nseg - 1) * query_stride + nq prepared rows
    if (nq && (!mul_add_ok(nseg - 1, query_stride, nq, &rows_needed) || rows_needed > prepared_rows))
        return PKV_ERR_DIM_MISMATCH;
    const uint32_t plen = turbo_plen(p, radii);
    const uint32_t hdr = hdr_len(p);
    uint64_t rows_end = 0;
    if (nq && !mul_add_ok(nq - 1, ld, 0, &rows_end)) return PKV_ERR_DIM_MISMATCH;
    tile_start.assign(nseg + 1, 0);
    uint64_t total = 0;
    for (uint32_t i = 0; i < nseg; ++i) {
        const pkv_seg& s = segs[i];
        if (s.group == 0 || s.n_vectors > MAX_SEG_VECTORS) return PKV_ERR_INVALID_ARG;
        uint64_t end;   // one past the largest column
        if (!seg_extent(s, 1, &end)) return PKV_ERR_DIM_MISMATCH;
        if (s.n_vectors && nq) {
            uint64_t last;
            if (end > ld || __builtin_add_overflow(rows_end, end, &last) || last > score_elems)
                return PKV_ERR_DIM_MISMATCH;
        }
        uint64_t blob_end;
        if (!mul_add_ok(s.n_vectors, plen, hdr, &blob_end) ||
            __builtin_add_overflow(blob_end, s.wire_offset, &blob_end) || blob_end > wire_bytes)
            return PKV_ERR_CAPACITY;
        uint64_t tiles = (static_cast<uint64_t>(s.n_vectors) + TILE - 1) / TILE;
        if (tiles == 0) tiles = 1;
        tile_start[i] = static_cast<uint32_t>(total);
        total += tiles;
        if (total > 0x7fffffffull) return PKV_ERR_INVALID_ARG;
    }
    tile_start[nseg] = static_cast<uint32_t>(total);
    return PKV_OK;
}

// Status of a scoring launch: per segment, a rejected code (word 0: the blob
// is validated as a whole before any score, wire.rs:401-568) precedes a
// non-finite score (word 1); segments in order.
int resolve_score_status(const uint32_t* st, uint32_t nseg, pkv_error* err) {
    for (uint32_t s = 0; s < nseg; ++s) {
        const uint32_t w0 = st[2 * s], w1 = st[2 * s + 1];
        if (w0 == STATUS_NONE && w1 == STATUS_NONE) continue;
        const uint32_t pick = w0 != STATUS_NONE ? w0 : w1;
        if (err) {
            err->status = PKV_ERR_CORRUPT_PAYLOAD;
            err->segment = static_cast<int32_t>(s);
            err->index = pick >> 4;
        }
        return PKV_ERR_CORRUPT_PAYLOAD;
    }
    if (err) { err->status = PKV_OK; err->segment = -1; err->index = 0; }
    return PKV_OK;
}

int prepare_locked(pkv_ctx* ctx, const pkv_profile* prof, const float* d_q, uint32_t nq, float* d_prepared,
                   uint32_t* d_status, hipStream_t stream) {
    if (d_status) {
        int rc = launch_fill_u32(d_status, STATUS_NONE, 2, stream);
        if (rc) return hip_status(static_cast<hipError_t>(rc));
    }
    if (nq == 0) return PKV_OK;
    const float rscale = 1.0f / std::sqrt(static_cast<float>(prof->dim));   // rotation.rs:393-397
    int e = launch_turbo_prepare(turbo_dev(prof), d_q, nq, d_prepared, rscale, d_status, stream);
    return e ? hip_status(static_cast<hipError_t>(e)) : PKV_OK;
}

int score_locked(pkv_ctx* ctx, const pkv_profile* prof, int radii, const uint8_t* d_wire, uint64_t wire_bytes,
                 const pkv_seg* segs, uint32_t nseg, const float* d_prepared, uint64_t prepared_rows, uint32_t nq,
                 uint64_t query_stride, float post, float* d_scores, uint64_t score_elems, uint64_t ld,
                 uint32_t* d_status, hipStream_t stream) {
    std::vector<uint32_t> tiles;
    int rc = validate_score_segments(prof, radii, segs, nseg, nq, prepared_rows, query_stride, ld, score_elems,
                                     wire_bytes, tiles);
    if (rc) return rc;
    Slot* sl;
    SegDev* dsegs;
    uint32_t *dtiles, *dstat, *dmap;
    rc = stage_table(ctx, segs, nseg, tiles, d_status == nullptr, stream, &sl, &dsegs, &dtiles, &dstat, &dmap);
    if (rc) return rc;
    uint32_t* status = d_status ? d_status : dstat;
    rc = launch_fill_u32(status, STATUS_NONE, 2ull * nseg, stream);
    if (rc) { finish_slot(sl, stream); return hip_status(static_cast<hipError_t>(rc)); }
    LaunchCommon lc;
    lc.segs = dsegs;
    lc.tile_start = dtiles;
    lc.tile_seg = dmap;
    lc.nseg = nseg;
    lc.status = status;
    lc.radii = static_cast<uint32_t>(radii);
    lc.plen = turbo_plen(prof, radii);
    lc.in_bf16 = 0;
    lc.per_vector = 0;
    lc.out_dtype = PKV_F32;
    lc.fanout = 1;
    lc.fanout_stride = 0;
    const float qscale = prof->mode ? qjl_score_scale(prof->proj) : 0.0f;
    int e = launch_turbo_score(lc, turbo_dev(prof), d_wire, d_prepared, nq, query_stride, d_scores, ld, qscale, post,
                               tiles[nseg], stream);
    int rc2 = finish_slot(sl, stream);
    if (e) return hip_status(static_cast<hipError_t>(e));
    return rc2;
}

bool score_profile_ok(const pkv_profile* p) {
    return p && p->kind == PKV_CODEC_TURBO && (p->dim == 64 || p->dim == 128) && p->pbits >= 1 && p->pbits <= 8 &&
           (!p->mode || p->proj == 32 || p->proj == 64);
}

}  // namespace

uint32_t pkv_prepared_len(const pkv_profile* p) {
    if (!p || p->kind != PKV_CODEC_TURBO) return 0;
    return p->dim + (p->mode ? p->proj : 0);
}

int pkv_turbo_prepare_queries(pkv_ctx* ctx, const pkv_profile* prof, const float* d_queries, uint32_t nq,
                              float* d_prepared, uint32_t* d_status, void* stream) {
    if (!ctx || !prof) return PKV_ERR_INVALID_ARG;
    if (prof->kind != PKV_CODEC_TURBO) return PKV_ERR_INVALID_ARG;
    if (!score_profile_ok(prof)) return PKV_ERR_UNSUPPORTED;
    if (nq && (!d_queries || !d_prepared)) return PKV_ERR_INVALID_ARG;
    if (reinterpret_cast<uintptr_t>(d_queries) % 4 || reinterpret_cast<uintptr_t>(d_prepared) % 4)
        return PKV_ERR_INVALID_ARG;
    if (nq > 0x7fffffffu) return PKV_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(ctx->mu);
    HIP_TRY(hipSetDevice(ctx->device));
    return prepare_locked(ctx, prof, d_queries, nq, d_prepared, d_status, static_cast<hipStream_t>(stream));
}

int pkv_turbo_score_segments(pkv_ctx* ctx, const pkv_profile* prof, int radii_codec, const uint8_t* d_wire,
                             uint64_t wire_bytes, const pkv_seg* segs, uint32_t nseg, const float* d_prepared,
                             uint64_t prepared_rows, uint32_t nq, uint64_t query_stride, float post_scale,
                             float* d_scores, uint64_t score_elems, uint64_t ld, uint32_t* d_status, void* stream) {
    if (!ctx || !prof) return PKV_ERR_INVALID_ARG;
    if (prof->kind != PKV_CODEC_TURBO) return PKV_ERR_INVALID_ARG;
    if (!score_profile_ok(prof)) return PKV_ERR_UNSUPPORTED;
    if (radii_codec != PKV_RADII_F32 && radii_codec != PKV_RADII_LOG_U8) return PKV_ERR_INVALID_ARG;
    if (!std::isfinite(post_scale)) return PKV_ERR_INVALID_ARG;   // kv.rs:309-313
    if (!d_wire || (nq && (!d_prepared || !d_scores))) return PKV_ERR_INVALID_ARG;
    if (reinterpret_cast<uintptr_t>(d_scores) % 4 || reinterpret_cast<uintptr_t>(d_prepared) % 4)
        return PKV_ERR_INVALID_ARG;
    std::lock_guard<std::mutex> lock(ctx->mu);
    HIP_TRY(hipSetDevice(ctx->device));
    return score_locked(ctx, prof, radii_codec, d_wire, wire_bytes, segs, nseg, d_prepared, prepared_rows, nq,
                        query_stride, post_scale, d_scores, score_elems, ld, d_status,
                        static_cast<hipStream_t>(stream));
}

int pkv_score_status(const uint32_t* host_status, uint32_t nseg, pkv_error* err) {
    if (!host_status && nseg) return PKV_ERR_INVALID_ARG;
    return resolve_score_status(host_status, nseg, err);
}

int pkv_turbo_score_batch(pkv_ctx* ctx, const pkv_profile* prof, const uint8_t* payload, uint64_t len,
                          const float* queries, uint32_t nq, float post_scale, float* scores, uint64_t scores_cap,
                          uint64_t* n_out, pkv_error* err) {
    if (err) { err->status = PKV_OK; err->segment = -1; err->index = 0; }
    if (!ctx || !prof || !payload || (nq && !queries)) return PKV_ERR_INVALID_ARG;
    if (prof->kind != PKV_CODEC_TURBO) return PKV_ERR_INVALID_ARG;
    if (!score_profile_ok(prof)) return PKV_ERR_UNSUPPORTED;
    if (!std::isfinite(post_scale)) return PKV_ERR_INVALID_ARG;
    uint64_t n = 0;
    int radii = 0;
    int rc = pkv_parse_header(prof, payload, len, &n, &radii);
    if (rc) { if (err) err->status = rc; return rc; }
    if (n_out) *n_out = n;
    if (n > MAX_SEG_VECTORS || nq > (1u << 24)) return PKV_ERR_INVALID_ARG;
    uint64_t need;
    if (__builtin_mul_overflow(n, static_cast<uint64_t>(nq), &need)) return PKV_ERR_INVALID_ARG;
    if (need && (!scores || scores_cap < need)) return PKV_ERR_CAPACITY;
    const uint64_t blob = pkv_blob_len(prof, radii, n);
    const uint32_t W = pkv_prepared_len(prof);
    auto pad = [](uint64_t b) { return (b + 255) & ~static_cast<uint64_t>(255); };
    const uint64_t q_bytes = static_cast<uint64_t>(nq) * prof->dim * sizeof(float);
    const uint64_t p_bytes = static_cast<uint64_t>(nq) * W * sizeof(float);
    const uint64_t s_bytes = need * sizeof(float);
    std::lock_guard<std::mutex> lock(ctx->mu);
    HIP_TRY(hipSetDevice(ctx->device));
    rc = ensure_io_buf(ctx, pad(blob) + pad(q_bytes) + pad(p_bytes) + pad(s_bytes) + 256);
    if (rc) return rc;
    auto* base = static_cast<uint8_t*>(ctx->io_buf);
    uint8_t* d_wire = base;
    auto* d_q = reinterpret_cast<float*>(base + pad(blob));
    auto* d_p = reinterpret_cast<float*>(base + pad(blob) + pad(q_bytes));
    auto* d_s = reinterpret_cast<float*>(base + pad(blob) + pad(q_bytes) + pad(p_bytes));
    auto* d_st = reinterpret_cast<uint32_t*>(base + pad(blob) + pad(q_bytes) + pad(p_bytes) + pad(s_bytes));
    hipStream_t st = ctx->own_stream;
    HIP_TRY(hipMemcpyAsync(d_wire, payload, blob, hipMemcpyHostToDevice, st));
    if (q_bytes) HIP_TRY(hipMemcpyAsync(d_q, queries, q_bytes, hipMemcpyHostToDevice, st));
    rc = prepare_locked(ctx, prof, d_q, nq, d_p, d_st, st);
    pkv_seg seg{0, 1, 1, 0, static_cast<uint32_t>(n), 1};
    if (!rc)
        rc = score_locked(ctx, prof, radii, d_wire, blob, &seg, 1, d_p, nq, nq, 0, post_scale, d_s, need ? need : 1,
                          n ? n : 1, d_st + 2, st);
    if (rc) { (void)hipStreamSynchronize(st); return rc; }
    uint32_t hs[4];
    {
        const int crc = copy_back(st, hs, d_st, sizeof hs, scores, d_s, s_bytes);
        if (crc) return crc;
    }
    if (hs[0] != STATUS_NONE) {   // prepare_query runs before any score (turbo.rs:316-319)
        if (err) { err->status = PKV_ERR_NONFINITE_INPUT; err->segment = -1; err->index = hs[0] >> 4; }
        return PKV_ERR_NONFINITE_INPUT;
    }
    // the blob is decoded (every code validated, then cursor.finish() rejects
    // trailing bytes, wire.rs:566) before any score is computed
    if (hs[2] == STATUS_NONE && len != blob) {
        if (err) { err->status = PKV_ERR_CORRUPT_PAYLOAD; err->segment = -1; err->index = 0; }
        return PKV_ERR_CORRUPT_PAYLOAD;
    }
    return resolve_score_status(hs + 2, 1, err);
}

uint32_t pkv_record_len(const pkv_profile* prof) { return prof ? record_hdr_len(prof) + record_plen(prof) : 0; }

int pkv_encode_vectors(pkv_ctx* ctx, const pkv_profile* prof, int each, const float* vectors, uint64_t n,
                       uint8_t* out, uint64_t out_cap, uint64_t* out_len, pkv_error* err) {
    if (err) { err->status = PKV_OK; err->segment = -1; err->index = 0; }
    if (!ctx || !prof || (!vectors && n)) return PKV_ERR_INVALID_ARG;
    const uint32_t plen = record_plen(prof), rh = record_hdr_len(prof), hdr = hdr_len(prof);
    const uint64_t rec_bytes = n * (static_cast<uint64_t>(rh) + plen);
    if (out_len) *out_len = rec_bytes;
    if (n == 0) return PKV_OK;                    // Ok(vec![]) (codec.rs:28-30, 596-610)
    if (n > MAX_SEG_VECTORS) return PKV_ERR_INVALID_ARG;
    if (!out || out_cap < rec_bytes) return PKV_ERR_CAPACITY;
    const uint64_t in_bytes = n * prof->dim * sizeof(float);
    const uint64_t blob = hdr + n * static_cast<uint64_t>(plen);
    const uint64_t o_in = 0, o_blob = pad256(in_bytes), o_rec = o_blob + pad256(blob + 4);
    const uint64_t o_st = o_rec + pad256(rec_bytes + 4);
    std::lock_guard<std::mutex> lock(ctx->mu);
    HIP_TRY(hipSetDevice(ctx->device));
    int rc = ensure_io_buf(ctx, o_st + 256);
    if (rc) return rc;
    auto* base = static_cast<uint8_t*>(ctx->io_buf);
    uint8_t* d_blob = base + o_blob;
    uint32_t* d_stat = reinterpret_cast<uint32_t*>(base + o_st);
    hipStream_t st = ctx->own_stream;
    HIP_TRY(hipMemcpyAsync(base + o_in, vectors, in_bytes, hipMemcpyHostToDevice, st));
    pkv_seg seg{0, 0, prof->dim, 0, static_cast<uint32_t>(n), static_cast<uint32_t>(n)};
    const bool per_vector = each != 0 && prof->kind == PKV_CODEC_FIB;
    rc = run_segments_locked(ctx, prof, PKV_RADII_F32, true, PKV_F32, base + o_in, n * prof->dim, &seg, 1, d_blob,
                             blob, d_stat, st, per_vector);
    if (rc) { (void)hipStreamSynchronize(st); return rc; }
    int e = launch_records_pack(d_blob + hdr, base + o_rec, n, plen, rh, record_header(prof), st);
    if (e) { (void)hipStreamSynchronize(st); return hip_status(static_cast<hipError_t>(e)); }
    uint32_t hs[2];
    {
        const int crc = copy_back(st, hs, d_stat, sizeof hs, out, base + o_rec, rec_bytes);
        if (crc) return crc;
    }
    return resolve_status(prof, hs, 1, &seg, err, per_vector);
}

int pkv_decode_vectors(pkv_ctx* ctx, const pkv_profile* prof, int each, const uint8_t* records,
                       const uint64_t* offsets, uint64_t n, float* out, uint64_t out_cap_vectors, pkv_error* err) {
    if (err) { err->status = PKV_OK; err->segment = -1; err->index = 0; }
    if (!ctx || !prof || (n && (!offsets || !records))) return PKV_ERR_INVALID_ARG;
    if (n == 0) return PKV_OK;
    if (n > MAX_SEG_VECTORS) return PKV_ERR_INVALID_ARG;
    if (!out || out_cap_vectors < n) return PKV_ERR_CAPACITY;
    const uint32_t plen = record_plen(prof), rh = record_hdr_len(prof), hdr = hdr_len(prof);
    const uint32_t rec_len = rh + plen;
    for (uint64_t i = 0; i < n; ++i)
        if (offsets[i + 1] < offsets[i]) return PKV_ERR_INVALID_ARG;
    // The adapters' JSON fallback: a payload without the record magic is a
    // serde_json TurboCode / FibCodeV1 (proveKV/src/codec.rs:386-393, 552-561,
    // 622-630, 650-658).  Each one is parsed and checked here, on the host,
    // and stands in the batch as the record of the same code (a failed one as
    // a valid placeholder, its failure kept by index: a deserialize failure
    // at the parse stage, a code that does not fit the profile at the decode
    // stage), so the kernels below decode every payload alike.
    const bool fib = prof->kind == PKV_CODEC_FIB;
    const char* magic = fib ? "FB1" : "TQW1";
    const size_t mlen = fib ? 3 : 4;
    std::vector<uint8_t> conv;          // the batch with JSON payloads replaced
    std::vector<uint64_t> conv_off;
    uint32_t json_parse = STATUS_NONE, json_code = STATUS_NONE;
    for (uint64_t i = 0; i < n; ++i) {
        const uint64_t len_i = offsets[i + 1] - offsets[i];
        const bool json = !(len_i >= mlen && std::memcmp(records + offsets[i], magic, mlen) == 0);
        if (json && conv_off.empty()) {
            if (!prof->json_ok) return PKV_ERR_UNSUPPORTED;
            conv.assign(records + offsets[0], records + offsets[i]);
            conv_off.assign(offsets, offsets + i + 1);
            for (uint64_t& o : conv_off) o -= offsets[0];
        }
        if (conv_off.empty()) continue;
        if (!json) {
            conv.insert(conv.end(), records + offsets[i], records + offsets[i + 1]);
        } else {
            std::vector<uint8_t> pay;
            int stage = 0;
            const int jrc = code_from_json(prof->params, records + offsets[i], len_i, &pay, &stage);
            if (jrc && stage == 0) return jrc;   // not a payload fault (parameters, device)
            const HdrBytes hb = record_header(prof);
            const uint8_t* hbytes = reinterpret_cast<const uint8_t*>(hb.w);
            conv.insert(conv.end(), hbytes, hbytes + rh);
            if (jrc) {
                pay.assign(plen, 0);
                if (fib) { pay[0] = 0x00; pay[1] = 0x3C; }   // fp16 1.0: a valid placeholder norm
                uint32_t& slot = stage == 1 ? json_parse : json_code;
                slot = std::min(slot, static_cast<uint32_t>(i << 4) | KIND_CORRUPT);
            }
            conv.insert(conv.end(), pay.begin(), pay.end());
        }
        conv_off.push_back(conv.size());
    }
    if (!conv_off.empty()) {
        records = conv.data();
        offsets = conv_off.data();
    }
    bool packed = offsets[0] == 0;   // record i at i * rec_len: every valid batch
    for (uint64_t i = 0; i < n; ++i) packed = packed && offsets[i + 1] - offsets[i] == rec_len;
    const uint64_t total = offsets[n];
    const uint64_t blob = hdr + n * static_cast<uint64_t>(plen);
    const uint64_t out_bytes = n * prof->dim * sizeof(float);
    const uint64_t o_out = 0, o_rec = pad256(out_bytes), o_off = o_rec + pad256(total + 4);
    const uint64_t o_blob = o_off + pad256(8 * (n + 1)), o_st = o_blob + pad256(blob + 4);
    std::lock_guard<std::mutex> lock(ctx->mu);
    HIP_TRY(hipSetDevice(ctx->device));
    int rc = ensure_io_buf(ctx, o_st + 256);
    if (rc) return rc;
    auto* base = static_cast<uint8_t*>(ctx->io_buf);
    const uint8_t* d_rec = base + o_rec;
    const uint64_t* d_off = reinterpret_cast<const uint64_t*>(base + o_off);
    uint8_t* d_blob = base + o_blob;
    uint32_t* d_stat = reinterpret_cast<uint32_t*>(base + o_st);   // [0, 1] decode, [2, 3] records
    hipStream_t st = ctx->own_stream;
    if (total) HIP_TRY(hipMemcpyAsync(base + o_rec, records, total, hipMemcpyHostToDevice, st));
    HIP_TRY(hipMemcpyAsync(base + o_off, offsets, 8 * (n + 1), hipMemcpyHostToDevice, st));
    int e = launch_fill_u32(d_stat, STATUS_NONE, 4, st);
    if (!e)
        e = launch_records_check(d_rec, d_off, n, rec_len, rh, fib ? 1u : 0u, packed, record_header(prof), d_stat + 2,
                                 st);
    if (!e) e = launch_records_gather(d_rec, d_off, n, rec_len, rh, packed, d_blob, hdr, blob_header(prof, n), plen, st);
    if (e) { (void)hipStreamSynchronize(st); return hip_status(static_cast<hipError_t>(e)); }
    pkv_seg seg{0, 0, prof->dim, 0, static_cast<uint32_t>(n), static_cast<uint32_t>(n)};
    if (fib && each) {   // FibQuantizer::decode: f64 inverse rotation
        e = launch_fib_decode_f64(fib_dev(prof), d_blob + hdr, n, plen, reinterpret_cast<float*>(base + o_out),
                                  d_stat, st);
        if (e) { (void)hipStreamSynchronize(st); return hip_status(static_cast<hipError_t>(e)); }
    } else {
        rc = run_segments_locked(ctx, prof, PKV_RADII_F32, false, PKV_F32, base + o_out, n * prof->dim, &seg, 1,
                                 d_blob, blob, d_stat, st);
        if (rc) { (void)hipStreamSynchronize(st); return rc; }
    }
    uint32_t hs[4];
    {
        const int crc = copy_back(st, hs, d_stat, sizeof hs, out, base + o_out, out_bytes);
        if (crc) return crc;
    }
    // FibQuantAdapter::decode_batch parses every record before decoding any
    // (codec.rs:639-665); per-record decoding stops at the first failure.
    hs[2] = std::min(hs[2], json_parse);
    hs[3] = std::min(hs[3], json_code);
    uint32_t pick = std::min(std::min(hs[0], hs[1]), hs[3]);
    if (fib && !each && hs[2] != STATUS_NONE) pick = hs[2];
    else pick = std::min(pick, hs[2]);
    if (pick == STATUS_NONE) return PKV_OK;
    if (err) { err->status = PKV_ERR_CORRUPT_PAYLOAD; err->segment = 0; err->index = pick >> 4; }
    return PKV_ERR_CORRUPT_PAYLOAD;
}

int pkv_turbo_constants(uint32_t dim, uint32_t projections, uint64_t seed, float* signs, float* qjl) {
    if (dim == 0 || (dim & (dim - 1)) != 0 || dim > 4096 || !signs) return PKV_ERR_INVALID_ARG;
    std::vector<float> s, g;
    make_turbo_constants(dim, qjl ? projections : 0, seed, s, g);
    std::memcpy(signs, s.data(), s.size() * sizeof(float));
    if (qjl && !g.empty()) std::memcpy(qjl, g.data(), g.size() * sizeof(float));
    return PKV_OK;
}

int pkv_fib_constants(uint32_t dim, uint32_t k, uint32_t n, uint64_t seed, uint32_t training_samples,
                      uint32_t lloyd_restarts, uint32_t lloyd_iterations, float* codebook, double* rotation,
                      double* init_mse, double* training_mse) {
    if (dim == 0 || k == 0 || dim % k != 0 || n < 2 || dim > 4096) return PKV_ERR_INVALID_ARG;
    if (lloyd_restarts == 0 || lloyd_iterations == 0 || training_samples < n) return PKV_ERR_INVALID_ARG;
    if (codebook) {
        std::vector<float> cb;
        int rc = make_fib_codebook(dim, k, n, seed, training_samples, lloyd_restarts, lloyd_iterations, cb, init_mse,
                                   training_mse);
        if (rc) return rc;
        std::memcpy(codebook, cb.data(), cb.size() * sizeof(float));
    }
    if (rotation) {
        std::vector<double> rot, rot_t;
        int rc = make_fib_rotation(dim, seed, rot);
        if (rc) return rc;
        std::memcpy(rotation, rot.data(), rot.size() * sizeof(double));
    }
    return PKV_OK;
}

void pkv_constants_cache_stats(uint64_t* hits, uint64_t* misses, uint64_t* entries) {
    constants_cache_stats(hits, misses, entries);
}

void pkv_constants_cache_clear(void) { constants_cache_clear(); }

void pkv_host_angle_bins(const float* a, const float* b, uint64_t n, uint32_t pbits, uint32_t* out) {
    for (uint64_t i = 0; i < n; ++i) out[i] = pbits == 3 ? angle_bin3(a[i], b[i]) : angle_bin_exact(a[i], b[i], pbits);
}

void pkv_host_octant_bins(const float* a, const float* b, uint64_t n, uint32_t* bins, uint8_t* safe) {
    for (uint64_t i = 0; i < n; ++i) {
        bool unsafe;
        bins[i] = octant_bin_f(a[i], b[i], unsafe);
        // the encode kernels also send a pair whose squares do not sum to a
        // finite value down the exact path (its lane's radius sum is not finite)
        const float aa = a[i] * a[i], bb = b[i] * b[i];
        safe[i] = !unsafe && isfinite_f(aa + bb);
    }
}

void pkv_host_logf(const float* x, uint64_t n, float* out) {
    static const LogfEntry tab[16] = {PKV_LOGF_TABLE};
    for (uint64_t i = 0; i < n; ++i) out[i] = og_logf_normal(x[i], tab);
}

void pkv_host_expf(const float* x, uint64_t n, float* out) {
    static const uint64_t tab[32] = {PKV_EXP2F_TABLE};
    for (uint64_t i = 0; i < n; ++i) out[i] = og_expf(x[i], tab);
}

void pkv_host_expf_fused(const float* x, uint64_t n, float* out) {
    static const uint64_t tab[32] = {PKV_EXP2F_TABLE};
    for (uint64_t i = 0; i < n; ++i) out[i] = og_expf_fused(x[i], tab);
}

void pkv_host_div255(const float* u, uint64_t n, float* out) {
    for (uint64_t i = 0; i < n; ++i) out[i] = div255_f(u[i]);
}

void pkv_host_f32_stable_rel50(const double* v, uint64_t n, uint8_t* out) {
    for (uint64_t i = 0; i < n; ++i) out[i] = f32_rounding_stable_rel50(v[i]) ? 1 : 0;
}

}  // extern "C"
