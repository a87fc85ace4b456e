// lr_build.hip - the BVH builders on gfx950: LBVH (Karras 2012 numbering, built bottom-up in
// one pass after Apetrei 2014) and PLOC (Meister & Bittner 2018, radius 16), over Morton
// codes sorted by an LSD radix sort with decoupled look-back (one kernel per 8-bit digit).
//
// The rules are the reference's (engine/gpu/shaders/trace/trace_build.wgsl,
// trace_ploc.wgsl); the kernels are not: the reference's 210 bitonic steps become 4 radix
// passes, its 54 refit passes one bottom-up pass with per-node arrival counters, and each
// PLOC round (4 dispatches there) one kernel whose cluster windows sit in LDS.
#include <stdarg.h>
#include <stddef.h>
#include <algorithm>
#include <mutex>
#include <stdio.h>

#include "lr_device.h"
#include "lr_internal.h"

namespace {

// Wait until this thread's memory operations are done. Device-scope atomics and stores are
// coherent across the XCDs once done, so a hand-off needs this wait before its flag, not a
// __threadfence (on gfx950 a write-back of the whole L2, here once per wave)
__device__ __forceinline__ void wait_mem()
{
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}


constexpr int BLOCK = 256;
constexpr int SORT_BLOCK = 1024;                // 16 waves per tile: enough in flight per CU
constexpr int SORT_ITEMS = 4;
constexpr int SORT_TILE = SORT_BLOCK * SORT_ITEMS;   // 4096 keys per tile
constexpr int SORT_WAVES = SORT_BLOCK / 64;
constexpr int SORT_PASSES = 4;                  // 30-bit codes: bits 0-7, 8-15, 16-23, 24-29
constexpr int HIST_COPIES = 8;                  // one global histogram per XCD (less contention)
constexpr int PLOC_R = 16;
constexpr int PLOC_MAX_ROUNDS = 128;
// the clusters (estimated) from which a round takes 4 positions a lane (fewer instructions a pair) rather
// than 2 (more waves, each sooner done): at 114k 12.2 against 12.5 us, at 400k 19 against 27, below
// 50k 11 against 8
constexpr int PLOC_BIG = 1 << 17;
constexpr int BOUNDS_BLOCKS = 512;

constexpr uint32_t FLAG_AGG = 1u << 30;
constexpr uint32_t FLAG_PREFIX = 2u << 30;
constexpr int LOOK_BACK = 8;                     // predecessor tiles read at once in a sort pass's look-back
constexpr uint32_t VALUE_MASK = (1u << 30) - 1u;

// ---- block-wide scans (256 threads, wave64) ------------------------------------------------
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

// to the host's memory, seen there once the kernel has ended
__device__ __forceinline__ void tell_depth(LrBuildResult *res, uint32_t depth)
{
    if (res) __hip_atomic_store(&res->depth, depth, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// exclusive scan of one value per thread over a block of NW waves; *total gets the sum
template <int NW>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t *total, uint32_t *s_wsum)
{
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint32_t inc = wave_incl_scan(v);
    if (lane == 63) s_wsum[w] = inc;
    __syncthreads();
    uint32_t off = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < NW; k++) {
        uint32_t s = s_wsum[k];
        off += k < w ? s : 0u;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return off + inc - v;
}

// ---- triangle boxes (scene.c:65-74) --------------------------------------------------------
__global__ __launch_bounds__(BLOCK) void k_tri_boxes(const float4 *__restrict__ tris, int n, float4 *__restrict__ boxes)
{
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    const float4 q = tris[3 * (size_t)i], u = tris[3 * (size_t)i + 1], v = tris[3 * (size_t)i + 2];
    const float qq[3] = {q.x, q.y, q.z}, uu[3] = {u.x, u.y, u.z}, vv[3] = {v.x, v.y, v.z};
    float lo[3], hi[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float a = qq[k] + uu[k], b = qq[k] + vv[k];
        lo[k] = rfmin(rfmin(qq[k], a), b);
        hi[k] = rfmax(rfmax(qq[k], a), b);
    }
    boxes[2 * (size_t)i] = make_float4(lo[0] - 1e-3f, lo[1] - 1e-3f, lo[2] - 1e-3f, 0.0f);
    boxes[2 * (size_t)i + 1] = make_float4(hi[0] + 1e-3f, hi[1] + 1e-3f, hi[2] + 1e-3f, 0.0f);
}

// ---- the bounds of the boxes, and the Morton parameters ---------------------------------------
__device__ __forceinline__ void min6(float *a, const float *b)
{
#pragma unroll
    for (int k = 0; k < 3; k++) { a[k] = rfmin(a[k], b[k]); a[3 + k] = rfmax(a[3 + k], b[3 + k]); }
}

__device__ void block_min6(float *v, float (*s)[6])
{
    // within the wave, then across the 4 waves
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        float t[6];
#pragma unroll
        for (int k = 0; k < 6; k++) t[k] = __shfl_xor(v[k], o, 64);
        min6(v, t);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < 6; k++) s[w][k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int q = 1; q < BLOCK / 64; q++) min6(v, s[q]);
}

__global__ __launch_bounds__(BLOCK) void k_bounds(const float4 *__restrict__ boxes, int n, float *partial,
                                                    uint32_t *ticket, LrBuildParamsDev *out)
{
    __shared__ float s[BLOCK / 64][6];
    __shared__ bool last;
    float v[6] = {1e30f, 1e30f, 1e30f, -1e30f, -1e30f, -1e30f};
    for (int i = blockIdx.x * BLOCK + threadIdx.x; i < n; i += gridDim.x * BLOCK) {
        const float4 a = boxes[2 * (size_t)i], b = boxes[2 * (size_t)i + 1];
        const float t[6] = {a.x, a.y, a.z, b.x, b.y, b.z};
        min6(v, t);
    }
    block_min6(v, s);
    if (threadIdx.x == 0) {
        for (int k = 0; k < 6; k++) st_dev((uint32_t *)&partial[6 * blockIdx.x + k], __float_as_uint(v[k]));
        // the ticket releases this block's partials and, for the last block, acquires the others'
        last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    float w[6] = {1e30f, 1e30f, 1e30f, -1e30f, -1e30f, -1e30f};
    for (int b = threadIdx.x; b < (int)gridDim.x; b += BLOCK) {
        float t[6];
        for (int k = 0; k < 6; k++) t[k] = __uint_as_float(ld_dev((const uint32_t *)&partial[6 * b + k]));
        min6(w, t);
    }
    __syncthreads();
    block_min6(w, s);
    if (threadIdx.x == 0) {
        for (int k = 0; k < 3; k++) {
            const float e = w[3 + k] - w[k];
            out->lo[k] = w[k];
            out->hi[k] = w[3 + k];
            out->ext[k] = e > 0.0f ? (float)(1.0 / (double)e) : 0.0f;   // trace_gpu.c:609-611
        }
        out->lo[3] = out->ext[3] = out->hi[3] = 0.0f;
        *ticket = 0;
    }
}

// bounds given by the caller: only the parameters
__global__ void k_params(LrBuildParamsDev *out, float lx, float ly, float lz, float hx, float hy, float hz)
{
    const float lo[3] = {lx, ly, lz}, hi[3] = {hx, hy, hz};
    for (int k = 0; k < 3; k++) {
        const float e = hi[k] - lo[k];
        out->lo[k] = lo[k];
        out->hi[k] = hi[k];
        out->ext[k] = e > 0.0f ? (float)(1.0 / (double)e) : 0.0f;
    }
    out->lo[3] = out->ext[3] = out->hi[3] = 0.0f;
}

// ---- Morton codes (trace_build.wgsl:16-33) and the sort's global histograms ----------------------
__device__ __forceinline__ uint32_t spread(uint32_t v)
{
    uint32_t x = v & 1023u;
    x = (x | (x << 16u)) & 0x030000ffu;
    x = (x | (x << 8u)) & 0x0300f00fu;
    x = (x | (x << 4u)) & 0x030c30c3u;
    x = (x | (x << 2u)) & 0x09249249u;
    return x;
}

__device__ __forceinline__ uint32_t quant(float c, float lo, float ext)
{
    return (uint32_t)(wmin(wmax((c - lo) * ext, 0.0f), 0.999f) * 1024.0f);
}

// one tile of 4096 items per block: codes (and the items 0..n-1 as the sort's values), the
// four digits' counts into the histograms; the last block to finish turns them into each
// digit's start (exclusive scans) and clears them for the next build. Also clears the memory
// the later kernels expect zeroed (look-back states, tile counters, arrival counters).
__global__ __launch_bounds__(SORT_BLOCK) void k_morton(const float4 *__restrict__ boxes, int n, const LrBuildParamsDev *prm,
                                                    uint32_t *__restrict__ keys, uint32_t *__restrict__ vals,
                                                    uint32_t *hist, uint32_t *ticket, uint32_t *bucket_base,
                                                    uint32_t *zero, size_t zero_words)
{
    __shared__ uint32_t h[SORT_PASSES][256];
    __shared__ uint32_t s_wsum[SORT_WAVES];
    __shared__ bool last;
    for (int i = threadIdx.x; i < SORT_PASSES * 256; i += SORT_BLOCK) (&h[0][0])[i] = 0;
    for (size_t i = blockIdx.x * (size_t)SORT_BLOCK + threadIdx.x; i < zero_words; i += (size_t)gridDim.x * SORT_BLOCK) zero[i] = 0;
    __syncthreads();
    const float lx = prm->lo[0], ly = prm->lo[1], lz = prm->lo[2];
    const float ex = prm->ext[0], ey = prm->ext[1], ez = prm->ext[2];
    const int base = blockIdx.x * SORT_TILE;
    // all the tile's boxes in flight at once, then the codes
    float4 a[SORT_ITEMS], b[SORT_ITEMS];
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; r++) {
        const int i = base + r * SORT_BLOCK + threadIdx.x;
        if (i < n) {
            a[r] = boxes[2 * (size_t)i];
            b[r] = boxes[2 * (size_t)i + 1];
        }
    }
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; r++) {
        const int i = base + r * SORT_BLOCK + threadIdx.x;
        if (i >= n) continue;
        const float cx = (a[r].x + b[r].x) * 0.5f, cy = (a[r].y + b[r].y) * 0.5f, cz = (a[r].z + b[r].z) * 0.5f;
        const uint32_t code = (spread(quant(cx, lx, ex)) << 2u) | (spread(quant(cy, ly, ey)) << 1u) | spread(quant(cz, lz, ez));
        keys[i] = code;
        vals[i] = (uint32_t)i;
#pragma unroll
        for (int p = 0; p < SORT_PASSES; p++) atomicAdd(&h[p][(code >> (8 * p)) & 255u], 1u);
    }
    __syncthreads();
    uint32_t *mine = hist + (blockIdx.x % HIST_COPIES) * SORT_PASSES * 256;
    for (int i = threadIdx.x; i < SORT_PASSES * 256; i += SORT_BLOCK) {
        const uint32_t v = (&h[0][0])[i];
        if (v) atomicAdd(&mine[i], v);
    }
    // The ticket hands the histograms over. They move as device-scope atomics (coherent across
    // the XCDs once done), so the ticket needs every thread's adds done before it (wait_mem:
    // the wait, and compiler barriers on both sides; then the work-group barrier), and the last
    // work-group reads them with device-scope loads after it. An acquire-release ticket instead
    // writes back and invalidates the L2 once per work-group (about 3900 of them at 16M keys):
    // measured 1.68 -> 1.89 ms for a 16M build together with the bounds kernel's.
    wait_mem();
    __syncthreads();
    if (threadIdx.x == 0) last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    __syncthreads();
    if (!last) return;
    // the last block: thread t sums digit t % 256 of pass t / 256 over the copies (all the
    // copies' loads in flight together), clears them, and the passes are scanned side by side
    // (four waves per pass)
    static_assert(SORT_BLOCK == SORT_PASSES * 256, "one thread per (pass, digit)");
    uint32_t c8[HIST_COPIES];
#pragma unroll
    for (int c = 0; c < HIST_COPIES; c++) c8[c] = ld_dev(&hist[c * SORT_PASSES * 256 + threadIdx.x]);
    uint32_t v = 0;
#pragma unroll
    for (int c = 0; c < HIST_COPIES; c++) {
        v += c8[c];
        st_dev(&hist[c * SORT_PASSES * 256 + threadIdx.x], 0u);
    }
    const int w = threadIdx.x >> 6;
    const uint32_t inc = wave_incl_scan(v);
    if ((threadIdx.x & 63) == 63) s_wsum[w] = inc;
    __syncthreads();
    uint32_t off = 0;
    for (int k = w & ~3; k < w; k++) off += s_wsum[k];
    bucket_base[threadIdx.x] = off + inc - v;
    if (threadIdx.x == 0) *ticket = 0;
}

// ---- one radix-sort pass: 8 bits, stable, decoupled look-back (onesweep) -------------------------
// Each wave ranks its 1024 keys (16 rounds of 64, wave-contiguous, so the rank order is the
// input order) with a 64-lane match over the digit's 8 bits; per-wave digit counts give each
// key its place in the tile; the tile's place in each digit's run comes from the tiles before
// it (look-back over per-tile, per-digit states). The tile is reordered in LDS first, so that
// the stores to each digit's run are contiguous.
__global__ __launch_bounds__(SORT_BLOCK) void k_sort_pass(const uint32_t *__restrict__ kin, const uint32_t *__restrict__ vin,
                                                       uint32_t *__restrict__ kout, uint32_t *__restrict__ vout, int n,
                                                       int shift, const uint32_t *__restrict__ bucket_base,
                                                       uint32_t *status, uint32_t *tile_ctr)
{
    __shared__ uint32_t s_tile;
    __shared__ uint32_t wc[SORT_WAVES][256];
    __shared__ uint32_t s_start[256];
    __shared__ uint32_t s_glob[256];
    __shared__ uint32_t s_wsum[SORT_WAVES];
    __shared__ uint32_t s_k[SORT_TILE];
    __shared__ uint32_t s_v[SORT_TILE];
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    if (tid == 0) s_tile = atomicAdd(tile_ctr, 1u);
    for (int i = tid; i < SORT_WAVES * 256; i += SORT_BLOCK) (&wc[0][0])[i] = 0;
    __syncthreads();
    const uint32_t tile = s_tile;
    const int base = (int)tile * SORT_TILE;
    uint32_t k[SORT_ITEMS], v[SORT_ITEMS], rank[SORT_ITEMS];
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; r++) {
        const int i = base + w * (64 * SORT_ITEMS) + r * 64 + lane;
        const bool ok = i < n;
        k[r] = ok ? kin[i] : 0u;
        v[r] = ok ? vin[i] : 0u;
    }
    const uint64_t lt = lanemask_lt();
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; r++) {
        const int i = base + w * (64 * SORT_ITEMS) + r * 64 + lane;
        const bool ok = i < n;
        const uint32_t d = (k[r] >> shift) & 255u;
        uint64_t peers = __ballot(ok);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const uint64_t bal = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? bal : ~bal;
        }
        const uint32_t before = ok ? wc[w][d] : 0u;
        rank[r] = before + (uint32_t)__popcll(peers & lt);
        __builtin_amdgcn_wave_barrier();
        if (ok && (peers & lt) == 0) wc[w][d] = before + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // threads 0..255: digit tid
    const bool dig = tid < 256;
    uint32_t tot = 0;
    if (dig) {
        for (int q = 0; q < SORT_WAVES; q++) { const uint32_t c = wc[q][tid]; wc[q][tid] = tot; tot += c; }
        if (tile == 0) st_dev(&status[tid], FLAG_PREFIX | tot);
        else st_dev(&status[tile * 256 + tid], FLAG_AGG | tot);
    }
    uint32_t all;
    const uint32_t start = block_excl_scan<SORT_WAVES>(tot, &all, s_wsum);
    uint32_t excl = 0;
    if (dig && tile > 0) {
        // LOOK_BACK tiles at a time (their loads in flight together): the nearest prefix among
        // them ends the walk; a tile not yet posted means the same window again
        int t = (int)tile - 1;
        for (;;) {
            uint32_t sv[LOOK_BACK];
#pragma unroll
            for (int k = 0; k < LOOK_BACK; k++) sv[k] = t - k >= 0 ? ld_dev(&status[(t - k) * 256 + tid]) : FLAG_PREFIX;
            bool wait = false, done = false;
            uint32_t add = 0;
#pragma unroll
            for (int k = 0; k < LOOK_BACK; k++) {
                if (done || wait) continue;
                const uint32_t f = sv[k] & ~VALUE_MASK;
                if (f == 0) wait = true;
                else {
                    add += sv[k] & VALUE_MASK;
                    done = f == FLAG_PREFIX;
                }
            }
            if (wait) {
                __builtin_amdgcn_s_sleep(1);
                continue;
            }
            excl += add;
            if (done) break;
            t -= LOOK_BACK;
        }
        st_dev(&status[tile * 256 + tid], FLAG_PREFIX | (excl + tot));
    }
    if (dig) {
        s_start[tid] = start;
        s_glob[tid] = bucket_base[tid] + excl - start;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; r++) {
        const int i = base + w * (64 * SORT_ITEMS) + r * 64 + lane;
        if (i < n) {
            const uint32_t d = (k[r] >> shift) & 255u;
            const uint32_t pos = s_start[d] + wc[w][d] + rank[r];
            s_k[pos] = k[r];
            s_v[pos] = v[r];
        }
    }
    __syncthreads();
    const int cnt = n - base < SORT_TILE ? n - base : SORT_TILE;
    for (int s = tid; s < cnt; s += SORT_BLOCK) {
        const uint32_t key = s_k[s];
        const uint32_t g = s_glob[(key >> shift) & 255u] + (uint32_t)s;
        kout[g] = key;
        vout[g] = s_v[s];
    }
}

// ---- LBVH, bottom-up in one pass -----------------------------------------------------------------
// delta of adjacent keys k, k+1 (trace_build.wgsl:52-58)
__device__ __forceinline__ int dadj(const uint32_t *codes, int k)
{
    const uint32_t a = codes[k], b = codes[k + 1];
    return a == b ? 32 + __clz((uint32_t)k ^ (uint32_t)(k + 1)) : __clz(a ^ b);
}

// is the node over keys [l, r] (not the root) its parent's left child? (its parent splits at r)
__device__ __forceinline__ bool is_left(const uint32_t *codes, int n, int l, int r)
{
    return l == 0 || (r != n - 1 && dadj(codes, r) > dadj(codes, l - 1));
}

__device__ __forceinline__ void put_node(LrNode *p, float lx, float ly, float lz, uint32_t a, float hx, float hy, float hz, uint32_t b)
{
    float4 *q = reinterpret_cast<float4 *>(p);
    q[0] = make_float4(lx, ly, lz, __uint_as_float(a));
    q[1] = make_float4(hx, hy, hz, __uint_as_float(b));
}

// a node record written through to the coherence point (sc1 stores), so that another XCD's
// thread reading it with ld_dev64 sees it without a cache-wide write-back
__device__ __forceinline__ void put_node_dev(LrNode *p, float lx, float ly, float lz, uint32_t a, float hx, float hy, float hz,
                                             uint32_t b)
{
    uint64_t *q = reinterpret_cast<uint64_t *>(p);
    st_dev64(q + 0, ((uint64_t)__float_as_uint(ly) << 32) | __float_as_uint(lx));
    st_dev64(q + 1, ((uint64_t)a << 32) | __float_as_uint(lz));
    st_dev64(q + 2, ((uint64_t)__float_as_uint(hy) << 32) | __float_as_uint(hx));
    st_dev64(q + 3, ((uint64_t)b << 32) | __float_as_uint(hz));
}

// The same through a buffer resource: a record as two 16-byte stores (and loads), sc1 (device
// scope, through to the coherence point) as st_dev64 / ld_dev64 but half the transactions. The
// resource covers 2 GiB from the records' base (the host takes this path only below that).
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
constexpr int CPOL_SC1 = 16;   // the sc1 cache-policy bit of gfx950's memory instructions
__device__ __forceinline__ __amdgpu_buffer_rsrc_t node_rsrc(LrNode *base)
{
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, 0x7fffffff, 0x00020000);
}
__device__ __forceinline__ void put_node_buf(__amdgpu_buffer_rsrc_t rs, int idx, float lx, float ly, float lz, uint32_t a,
                                             float hx, float hy, float hz, uint32_t b)
{
    const u32x4 lo = {__float_as_uint(lx), __float_as_uint(ly), __float_as_uint(lz), a};
    const u32x4 hi = {__float_as_uint(hx), __float_as_uint(hy), __float_as_uint(hz), b};
    __builtin_amdgcn_raw_buffer_store_b128(lo, rs, idx * 32, 0, CPOL_SC1);
    __builtin_amdgcn_raw_buffer_store_b128(hi, rs, idx * 32 + 16, 0, CPOL_SC1);
}

// min-scans over a group of NT threads (NT / 64 waves): forward (the minimum of this and every
// earlier thread's value) and backward (this and every later thread's)
template <int NT>
__device__ __forceinline__ int block_min_scan(int v, bool backward, int *s_w)
{
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = backward ? __shfl_down(v, o, 64) : __shfl_up(v, o, 64);
        if (backward ? lane + o < 64 : lane >= o) v = t < v ? t : v;
    }
    if (lane == (backward ? 0 : 63)) s_w[w] = v;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NT / 64; k++) {
        const int t = s_w[k];
        if (backward ? k > w : k < w) v = t < v ? t : v;
    }
    __syncthreads();
    return v;
}

// The LBVH's nodes bottom-up (leaves, trace_build.wgsl:98-107; up, :109-122): from each
// leaf a thread climbs; at each parent the first of the two children to arrive stops, the
// second joins their boxes (min / max of left, right), writes the parent with Karras's
// numbering (internal i at node0 + i, leaf j at node0 + n - 1 + j) and goes on.
//
// Two kernels. k_lbvh: a work-group's LBVH_GROUP leaves climb through the nodes whose key ranges lie
// inside the group's: the two children's threads are then both in the group, and hand their
// boxes over in LDS (a slot per side, an LDS arrival counter). Whether a node's parent lies
// inside is decided from the adjacent-key deltas d(k) alone: a left child [l, p]'s parent ends
// at the first k > p with d(k) < d(p), a right child [p + 1, r]'s starts after the last k < p
// with d(k) < d(p); a min-scan of the group's deltas each way answers both with one
// comparison. A node whose parent lies outside (the root of a largest subtree inside the
// group: at most LBVH_GROUP of them, about 10 on random keys) is written and listed in the group's
// slots. k_lbvh_top then climbs from the listed nodes, one wave per group's list, through
// device memory: the two children's threads are on any XCDs, whose L2s are not coherent, so a
// record is stored through to the coherence point (sc1), the stores are waited for (vmcnt 0),
// and only then does the thread mark its arrival, with its subtree's far end and height in the
// one 64-bit word it swaps in; the second thread reads the record back with sc1 loads (a leaf
// child's box from the input boxes). Kept apart, the few long climbs through device memory
// do not hold the groups of the first kernel, and their LDS, on the compute units.
constexpr int LBVH_GROUP = 512;      // leaves per work-group of k_lbvh (1024 measured 13 % slower: one per CU)
constexpr int LBVH_SLOTS = LBVH_GROUP;   // listed nodes per group, at most

__global__ __launch_bounds__(LBVH_GROUP) void k_lbvh(const uint32_t *__restrict__ codes, const uint32_t *__restrict__ items,
                                                const float4 *__restrict__ boxes, int n, uint32_t node0, uint32_t ref0,
                                                uint32_t ref_add, LrNode *__restrict__ nodes, uint32_t *__restrict__ aux,
                                                uint4 *__restrict__ esc, uint32_t *__restrict__ esc_count,
                                                LrBuildResult *res)
{
    __shared__ int s_d[LBVH_GROUP + 1];        // d(B0 - 1 + i); -1 (below every delta) off the keys' ends
    __shared__ int s_pmin[LBVH_GROUP + 1];     // min of s_d[0 .. i]
    __shared__ int s_smin[LBVH_GROUP + 1];     // min of s_d[i .. LBVH_GROUP] (i >= 1)
    __shared__ float s_box[LBVH_GROUP][2][6];  // per parent split, per side: the arriving child's box
    __shared__ uint32_t s_end[LBVH_GROUP][2], s_h[LBVH_GROUP][2], s_arrive[LBVH_GROUP];
    __shared__ int s_w[LBVH_GROUP / 64];
    __shared__ uint32_t s_nesc;
    const int t = threadIdx.x;
    const int B0 = blockIdx.x * LBVH_GROUP;
    const int j = B0 + t;
    const bool live = j < n;
    float lx = 0.0f, ly = 0.0f, lz = 0.0f, hx = 0.0f, hy = 0.0f, hz = 0.0f;
    if (live) {
        const uint32_t item = items[j];
        const float4 blo = boxes[2 * (size_t)item], bhi = boxes[2 * (size_t)item + 1];
        lx = blo.x; ly = blo.y; lz = blo.z; hx = bhi.x; hy = bhi.y; hz = bhi.z;
        aux[j] = item + ref_add;
        if (n > 1) put_node(&nodes[n - 1 + j], lx, ly, lz, ref0 + (uint32_t)j, hx, hy, hz, 0x80000001u);
        else {
            put_node(&nodes[0], lx, ly, lz, ref0, hx, hy, hz, 0x80000001u);
            tell_depth(res, 1u);
        }
    }
    if (n == 1) {   // (uniform: the one group returns before any barrier)
        if (t == 0) esc_count[0] = 0u;
        return;
    }
    const int dj = j < n - 1 ? dadj(codes, j) : -1;
    s_d[t + 1] = dj;
    if (t == 0) {
        s_d[0] = B0 > 0 ? dadj(codes, B0 - 1) : -1;
        s_nesc = 0u;
    }
    s_arrive[t] = 0u;
    __syncthreads();
    const int d0 = s_d[0];
    const int pm = block_min_scan<LBVH_GROUP>(dj, false, s_w);
    const int sm = block_min_scan<LBVH_GROUP>(dj, true, s_w);
    s_pmin[t + 1] = pm < d0 ? pm : d0;
    s_smin[t + 1] = sm;
    if (t == 0) s_pmin[0] = d0;
    __syncthreads();

    // d(k) = s_d[k - B0 + 1] for B0 - 1 <= k <= B0 + LBVH_GROUP - 1
    int l = j, r = j;      // the node reached: keys [l, r] (a leaf while l == r)
    int lc = 0, rc = 0;    // an inner node's children
    uint32_t h = 1;
    bool climbing = live;
    bool left = live && s_d[r - B0 + 1] > s_d[l - B0];
    while (climbing) {
        const int p = left ? r : l - 1;
        const int dp = s_d[p - B0 + 1];
        const bool inside = left ? (p <= B0 + LBVH_GROUP - 2 && s_smin[p - B0 + 2] < dp) : (p >= B0 && s_pmin[p - B0] < dp);
        if (l != r) put_node(&nodes[left ? r : l], lx, ly, lz, node0 + (uint32_t)lc, hx, hy, hz, node0 + (uint32_t)rc);
        if (!inside) {   // listed for k_lbvh_top (its record, or its leaf's, holds its box)
            const uint32_t k = atomicAdd(&s_nesc, 1u);
            esc[(size_t)blockIdx.x * LBVH_SLOTS + k] = make_uint4((uint32_t)l, (uint32_t)r, h, 0u);
            break;
        }
        const int sl = p - B0, side = left ? 0 : 1;
        float *bx = s_box[sl][side];
        bx[0] = lx; bx[1] = ly; bx[2] = lz; bx[3] = hx; bx[4] = hy; bx[5] = hz;
        s_end[sl][side] = (uint32_t)(left ? l : r);
        s_h[sl][side] = h;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        if (atomicAdd(&s_arrive[sl], 1u) == 0u) break;   // the sibling's thread goes on
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        const float *ob = s_box[sl][side ^ 1];
        const int oend = (int)s_end[sl][side ^ 1];
        const uint32_t sh = s_h[sl][side ^ 1];
        const int L = left ? l : oend, R = left ? oend : r;
        if (left) {
            lx = wmin(lx, ob[0]); ly = wmin(ly, ob[1]); lz = wmin(lz, ob[2]);
            hx = wmax(hx, ob[3]); hy = wmax(hy, ob[4]); hz = wmax(hz, ob[5]);
        } else {
            lx = wmin(ob[0], lx); ly = wmin(ob[1], ly); lz = wmin(ob[2], lz);
            hx = wmax(ob[3], hx); hy = wmax(ob[4], hy); hz = wmax(ob[5], hz);
        }
        h = 1 + (h > sh ? h : sh);
        lc = L == p ? n - 1 + p : p;
        rc = p + 1 == R ? n + p : p + 1;
        l = L; r = R;
        if (l == 0 && r == n - 1) {
            put_node(&nodes[0], lx, ly, lz, node0 + (uint32_t)lc, hx, hy, hz, node0 + (uint32_t)rc);
            tell_depth(res, h);
            break;
        }
        left = s_d[r - B0 + 1] > s_d[l - B0];
    }
    __syncthreads();
    if (t == 0) esc_count[blockIdx.x] = s_nesc;
}

// BUF: the records through a buffer resource (16-byte device-scope accesses)
template <bool BUF>
__global__ __launch_bounds__(BLOCK) void k_lbvh_top(const uint32_t *__restrict__ codes, const uint32_t *__restrict__ items,
                                                      const float4 *__restrict__ boxes, int n, int groups, uint32_t node0,
                                                      LrNode *nodes, unsigned long long *other, const uint4 *__restrict__ esc,
                                                      const uint32_t *__restrict__ esc_count, LrBuildResult *res)
{
    const int g = blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6);   // one wave per group's list
    if (g >= groups) return;
    const uint32_t cnt = esc_count[g];
    const __amdgpu_buffer_rsrc_t rs = node_rsrc(nodes);
    for (uint32_t k = threadIdx.x & 63; k < cnt; k += 64) {
        const uint4 q = esc[(size_t)g * LBVH_SLOTS + k];
        int l = (int)q.x, r = (int)q.y;
        uint32_t h = q.z;
        bool left = is_left(codes, n, l, r);
        const int me = l == r ? n - 1 + l : (left ? r : l);
        const float4 *rec = reinterpret_cast<const float4 *>(&nodes[me]);   // written by k_lbvh
        const float4 blo = rec[0], bhi = rec[1];
        float lx = blo.x, ly = blo.y, lz = blo.z, hx = bhi.x, hy = bhi.y, hz = bhi.z;
        for (;;) {
            const int p = left ? r : l - 1;             // the parent's split
            const int end = left ? l : r;
            // The arrival hands this subtree's record over. The records move as device-scope
            // accesses (sc1 stores and loads, coherent across the XCDs once done), so the
            // exchange needs only this thread's stores done before it (wait_mem: the wait, and
            // compiler barriers on both sides), and the second to arrive reads the first's record
            // at an address taken from the exchanged value, after it. An acquire-release exchange
            // instead writes back and invalidates the L2 at every climb: measured 1.68 -> 6.9 ms
            // for a 16M build.
            wait_mem();
            const unsigned long long mine = ((unsigned long long)h << 32) | ((uint32_t)end + 1u);
            const unsigned long long o = __hip_atomic_exchange(&other[p], mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (o == 0) break;                          // the sibling is not done: it goes on
            const int oend = (int)(uint32_t)o - 1;
            const uint32_t sh = (uint32_t)(o >> 32);
            const int L = left ? end : oend, R = left ? oend : end;
            const int lc = L == p ? n - 1 + p : p, rc = p + 1 == R ? n + p : p + 1;
            const int sib = left ? rc : lc;
            float sx, sy, sz, tx, ty, tz;
            if (sib >= n - 1) {   // a leaf: its box is the input's
                const uint32_t it = items[sib - (n - 1)];
                const float4 a = boxes[2 * (size_t)it], b = boxes[2 * (size_t)it + 1];
                sx = a.x; sy = a.y; sz = a.z; tx = b.x; ty = b.y; tz = b.z;
            } else if (BUF) {
                const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(rs, sib * 32, 0, CPOL_SC1);
                const u32x4 b = __builtin_amdgcn_raw_buffer_load_b128(rs, sib * 32 + 16, 0, CPOL_SC1);
                sx = __uint_as_float(a.x); sy = __uint_as_float(a.y); sz = __uint_as_float(a.z);
                tx = __uint_as_float(b.x); ty = __uint_as_float(b.y); tz = __uint_as_float(b.z);
            } else {
                const uint64_t *sp = reinterpret_cast<const uint64_t *>(&nodes[sib]);
                const uint64_t q0 = ld_dev64(sp), q1 = ld_dev64(sp + 1), q2 = ld_dev64(sp + 2), q3 = ld_dev64(sp + 3);
                sx = __uint_as_float((uint32_t)q0); sy = __uint_as_float((uint32_t)(q0 >> 32));
                sz = __uint_as_float((uint32_t)q1);
                tx = __uint_as_float((uint32_t)q2); ty = __uint_as_float((uint32_t)(q2 >> 32));
                tz = __uint_as_float((uint32_t)q3);
            }
            float nlx, nly, nlz, nhx, nhy, nhz;
            if (left) {
                nlx = wmin(lx, sx); nly = wmin(ly, sy); nlz = wmin(lz, sz);
                nhx = wmax(hx, tx); nhy = wmax(hy, ty); nhz = wmax(hz, tz);
            } else {
                nlx = wmin(sx, lx); nly = wmin(sy, ly); nlz = wmin(sz, lz);
                nhx = wmax(tx, hx); nhy = wmax(ty, hy); nhz = wmax(tz, hz);
            }
            lx = nlx; ly = nly; lz = nlz; hx = nhx; hy = nhy; hz = nhz;
            h = 1 + (h > sh ? h : sh);
            l = L; r = R;
            if (l == 0 && r == n - 1) {
                put_node(&nodes[0], lx, ly, lz, node0 + (uint32_t)lc, hx, hy, hz, node0 + (uint32_t)rc);
                tell_depth(res, h);
                break;
            }
            left = is_left(codes, n, l, r);
            const int mi = left ? r : l;
            if (BUF) put_node_buf(rs, mi, lx, ly, lz, node0 + (uint32_t)lc, hx, hy, hz, node0 + (uint32_t)rc);
            else put_node_dev(&nodes[mi], lx, ly, lz, node0 + (uint32_t)lc, hx, hy, hz, node0 + (uint32_t)rc);
        }
    }
}

// ---- PLOC ------------------------------------------------------------------------------------
struct PlocState {
    uint32_t nc;          // clusters in the current list
    uint32_t parity;      // which of the two lists is current
    uint64_t live;        // the live clusters summed over the rounds (the build's traffic)
    uint32_t made;        // the rounds k_ploc_round made (a launch may find nothing left to do)
    uint32_t pad[59];
    uint32_t ctr[PLOC_MAX_ROUNDS];   // each round's tile counter
};

// area (trace_ploc.wgsl:18), no fused multiply-add: ((ex*ey) + (ey*ez)) + (ez*ex)
__device__ __forceinline__ float half_area(float lx, float ly, float lz, float hx, float hy, float hz)
{
    const float ex = hx - lx, ey = hy - ly, ez = hz - lz;
    const float a = ex * ey, b = ey * ez, c = ez * ex;
    const float s = a + b;
    return s + c;
}

// nearer (trace_ploc.wgsl:60-66)
__device__ __forceinline__ bool nearer(float d, uint32_t i, uint32_t j, float bd, uint32_t bj)
{
    if (bj == LR_NONE || d < bd) return true;
    if (d > bd) return false;
    const uint32_t mn = min(i, j), bmn = min(i, bj);
    return mn < bmn || (mn == bmn && max(i, j) < max(i, bj));
}

// final_node (trace_ploc.wgsl:33-38) of cluster x with box (lo, hi)
__device__ __forceinline__ void put_final(LrNode *slot, uint32_t x, float4 lo, float4 hi, uint32_t n, uint32_t node0, uint32_t ref0)
{
    if (x < n - 1u) put_node(slot, lo.x, lo.y, lo.z, node0 + 1u + 2u * x, hi.x, hi.y, hi.z, node0 + 2u + 2u * x);
    else put_node(slot, lo.x, lo.y, lo.z, ref0 + x - (n - 1u), hi.x, hi.y, hi.z, 0x80000001u);
}

// merge (trace_ploc.wgsl:39-46): clusters c (the lower position) and d into internal k. A cluster's
// box carries its height in its first word's fourth place (one load less for each side of a merge)
__device__ __forceinline__ uint32_t height_of(float4 lo) { return __float_as_uint(lo.w); }
__device__ __forceinline__ void ploc_merge(uint32_t k, uint32_t c, float4 clo, float4 chi, uint32_t d, float4 dlo, float4 dhi,
                                           uint32_t n, uint32_t node0, uint32_t ref0, float4 *bx, LrNode *nodes)
{
    const float4 lo = make_float4(wmin(clo.x, dlo.x), wmin(clo.y, dlo.y), wmin(clo.z, dlo.z),
                                  __uint_as_float(1u + max(height_of(clo), height_of(dlo))));
    const float4 hi = make_float4(wmax(chi.x, dhi.x), wmax(chi.y, dhi.y), wmax(chi.z, dhi.z), 0.0f);
    bx[2 * (size_t)k] = lo;
    bx[2 * (size_t)k + 1] = hi;
    put_final(&nodes[1 + 2 * (size_t)k], c, clo, chi, n, node0, ref0);
    put_final(&nodes[2 + 2 * (size_t)k], d, dlo, dhi, n, node0, ref0);
    if (k == 0) put_node(&nodes[0], lo.x, lo.y, lo.z, node0 + 1u, hi.x, hi.y, hi.z, node0 + 2u);
}

// init (trace_ploc.wgsl:68-82): the leaves in Morton order are the first clusters
__global__ __launch_bounds__(BLOCK) void k_ploc_init(const uint32_t *__restrict__ items, const float4 *__restrict__ boxes, int n,
                                                       uint32_t ref0, uint32_t ref_add, uint32_t *aux, float4 *bx, uint32_t *list0,
                                                       PlocState *st, uint64_t *status, size_t status_words)
{
    const size_t g = blockIdx.x * (size_t)BLOCK + threadIdx.x;
    for (size_t i = g; i < status_words; i += (size_t)gridDim.x * BLOCK) status[i] = 0;
    if (g < sizeof(PlocState) / 4) reinterpret_cast<uint32_t *>(st)[g] = g == 0 ? (uint32_t)n : 0u;
    if (g >= (size_t)n) return;
    const int i = (int)g;
    const uint32_t item = items[i];
    const size_t x = (size_t)n - 1 + i;
    const float4 lo = boxes[2 * (size_t)item];
    bx[2 * x] = make_float4(lo.x, lo.y, lo.z, __uint_as_float(1u));
    bx[2 * x + 1] = boxes[2 * (size_t)item + 1];
    aux[i] = item + ref_add;
    list0[i] = (uint32_t)x;
}

// The nearest search of a wave, P adjacent positions a lane (their boxes b: three lows, three highs).
// Each pair i, i + k (k <= R) is measured once, for both: by the lane of i, against a copy of the
// boxes that turns by one lane after another, along with the best found so far for its positions
// from below. No memory is read, and a distance serves two positions: 11 to 14 instructions a position
// and neighbour, where a search of R neighbours a side from LDS took about 40 and waited for each. off: the nearest as an offset (0: none) by
// nearer's order (of equal ones the lower position), right for the wave's positions that have all
// R neighbours in it on either side (the others' are not to be used). Where there is no position,
// NEAR_NONE boxes: their distances are infinite and never taken. Floats compare as in nearer but
// for NaN, so boxes must be `measurable`; others take nearest_in.
constexpr float NEAR_NONE = 1e30f;   // lows -, highs +: the area overflows
__device__ __forceinline__ bool measurable(float lx, float ly, float lz, float hx, float hy, float hz)
{
    // finite, and any two boxes' area finite: at most 3 (2e18)^2
    return fabsf(lx) + fabsf(ly) + fabsf(lz) + fabsf(hx) + fabsf(hy) + fabsf(hz) <= 1e18f;
}
__device__ __forceinline__ float turn_lane(float v)   // lane l gets lane l + 1's, the last the first's
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x134, 0xf, 0xf, true));
}
__device__ __forceinline__ int turn_lane(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x134, 0xf, 0xf, true); }

template <int P>
__device__ __forceinline__ void nearest_wave(const float (&b)[6][P], int (&off)[P])
{
    static_assert(PLOC_R % P == 0, "a lane's positions divide the radius");
    const float inf = __builtin_inff();
    float s[6][P], fd[P], sd[P];   // the turning boxes; the best distance above, below
    int fk[P], sk[P];
#pragma unroll
    for (int q = 0; q < P; q++) {
        for (int c = 0; c < 6; c++) s[c][q] = b[c][q];
        fd[q] = sd[q] = inf;
        fk[q] = sk[q] = 0;
    }
#pragma unroll
    for (int t = 0; t <= PLOC_R / P; t++) {
        if (t > 0) {
#pragma unroll
            for (int q = 0; q < P; q++) {
                for (int c = 0; c < 6; c++) s[c][q] = turn_lane(s[c][q]);
                sd[q] = turn_lane(sd[q]);
                sk[q] = turn_lane(sk[q]);
            }
        }
        // (in this order both sides see their distances by rising k: above, the first of equal
        // ones is the lower position; below, the last)
#pragma unroll
        for (int r = P - 1; r >= 0; r--)
#pragma unroll
            for (int q = 0; q < P; q++) {
                const int k = t * P + q - r;
                if (k < 1 || k > PLOC_R) continue;
                const float d = half_area(fminf(b[0][r], s[0][q]), fminf(b[1][r], s[1][q]), fminf(b[2][r], s[2][q]),
                                          fmaxf(b[3][r], s[3][q]), fmaxf(b[4][r], s[4][q]), fmaxf(b[5][r], s[5][q]));
                if (d < fd[r]) { fd[r] = d; fk[r] = k; }
                if (d <= sd[q]) { sd[q] = d; sk[q] = k; }
            }
    }
    const int home = ((int)(threadIdx.x & 63u) - PLOC_R / P) & 63;
#pragma unroll
    for (int q = 0; q < P; q++) {
        const float bd = __shfl(sd[q], home, 64);
        const int bk = __shfl(sk[q], home, 64);
        off[q] = bd <= fd[q] ? (bd < inf ? -bk : 0) : fk[q];
    }
}

// the offset to the nearest of position i (< nc) in a list of nc whose boxes are l[0..5][at + position]:
// any boxes, NaN too
template <class Arr>
__device__ int nearest_in(int i, int nc, int at, const Arr &l)
{
    const int j0 = max(i - PLOC_R, 0), j1 = min(i + PLOC_R, nc - 1);
    const int li = at + i;
    float bd = 0.0f;
    uint32_t bj = LR_NONE;
    for (int j = j0; j <= j1; j++) {
        if (j == i) continue;
        const int lj = at + j;
        const float d = half_area(wmin(l[0][li], l[0][lj]), wmin(l[1][li], l[1][lj]), wmin(l[2][li], l[2][lj]),
                                  wmax(l[3][li], l[3][lj]), wmax(l[4][li], l[4][lj]), wmax(l[5][li], l[5][lj]));
        if (nearer(d, (uint32_t)i, (uint32_t)j, bd, bj)) { bd = d; bj = (uint32_t)j; }
    }
    return bj == LR_NONE ? 0 : (int)bj - i;
}

// The nearest of the positions i0 .. i0 + 64 P - 2R of a list of nc, by one wave, as offsets to
// nn[i - i0], from boxes in LDS (l[c][at + position]; readable from position i0 - R to
// i0 + 64 P - R, whatever they hold where there is none). at + i0 - R is a multiple of P.
template <int P, class Arr>
__device__ __forceinline__ void nearest_range(int i0, int nc, int at, const Arr &l, int8_t *nn)
{
    const int lane = (int)(threadIdx.x & 63u), p0 = i0 - PLOC_R + P * lane;
    float b[6][P];
    bool bad = false;
#pragma unroll
    for (int c = 0; c < 6; c++) {
        struct alignas(4 * P) Row { float v[P]; };
        const Row row = *reinterpret_cast<const Row *>(&l[c][at + p0]);
#pragma unroll
        for (int q = 0; q < P; q++) b[c][q] = row.v[q];
    }
#pragma unroll
    for (int q = 0; q < P; q++) {
        const bool is = p0 + q >= 0 && p0 + q < nc;
        bad |= is && !measurable(b[0][q], b[1][q], b[2][q], b[3][q], b[4][q], b[5][q]);
#pragma unroll
        for (int c = 0; c < 6; c++) b[c][q] = is ? b[c][q] : c < 3 ? -NEAR_NONE : NEAR_NONE;
    }
    if (__any(bad)) {
        for (int o = lane; o < 64 * P - 2 * PLOC_R; o += 64)
            if (i0 + o >= 0 && i0 + o < nc) nn[o] = (int8_t)nearest_in(i0 + o, nc, at, l);
        return;
    }
    int off[P];
    nearest_wave<P>(b, off);
#pragma unroll
    for (int q = 0; q < P; q++) {
        const int o = P * lane + q - PLOC_R;
        if (o >= 0 && o < 64 * P - 2 * PLOC_R && i0 + o >= 0 && i0 + o < nc) nn[o] = (int8_t)off[q];
    }
}

// The places of a thread's positions among a work-group's that stay and that merge (high and low 16
// bits; PER adjacent positions a thread, so the order is the positions'), from ballots: `total`
// the work-group's, by one barrier. wsum (NW words) is free again at the caller's next barrier.
template <int NW, int PER>
__device__ __forceinline__ uint32_t places(const bool (&keep)[PER], const bool (&merge)[PER], uint32_t *total, uint32_t *wsum)
{
    uint32_t before = 0, sum = 0;
#pragma unroll
    for (int q = 0; q < PER; q++) {
        const uint64_t kb = __ballot(keep[q]), mb = __ballot(merge[q]);
        before += (__builtin_amdgcn_mbcnt_hi((uint32_t)(kb >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)kb, 0u)) << 16) +
                  __builtin_amdgcn_mbcnt_hi((uint32_t)(mb >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mb, 0u));
        sum += ((uint32_t)__popcll(kb) << 16) + (uint32_t)__popcll(mb);
    }
    if constexpr (NW > 1) {
        const uint32_t w = threadIdx.x >> 6;
        if ((threadIdx.x & 63u) == 0) wsum[w] = sum;
        __syncthreads();
        sum = 0;
#pragma unroll
        for (uint32_t k = 0; k < NW; k++) {
            const uint32_t v = wsum[k];
            before += k < w ? v : 0u;
            sum += v;
        }
    }
    *total = sum;
    return before;
}

// One PLOC round (nn + mark + top + scatter of trace_ploc.wgsl:84-234 in one kernel): tiles of
// positions taken in order from a counter; each loads the boxes of its positions +- 2R
// into LDS, finds the nearest of positions +- R, marks who stays and who merges, takes its
// place in the next list from the tiles before it (look-back), writes the merged nodes and
// its part of the next list. Blocks loop over tiles, so any grid size covers the round. Large rounds
// are bound by their claims, gathers and searches together (1M clusters: 94 -> 45 us), small ones by
// the chain of one tile (launch, claim, list, boxes, search, look-back: 26 -> 8 us, of which the search
// was half); a grid short of the tiles made a round twice as long (49 us).
constexpr int ploc_tile(int P) { return (BLOCK / 64) * (64 * P - 2 * PLOC_R) - 2 * PLOC_R; }   // 864 of P = 4, 352 of P = 2
constexpr int PLOC_CLEAR = (ploc_tile(4) + ploc_tile(2) - 1) / ploc_tile(2);   // the next round's tiles a tile may stand for

template <int P>
__global__ __launch_bounds__(BLOCK, 4) void k_ploc_round(int round, int n, uint32_t small, uint32_t node0, uint32_t ref0,
                                                        float4 *bx, uint32_t *list0, uint32_t *list1, LrNode *nodes,
                                                        PlocState *st, uint64_t *status0, uint64_t *status1, uint32_t status_n)
{
    constexpr int TILE = ploc_tile(P), WIN = TILE + 4 * PLOC_R, NN = TILE + 2 * PLOC_R, RANGE = 64 * P - 2 * PLOC_R;
    constexpr int PER = (TILE + BLOCK - 1) / BLOCK, LOADS = (WIN + BLOCK - 1) / BLOCK;
    __shared__ __attribute__((aligned(16))) float l[6][WIN];
    __shared__ uint32_t wid[WIN], wh[WIN];
    __shared__ int8_t snn[NN];   // the nearest as an offset from the position (within +-R; 0: none)
    __shared__ uint32_t s_wsum[BLOCK / 64];
    __shared__ uint32_t s_tile, s_ek, s_em;
    const int tid = threadIdx.x;
    for (;;) {
        if (tid == 0) s_tile = atomicAdd(&st->ctr[round], 1u);
        // (beside the claim: the round's last tile changes them, once every tile of the round is claimed)
        const uint32_t nc = ld_dev(&st->nc), p = ld_dev(&st->parity);
        __syncthreads();
        const uint32_t tile = s_tile;
        const uint32_t ntiles = (nc + TILE - 1) / TILE;
        if (nc <= small || tile >= ntiles) return;
        const uint32_t *cur = p ? list1 : list0;
        uint32_t *nxt = p ? list0 : list1;
        uint64_t *status = p ? status1 : status0;
        uint64_t *status_next = p ? status0 : status1;
        // (the next round's, cleared for it: it may have smaller tiles)
        if (tid < PLOC_CLEAR && tile * PLOC_CLEAR + tid < status_n) status_next[tile * PLOC_CLEAR + tid] = 0;
        const int base = (int)tile * TILE;
        uint32_t x[LOADS];
#pragma unroll
        for (int q = 0; q < LOADS; q++) {
            const int o = tid + q * BLOCK, g = base - 2 * PLOC_R + o;
            x[q] = o < WIN && g >= 0 && g < (int)nc ? cur[g] : LR_NONE;
        }
#pragma unroll
        for (int q = 0; q < LOADS; q++) {
            const int o = tid + q * BLOCK;
            if (x[q] == LR_NONE) continue;
            const float4 lo = bx[2 * (size_t)x[q]], hi = bx[2 * (size_t)x[q] + 1];
            wid[o] = x[q];
            wh[o] = height_of(lo);
            l[0][o] = lo.x; l[1][o] = lo.y; l[2][o] = lo.z;
            l[3][o] = hi.x; l[4][o] = hi.y; l[5][o] = hi.z;
        }
        __syncthreads();
        {
            const int w = tid >> 6;
            nearest_range<P>(base - PLOC_R + w * RANGE, (int)nc, 2 * PLOC_R - base, l, snn + w * RANGE);
        }
        __syncthreads();
        // keep_merge (trace_ploc.wgsl:130-145)
        uint32_t j[PER];
        bool keep[PER], merge[PER];
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int o = PER * tid + q, i = base + o;
            const bool valid = o < TILE && i < (int)nc;
            const int dj = valid ? (int)snn[o + PLOC_R] : 0;
            j[q] = dj != 0 ? (uint32_t)(i + dj) : LR_NONE;
            bool mu = false;
            if (j[q] < nc) mu = (int)j[q] + (int)snn[(int)j[q] - base + PLOC_R] == i;
            keep[q] = valid && !(mu && (uint32_t)i > j[q]);
            merge[q] = valid && mu && (uint32_t)i < j[q];
        }
        uint32_t both;
        const uint32_t xkm = places<BLOCK / 64>(keep, merge, &both, s_wsum);
        const uint32_t xk = xkm >> 16, xm = xkm & 0xffffu, tk = both >> 16, tm = both & 0xffffu;
        if (tid < 64) {
            // the look-back by the first wave, 64 predecessor tiles at once (lane l: tile t - l):
            // the nearest inclusive prefix among them ends it; a needed tile not yet posted means
            // the same window again
            const uint64_t mine = ((uint64_t)tk << 31) | tm;
            uint64_t ek = 0, em = 0;
            if (tile == 0) {
                if (tid == 0) st_dev64(&status[0], (2ull << 62) | mine);
            } else {
                if (tid == 0) st_dev64(&status[tile], (1ull << 62) | mine);
                for (int t = (int)tile - 1;;) {
                    const int q = t - tid;
                    const uint64_t sv = q >= 0 ? ld_dev64(&status[q]) : (2ull << 62);
                    const uint64_t f = sv >> 62;
                    const uint64_t inc = __ballot(f == 2), zero = __ballot(f == 0);
                    const int stop = inc ? __ffsll((unsigned long long)inc) - 1 : 63;
                    const uint64_t need = stop == 63 ? ~0ull : ((2ull << stop) - 1ull);
                    if (zero & need) {
                        __builtin_amdgcn_s_sleep(1);
                        continue;
                    }
                    uint64_t ak = tid <= stop ? (sv >> 31) & 0x7fffffffull : 0ull;
                    uint64_t am = tid <= stop ? sv & 0x7fffffffull : 0ull;
#pragma unroll
                    for (int o = 32; o > 0; o >>= 1) {
                        ak += __shfl_xor(ak, o, 64);
                        am += __shfl_xor(am, o, 64);
                    }
                    ek += ak;
                    em += am;
                    if (inc) break;
                    t -= 64;
                }
                if (tid == 0) st_dev64(&status[tile], (2ull << 62) | ((ek + tk) << 31) | (em + tm));
            }
            if (tid == 0) {
                s_ek = (uint32_t)ek;
                s_em = (uint32_t)em;
                if (tile == ntiles - 1) {              // the round's last tile: the next count
                    st_dev(&st->nc, (uint32_t)ek + tk);
                    st_dev(&st->parity, 1u - p);
                    st_dev64(&st->live, ld_dev64(&st->live) + nc);   // (one writer a round)
                    st_dev(&st->made, ld_dev(&st->made) + 1u);
                }
            }
        }
        __syncthreads();
        uint32_t dk = s_ek + xk, dm = s_em + xm;
#pragma unroll
        for (int q = 0; q < PER; q++) {
            if (!keep[q]) continue;
            const int li = PER * tid + q + 2 * PLOC_R;
            const uint32_t c = wid[li];
            uint32_t out = c;
            if (merge[q]) {
                const int lj = (int)j[q] - base + 2 * PLOC_R;
                const uint32_t k = ((uint32_t)n - 2u) - ((uint32_t)n - nc + dm);
                dm++;
                ploc_merge(k, c, make_float4(l[0][li], l[1][li], l[2][li], __uint_as_float(wh[li])),
                           make_float4(l[3][li], l[4][li], l[5][li], 0.0f), wid[lj],
                           make_float4(l[0][lj], l[1][lj], l[2][lj], __uint_as_float(wh[lj])),
                           make_float4(l[3][lj], l[4][lj], l[5][lj], 0.0f), (uint32_t)n, node0, ref0, bx, nodes);
                out = k;
            }
            nxt[dk++] = out;
        }
        __syncthreads();
    }
}

// small (trace_ploc.wgsl:236-301): the rounds left, in one workgroup, from 1024 clusters (the
// context's ploc_small: below it a round's launch costs more than its work). While
// more than SMALL_MAX clusters are left (only when the rounds before could not merge enough:
// boxes that tie everywhere merge one pair a round) a round goes through device memory; from
// SMALL_MAX down, the list, its boxes (six arrays of floats) and heights live in LDS, and only the
// merged nodes' records go out. From 96 clusters down one wave goes on alone, without barriers:
// most of the rounds are there. Bound by one compute unit's VALU down to some 100 clusters (3 waves
// a SIMD search), then by the chain of a round (2 us): 5001 boxes' 292 -> 127 us.
constexpr int SMALL_BLOCK = 1024;
constexpr int SMALL_MAX = 4096;
constexpr int SMALL_PAD = 64 * 2 + PLOC_R;   // LDS places around the list that a wave's search may read
struct SmallLds {
    __attribute__((aligned(16))) float b[6][SMALL_MAX + SMALL_PAD];   // position i at i + R
    uint32_t id[SMALL_MAX], h[SMALL_MAX];
    int8_t nn[SMALL_MAX];
    uint32_t wsum[SMALL_BLOCK / 64];
};

// one round of the list of nc in LDS by the first WAVES waves, P positions a lane in the search, PER a
// thread after it; returns the clusters left
template <int P, int PER, int WAVES>
__device__ __forceinline__ uint32_t small_round(SmallLds &S, uint32_t nc, uint32_t n, uint32_t node0, uint32_t ref0, LrNode *nodes)
{
    constexpr int RANGE = 64 * P - 2 * PLOC_R;
    const int tid = threadIdx.x;
    auto sync = [] {
        if constexpr (WAVES == 1) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        } else {
            // (LDS only: the records on their way out are not waited for)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        }
    };
    for (int i0 = (tid >> 6) * RANGE; i0 < (int)nc; i0 += WAVES * RANGE)
        nearest_range<P>(i0, (int)nc, PLOC_R, S.b, S.nn + i0);
    sync();
    // each thread takes a run of positions, holds what it writes in registers, and writes after
    // every read of the round is done
    uint32_t j[PER];
    bool keep[PER], merge[PER];
#pragma unroll
    for (int q = 0; q < PER; q++) {
        const int i = PER * tid + q;
        keep[q] = merge[q] = false;
        if (i >= (int)nc) continue;
        const int dj = S.nn[i];
        const bool mu = dj != 0 && S.nn[i + dj] == -dj;
        j[q] = (uint32_t)(i + dj);
        keep[q] = !(mu && dj < 0);
        merge[q] = mu && dj > 0;
    }
    uint32_t both;
    const uint32_t x = places<WAVES>(keep, merge, &both, S.wsum);
    uint32_t dk = x >> 16, dm = x & 0xffffu;
    uint32_t o_id[PER], o_h[PER];
    float o_b[PER][6];
#pragma unroll
    for (int q = 0; q < PER; q++) {
        const int i = PER * tid + q;
        if (!keep[q]) continue;
#pragma unroll
        for (int c = 0; c < 6; c++) o_b[q][c] = S.b[c][PLOC_R + i];
        o_id[q] = S.id[i];
        o_h[q] = S.h[i];
        if (!merge[q]) continue;
        const uint32_t k = (n - 2u) - (n - nc + dm);
        dm++;
        float d[6];
#pragma unroll
        for (int c = 0; c < 6; c++) d[c] = S.b[c][PLOC_R + j[q]];
        put_final(&nodes[1 + 2 * (size_t)k], o_id[q], make_float4(o_b[q][0], o_b[q][1], o_b[q][2], 0.0f),
                  make_float4(o_b[q][3], o_b[q][4], o_b[q][5], 0.0f), n, node0, ref0);
        put_final(&nodes[2 + 2 * (size_t)k], S.id[j[q]], make_float4(d[0], d[1], d[2], 0.0f), make_float4(d[3], d[4], d[5], 0.0f),
                  n, node0, ref0);
#pragma unroll
        for (int c = 0; c < 6; c++) o_b[q][c] = c < 3 ? wmin(o_b[q][c], d[c]) : wmax(o_b[q][c], d[c]);
        if (k == 0)
            put_node(&nodes[0], o_b[q][0], o_b[q][1], o_b[q][2], node0 + 1u, o_b[q][3], o_b[q][4], o_b[q][5], node0 + 2u);
        o_id[q] = k;
        o_h[q] = 1u + max(o_h[q], S.h[j[q]]);
    }
    sync();
#pragma unroll
    for (int q = 0; q < PER; q++) {
        if (!keep[q]) continue;
        S.id[dk] = o_id[q];
        S.h[dk] = o_h[q];
#pragma unroll
        for (int c = 0; c < 6; c++) S.b[c][PLOC_R + dk] = o_b[q][c];
        dk++;
    }
    sync();
    return both >> 16;
}

__global__ __launch_bounds__(SMALL_BLOCK) void k_ploc_small(int n, uint32_t node0, uint32_t ref0, float4 *bx, uint32_t *list0,
                                                              uint32_t *list1, uint32_t *nnbuf, LrNode *nodes,
                                                              PlocState *st, int planned, LrBuildResult *res)
{
    __shared__ SmallLds S;
    uint32_t *const s_wsum = S.wsum;
    const int tid = threadIdx.x;
    uint32_t nc = st->nc, p = st->parity;
    uint32_t rounds = 0;
    uint64_t live = 0;
    // rounds through device memory while the list does not fit in LDS
    while (nc > (uint32_t)SMALL_MAX) {
        live += nc;
        const uint32_t *cur = p ? list1 : list0;
        uint32_t *nxt = p ? list0 : list1;
        for (int i = tid; i < (int)nc; i += SMALL_BLOCK) {
            const uint32_t xi = cur[i];
            const float4 lo = bx[2 * (size_t)xi], hi = bx[2 * (size_t)xi + 1];
            const int j0 = i - PLOC_R > 0 ? i - PLOC_R : 0;
            const int j1 = i + PLOC_R < (int)nc - 1 ? i + PLOC_R : (int)nc - 1;
            float bd = 0.0f;
            uint32_t bj = LR_NONE;
            for (int j = j0; j <= j1; j++) {
                if (j == i) continue;
                const uint32_t xj = cur[j];
                const float4 ol = bx[2 * (size_t)xj], oh = bx[2 * (size_t)xj + 1];
                const float d = half_area(wmin(lo.x, ol.x), wmin(lo.y, ol.y), wmin(lo.z, ol.z),
                                          wmax(hi.x, oh.x), wmax(hi.y, oh.y), wmax(hi.z, oh.z));
                if (nearer(d, (uint32_t)i, (uint32_t)j, bd, bj)) { bd = d; bj = (uint32_t)j; }
            }
            nnbuf[i] = bj;
        }
        __syncthreads();
        const int per = ((int)nc + SMALL_BLOCK - 1) / SMALL_BLOCK;
        const int s0 = min(tid * per, (int)nc), s1 = min(s0 + per, (int)nc);
        uint32_t ck = 0, cm = 0;
        for (int i = s0; i < s1; i++) {
            const uint32_t j = nnbuf[i];
            const bool mu = j < nc && nnbuf[j] == (uint32_t)i;
            ck += !(mu && (uint32_t)i > j);
            cm += mu && (uint32_t)i < j;
        }
        uint32_t tk, tm;
        uint32_t dk = block_excl_scan<SMALL_BLOCK / 64>(ck, &tk, s_wsum);
        uint32_t dm = block_excl_scan<SMALL_BLOCK / 64>(cm, &tm, s_wsum);
        for (int i = s0; i < s1; i++) {
            const uint32_t j = nnbuf[i];
            const bool mu = j < nc && nnbuf[j] == (uint32_t)i;
            if (mu && (uint32_t)i > j) continue;
            const uint32_t c = cur[i];
            uint32_t out = c;
            if (mu && (uint32_t)i < j) {
                const uint32_t d = cur[j];
                const uint32_t k = ((uint32_t)n - 2u) - ((uint32_t)n - nc + dm);
                dm++;
                ploc_merge(k, c, bx[2 * (size_t)c], bx[2 * (size_t)c + 1], d, bx[2 * (size_t)d], bx[2 * (size_t)d + 1],
                           (uint32_t)n, node0, ref0, bx, nodes);
                out = k;
            }
            nxt[dk++] = out;
        }
        __syncthreads();
        // every round merges at least the pair nearest of all (it is mutual); a round that
        // merges nothing (NaN boxes) ends the loop instead of spinning
        if (tk >= nc) {
            nc = 0;
            break;
        }
        nc = tk;
        p = 1u - p;
        rounds++;
    }
    // the rest in LDS
    if (nc > 0) {
        const uint32_t *cur = p ? list1 : list0;
        for (int i = tid; i < (int)nc; i += SMALL_BLOCK) {
            const uint32_t x = cur[i];
            const float4 lo = bx[2 * (size_t)x], hi = bx[2 * (size_t)x + 1];
            S.id[i] = x;
            S.h[i] = height_of(lo);
            S.b[0][PLOC_R + i] = lo.x; S.b[1][PLOC_R + i] = lo.y; S.b[2][PLOC_R + i] = lo.z;
            S.b[3][PLOC_R + i] = hi.x; S.b[4][PLOC_R + i] = hi.y; S.b[5][PLOC_R + i] = hi.z;
        }
        __syncthreads();
    }
    constexpr int WAVES = SMALL_BLOCK / 64;
    while (nc > 1) {
        if (nc <= 96 && tid >= 64) return;   // one wave goes on
        const uint32_t left = nc > SMALL_BLOCK ? small_round<2, SMALL_MAX / SMALL_BLOCK, WAVES>(S, nc, (uint32_t)n, node0, ref0, nodes)
                              : nc > 96        ? small_round<2, 1, WAVES>(S, nc, (uint32_t)n, node0, ref0, nodes)
                              : nc > 32        ? small_round<2, 2, 1>(S, nc, (uint32_t)n, node0, ref0, nodes)
                                               : small_round<1, 1, 1>(S, nc, (uint32_t)n, node0, ref0, nodes);
        live += nc;
        if (left >= nc) break;   // merged nothing (NaN boxes): ends instead of spinning
        nc = left;
        rounds++;
    }
    if (tid == 0) {
        if (res) {
            __hip_atomic_store(&res->rounds, rounds + max((uint32_t)planned, st->made), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(&res->live, st->live + live, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        tell_depth(res, nc == 1 ? S.h[0] : height_of(bx[0]));
    }
}

// ---- the scratch layout of one build --------------------------------------------------------------
struct Layout {
    size_t params, bounds_tmp, hist, ticket, bucket, keys0, vals0, keys1, vals1, zero, zero_words, status,
        ctr, other, esc_count, bx, list0, list1, nnbuf, pst, pstatus, pstatus_words, total;
};

Layout layout(int n)
{
    Layout L;
    const size_t N = n > 0 ? (size_t)n : 1;
    const size_t tiles = (N + SORT_TILE - 1) / SORT_TILE;
    const size_t ptiles = (N + ploc_tile(2) - 1) / ploc_tile(2);
    size_t o = 0;
    auto take = [&](size_t bytes) { size_t at = o; o += lr_align(bytes); return at; };
    L.params = take(sizeof(LrBuildParamsDev));
    L.bounds_tmp = take(BOUNDS_BLOCKS * 6 * 4 + 64);
    L.hist = take(HIST_COPIES * SORT_PASSES * 256 * 4);
    L.ticket = take(64);
    L.bucket = take(SORT_PASSES * 256 * 4);
    L.keys0 = take(N * 4);
    L.vals0 = take(N * 4);
    L.keys1 = take(N * 4);
    L.vals1 = take(N * 4);
    // one region the Morton kernel clears: tile counters, look-back states, arrivals
    L.zero = o;
    L.ctr = take(64);
    L.status = take(SORT_PASSES * tiles * 256 * 4);
    L.other = take(N * 8);
    L.zero_words = (o - L.zero) / 4;
    // PLOC's; an LBVH build's listed nodes (k_lbvh's slots, 16 bytes each) and their counts
    const size_t groups = (N + LBVH_GROUP - 1) / LBVH_GROUP;
    L.esc_count = take(groups * 4);
    L.bx = take(std::max((2 * N) * 32, groups * LBVH_SLOTS * 16));
    L.list0 = take(N * 4);
    L.list1 = take(N * 4);
    L.nnbuf = take(N * 4);
    L.pst = take(sizeof(PlocState));
    L.pstatus_words = 2 * (ptiles + 1);
    L.pstatus = take(L.pstatus_words * 8);
    L.total = o;
    return L;
}

// ploc_rounds (trace_gpu.c:563): the rounds from n down to `small`, two more to be safe: those a
// build counts even where fewer are made
int ploc_rounds(int n, int small)
{
    int r = 0;
    for (int64_t m = n; m > small; m = m * 5 / 6) r++;
    return std::min(r ? r + 2 : 0, PLOC_MAX_ROUNDS);
}

// the rounds launched: a round leaves 0.84 to 0.87 of its clusters, and one left to k_ploc_small above its
// best size costs it 30 us, where a launch with nothing left to do takes 2 and a round 8
int ploc_launches(int n, int small)
{
    int r = 0;
    for (double m = n; m > small; m *= 0.87) r++;
    return std::min(r ? r + 1 : 0, PLOC_MAX_ROUNDS);
}

}  // namespace

size_t lr_bounds_tmp_bytes() { return BOUNDS_BLOCKS * 6 * 4 + 64; }

int lr_launch_tri_boxes(LrhContext *c, const float *tris, int n, float *boxes)
{
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_tri_boxes, dim3((n + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, c->stream,
                       reinterpret_cast<const float4 *>(tris), n, reinterpret_cast<float4 *>(boxes));
    LR_HIP(hipGetLastError());
    return 0;
}

// tmp: BOUNDS_BLOCKS * 6 floats then a zeroed ticket word (at +BOUNDS_BLOCKS*24)
int lr_launch_bounds(LrhContext *c, const float *boxes, int n, LrBuildParamsDev *out, void *tmp)
{
    int blocks = (n + BLOCK - 1) / BLOCK;
    if (blocks > BOUNDS_BLOCKS) blocks = BOUNDS_BLOCKS;
    if (blocks < 1) blocks = 1;
    float *partial = (float *)tmp;
    uint32_t *ticket = (uint32_t *)((char *)tmp + BOUNDS_BLOCKS * 24);
    hipLaunchKernelGGL(k_bounds, dim3(blocks), dim3(BLOCK), 0, c->stream, reinterpret_cast<const float4 *>(boxes), n,
                       partial, ticket, out);
    LR_HIP(hipGetLastError());
    return 0;
}

size_t lr_build_scratch_bytes(int n) { return layout(n).total; }

namespace {

// one build with its scratch at S (layout(n).total bytes, the counters before keys0 at zero)
int build_at(LrhContext *c, char *S, const float *boxes, int n, const float *host_bounds, int builder, uint32_t node0,
             uint32_t ref0, uint32_t ref_add, uint32_t *nodes, uint32_t *aux, uint32_t *sorted_codes_out,
             uint32_t *sorted_items_out, LrhBuildStats *stats)
{
    const Layout L = layout(n);
    int rc = 0;
    auto at = [&](size_t off) { return (void *)(S + off); };
    LrBuildParamsDev *prm = (LrBuildParamsDev *)at(L.params);
    uint32_t *k0 = (uint32_t *)at(L.keys0), *v0 = (uint32_t *)at(L.vals0);
    uint32_t *k1 = (uint32_t *)at(L.keys1), *v1 = (uint32_t *)at(L.vals1);
    LrNode *nd = reinterpret_cast<LrNode *>(nodes) + node0;
    uint32_t *ax = aux + ref0;
    hipStream_t s = c->stream;
    if (stats) LR_HIP(hipEventRecord(c->ev[0], s));
    if (host_bounds)
        hipLaunchKernelGGL(k_params, dim3(1), dim3(1), 0, s, prm, host_bounds[0], host_bounds[1], host_bounds[2],
                           host_bounds[3], host_bounds[4], host_bounds[5]);
    else if ((rc = lr_launch_bounds(c, boxes, n, prm, at(L.bounds_tmp)))) return rc;
    const int tiles = (n + SORT_TILE - 1) / SORT_TILE;
    hipLaunchKernelGGL(k_morton, dim3(tiles), dim3(SORT_BLOCK), 0, s, reinterpret_cast<const float4 *>(boxes), n, prm, k0, v0,
                       (uint32_t *)at(L.hist), (uint32_t *)at(L.ticket), (uint32_t *)at(L.bucket), (uint32_t *)at(L.zero),
                       L.zero_words);
    LR_HIP(hipGetLastError());
    uint32_t *ctr = (uint32_t *)at(L.ctr);
    for (int pass = 0; pass < SORT_PASSES; pass++) {
        const uint32_t *ki = pass & 1 ? k1 : k0, *vi = pass & 1 ? v1 : v0;
        uint32_t *ko = pass & 1 ? k0 : k1, *vo = pass & 1 ? v0 : v1;
        hipLaunchKernelGGL(k_sort_pass, dim3(tiles), dim3(SORT_BLOCK), 0, s, ki, vi, ko, vo, n, 8 * pass,
                           (const uint32_t *)at(L.bucket) + 256 * pass,
                           (uint32_t *)at(L.status) + (size_t)pass * tiles * 256, ctr + pass);
        LR_HIP(hipGetLastError());
    }
    // sorted: k0 (codes), v0 (items)
    if (sorted_codes_out) LR_HIP(hipMemcpyAsync(sorted_codes_out, k0, (size_t)n * 4, hipMemcpyDeviceToDevice, s));
    if (sorted_items_out) LR_HIP(hipMemcpyAsync(sorted_items_out, v0, (size_t)n * 4, hipMemcpyDeviceToDevice, s));
    LrBuildResult *res = stats ? c->built : nullptr;
    if (res) *res = LrBuildResult{};
    const bool ploc = builder == LRH_PLOC && n > 2;
    if (!ploc) {
        const int groups = (n + LBVH_GROUP - 1) / LBVH_GROUP;
        uint4 *esc = (uint4 *)at(L.bx);
        uint32_t *esc_count = (uint32_t *)at(L.esc_count);
        hipLaunchKernelGGL(k_lbvh, dim3(groups), dim3(LBVH_GROUP), 0, s, k0, v0, reinterpret_cast<const float4 *>(boxes), n, node0,
                           ref0, ref_add, nd, ax, esc, esc_count, res);
        LR_HIP(hipGetLastError());
        // the climbs above the groups; the buffer path while the records lie within 2 GiB of
        // the array's base
        const dim3 tgrid((unsigned)((groups + BLOCK / 64 - 1) / (BLOCK / 64)));
        if ((2 * (size_t)n - 1) * 32 < 0x7fffffffu)
            hipLaunchKernelGGL(k_lbvh_top<true>, tgrid, dim3(BLOCK), 0, s, k0, v0, reinterpret_cast<const float4 *>(boxes), n,
                               groups, node0, nd, (unsigned long long *)at(L.other), esc, esc_count, res);
        else
            hipLaunchKernelGGL(k_lbvh_top<false>, tgrid, dim3(BLOCK), 0, s, k0, v0, reinterpret_cast<const float4 *>(boxes), n,
                               groups, node0, nd, (unsigned long long *)at(L.other), esc, esc_count, res);
        LR_HIP(hipGetLastError());
    } else {
        float4 *bx = (float4 *)at(L.bx);
        uint32_t *l0 = (uint32_t *)at(L.list0), *l1 = (uint32_t *)at(L.list1);
        PlocState *pst = (PlocState *)at(L.pst);
        uint64_t *ps = (uint64_t *)at(L.pstatus);
        const size_t ptiles = L.pstatus_words / 2;
        hipLaunchKernelGGL(k_ploc_init, dim3((n + BLOCK - 1) / BLOCK), dim3(BLOCK), 0, s, v0,
                           reinterpret_cast<const float4 *>(boxes), n, ref0, ref_add, ax, bx, l0, pst, ps,
                           L.pstatus_words);
        LR_HIP(hipGetLastError());
        const int small = std::min(c->ploc_small > 0 ? c->ploc_small : 1024, SMALL_MAX);
        const int planned = ploc_rounds(n, small), nr = std::max(planned, ploc_launches(n, small));
        // the grid from an estimate of the clusters left (a round leaves 0.84 to 0.87 of them; work-groups
        // without a tile end at once, one with two makes the round twice as long)
        double est = n;
        for (int r = 0; r < nr; r++) {
            const bool big = est >= PLOC_BIG;
            const int tile = big ? ploc_tile(4) : ploc_tile(2);
            const int grid = std::clamp((int)((est + tile - 1) / tile), 16, 4096);
            hipLaunchKernelGGL((big ? k_ploc_round<4> : k_ploc_round<2>), dim3(grid), dim3(BLOCK), 0, s, r, n, (uint32_t)small,
                               node0, ref0, bx, l0, l1, nd, pst, ps, ps + ptiles, (uint32_t)ptiles);
            LR_HIP(hipGetLastError());
            est *= 0.88;
        }
        hipLaunchKernelGGL(k_ploc_small, dim3(1), dim3(SMALL_BLOCK), 0, s, n, node0, ref0, bx, l0, l1,
                           (uint32_t *)at(L.nnbuf), nd, pst, planned, res);
        LR_HIP(hipGetLastError());
    }
    if (stats) {
        LR_HIP(hipEventRecord(c->ev[1], s));
        LR_HIP(hipEventSynchronize(c->ev[1]));
        float ms = 0;
        LR_HIP(hipEventElapsedTime(&ms, c->ev[0], c->ev[1]));
        stats->clusters = res->live;
        stats->refitted = 0;
        stats->depth = (int)res->depth;
        stats->rounds = (int)res->rounds;
        stats->ms = ms;
        c->last_build_ms = ms;
    }
    return 0;
}

}  // namespace

int lr_build_run(LrhContext *c, const float *boxes, int n, const float *host_bounds, int builder, uint32_t node0,
                 uint32_t ref0, uint32_t ref_add, uint32_t *nodes, uint32_t *aux, uint32_t *sorted_codes_out,
                 uint32_t *sorted_items_out, LrhBuildStats *stats)
{
    int rc = lr_scratch_reserve(c, LR_SCRATCH_BUILD, layout(n).total);
    if (rc) return rc;
    return build_at(c, (char *)c->scratch[LR_SCRATCH_BUILD].base, boxes, n, host_bounds, builder, node0, ref0, ref_add,
                    nodes, aux, sorted_codes_out, sorted_items_out, stats);
}

// ---- the build without allocation (lrh_build_noalloc) --------------------------------------------
// Its scratch is this file-scope array: each device holds its own copy from the library's load
// until the process ends. In host code `scratch` names a host-side stand-in, not the device
// copy: the device address is taken once per device (lr_noalloc_init, from lrh_create, with
// that device current) and only that address is handed to kernels.
constexpr int NOALLOC_MAX_DEVICES = 64;
constexpr size_t NOALLOC_BYTES = (size_t)8 << 20;
static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];
static char *g_noalloc_ptr[NOALLOC_MAX_DEVICES];
static std::mutex g_noalloc_mu;

namespace {

// clears n words (the counters that must start at zero: a kernel, so a caller may capture it)
__global__ __launch_bounds__(256) void k_clear_words(uint32_t *p, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = 0u;
}

}  // namespace

int lr_noalloc_init(int device)
{
    if (device < 0 || device >= NOALLOC_MAX_DEVICES)
        return lr_fail(LRH_EINVAL, "device %d: the no-allocation build keeps %d devices", device, NOALLOC_MAX_DEVICES);
    if (layout(LRH_NOALLOC_MAX_ITEMS).total > NOALLOC_BYTES)
        return lr_fail(LRH_EDEVICE, "the no-allocation build's scratch (%zu bytes) is below its %d items' %zu",
                       NOALLOC_BYTES, LRH_NOALLOC_MAX_ITEMS, layout(LRH_NOALLOC_MAX_ITEMS).total);
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    if (g_noalloc_ptr[device]) return 0;
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
        (void)hipGetLastError();
        return lr_fail(LRH_EDEVICE, "hipGetSymbolAddress(scratch) on device %d: %s", device, hipGetErrorString(e));
    }
    g_noalloc_ptr[device] = (char *)ptr;
    return 0;
}

int lr_build_noalloc(LrhContext *c, const float *boxes, int n, const float *host_bounds, int builder, uint32_t node0,
                     uint32_t ref0, uint32_t ref_add, uint32_t *nodes, uint32_t *aux, uint32_t *sorted,
                     LrhBuildStats *stats)
{
    char *S = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_noalloc_mu);
        if (c->device >= 0 && c->device < NOALLOC_MAX_DEVICES) S = g_noalloc_ptr[c->device];
    }
    if (!S) return lr_fail(LRH_EDEVICE, "lrh_build_noalloc: device %d has no scratch address", c->device);
    const Layout L = layout(n);
    if (L.total > NOALLOC_BYTES)
        return lr_fail(LRH_EREFUSED, "lrh_build_noalloc: %d items need %zu bytes of scratch, above its %zu", n, L.total,
                       NOALLOC_BYTES);
    // the counters before the keys start at zero (a call that ends normally leaves them so; this
    // clear makes the call independent of any earlier one)
    hipLaunchKernelGGL(k_clear_words, dim3(16), dim3(256), 0, c->stream, (uint32_t *)S, L.keys0 / 4);
    LR_HIP(hipGetLastError());
    return build_at(c, S, boxes, n, host_bounds, builder, node0, ref0, ref_add, nodes, aux, sorted,
                    sorted ? sorted + n : nullptr, stats);
}
