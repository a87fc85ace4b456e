// lr_engine.hip - the engine's host side (include/lr_hip.h: lrh_engine_*, lrh_pt_render): the
// device state, job admission and its image arena, the captured graph of iterations and the
// progress it reports, the plain per-job form, and the autotuner.
//
// Progress: after each graph the engine's counters and every job slot's retired-path count
// are copied to pinned host memory (two buffers, so the device never waits for the host); a
// job is done when all its paths have retired, at the device clock its last retire recorded.
#include <math.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <deque>
#include <map>
#include <vector>

#include "lr_device.h"
#include "lr_engine.h"

extern "C" void lrs_blue_noise(uint16_t *rank);
extern "C" void lrs_brdf_tables(float *out);

namespace {

constexpr int SBLOCK = 256;

// Bounce rays are ordered by direction (order_rays, lr_engine_k.h) while a job of a one-level scene of this
// many shapes runs, and none of a two-level scene. 1280 x 720 x 8 samples of 16,000 triangles 6.28 -> 5.90
// ms, of 4000 4.71 -> 4.52, of 1000 3.91 -> 3.85, of 500 3.76 -> 3.74, of 250 3.65 both, the Cornell
// room's 35 shapes 4.68 -> 4.77 (every ray visits much of so small a tree); medians, runs differ by 0.3
// %. Not with two-level scenes, whose rays part inside the instances (19.3 -> 19.9 ms for two frames of
// 5001 instances).
constexpr int LR_ORDER_SHAPES = 1000;

__global__ __launch_bounds__(SBLOCK) void k_eng_init(EngProgress *prog, uint32_t C)
{
    const size_t nw = sizeof(EngProgress) / 8;
    unsigned long long *w = (unsigned long long *)prog;
    for (size_t i = (size_t)blockIdx.x * SBLOCK + threadIdx.x; i < nw; i += (size_t)gridDim.x * SBLOCK)
        w[i] = (i == offsetof(EngCtl, tail) / 8) ? (unsigned long long)C : 0ull;
}

__global__ void k_job_put(JobDev *jobs, unsigned long long *jret, unsigned long long *jdone,
                          long long (*jpass)[LR_PILOT_PASSES], int slot, JobDev jd)
{
    jobs[slot] = jd;
    jret[slot] = 0;
    jdone[slot] = 0;
    for (int k = 0; k < LR_PILOT_PASSES; k++) jpass[slot][k] = 0;
}

// a pilot job's chosen size: its paths in all, and no more pilot sums
__global__ void k_job_total(JobDev *jobs, int slot, unsigned long long total)
{
    jobs[slot].total = total;
    jobs[slot].pilot = 0;
}

__global__ __launch_bounds__(SBLOCK) void k_zero64(long long *p, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * SBLOCK + threadIdx.x; i < n; i += (size_t)gridDim.x * SBLOCK) p[i] = 0;
}

// an issue record: global path indices [start, issue_end) are the job's q0, q0 + 1, ...
__global__ void k_issue(EngCtl *ctl, unsigned long long *iq_start, uint32_t *iq_job, uint32_t *iq_q0,
                        unsigned long long rec, unsigned long long start, uint32_t jslot, uint32_t q0,
                        unsigned long long issue_end, unsigned long long lo, uint32_t order)
{
    iq_start[rec & (LR_ISSUE - 1)] = start;
    iq_job[rec & (LR_ISSUE - 1)] = jslot;
    iq_q0[rec & (LR_ISSUE - 1)] = q0;
    ctl->iq_hi = rec + 1;
    ctl->issue_end = issue_end;
    ctl->iq_lo = lo;
    ctl->order = order;
}

// wf_resolve's output (trace_wave.wgsl:357-378): float4 (sum, count) per pixel
// a denoised job's moments to floats: the sum of its samples' irradiance luminance and of its square
__global__ __launch_bounds__(SBLOCK) void k_moments(const long long *mo, int npix, float2 *out)
{
    const int p = blockIdx.x * SBLOCK + threadIdx.x;
    if (p >= npix) return;
    out[p] = make_float2((float)((double)mo[2 * (size_t)p] / (double)(1u << LR_FIX_SHIFT)),
                         (float)((double)mo[2 * (size_t)p + 1] / (double)(1u << LR_MOM2_SHIFT)));
}

__global__ __launch_bounds__(SBLOCK) void k_resolve(const long long *acc, int npix, float count, float4 *out, int add)
{
    const int p = blockIdx.x * SBLOCK + threadIdx.x;
    if (p >= npix) return;
    const double u = 1.0 / (double)(1u << LR_FIX_SHIFT);
    const float4 v = make_float4((float)((double)acc[3 * (size_t)p] * u), (float)((double)acc[3 * (size_t)p + 1] * u),
                                 (float)((double)acc[3 * (size_t)p + 2] * u), count);
    if (add) {
        float4 o = out[p];
        o.x += v.x;
        o.y += v.y;
        o.z += v.z;
        o.w += v.w;
        out[p] = o;
    } else out[p] = v;
}

__global__ void k_clock(unsigned long long *out) { *out = (unsigned long long)wall_clock64(); }

double now_ms()
{
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

const LrEngTable &table()
{
    static LrEngTable t = [] {
        LrEngTable x;
        memset(&x, 0, sizeof(x));
        lr_eng_fill_b64(x);
        lr_eng_fill_b128(x);
        lr_eng_fill_b256(x);
        return x;
    }();
    return t;
}

struct HostJob {
    int state = 0;              // 0 free, LRH_JOB_RUNNING, LRH_JOB_DONE
    int64_t id = -1;
    LrhJob desc{};
    size_t off = 0, bytes = 0;  // its block in the arena: a denoised job's guide and moments, then its image
    size_t acc_off = 0, mom_off = 0, guide_off = 0;
    unsigned long long total = 0, issued = 0;   // its paths, and those issued so far
    int spp_done = 0;           // the samples per pixel it takes (a target error's: decided after its pilot)
    bool pilot = false;         // a target error's first 4 passes running (total: theirs)
    float rel_error = 0.0f;     // the estimated relative standard error at spp_done
    double t_submit = 0, t_done = 0;
    unsigned long long min_seq = 0;   // the first progress snapshot taken after its admission
    bool ordered = false, two_level = false;   // its scene's: bounce rays worth ordering; of two levels
    bool odd_eps = false;                      // ... and an eps that is not from +0 up (keys_ok)
};

struct IssueRec {
    unsigned long long rec, start, end;
};

struct ArenaChunk {
    size_t base, bytes;
    char *ptr;
};

}  // namespace

struct LrhEngine {
    LrhContext *ctx = nullptr;
    int device = 0;
    hipStream_t stream = nullptr;
    uint32_t C = 0;
    int ncu = 0, max_tree_depth = 0;
    size_t threads_cap = 0;
    int spill_cap = 0;                         // spill entries per thread (for a 16-entry LDS stack)
    // device memory
    void *dmem = nullptr;
    // job images: blocks of an offset space laid over device chunks (one chunk made at creation,
    // or, in a lazy arena, chunks made as images need them while the total stays within the cap);
    // consecutive chunks' offsets are kept 256 apart, so freed blocks never merge across chunks
    std::vector<ArenaChunk> chunks;
    size_t arena_bytes = 0, arena_cap = 0, arena_next = 0;
    bool arena_lazy = false;
    EngProgress *prog = nullptr;
    JobDev *jobs = nullptr;
    unsigned long long *iq_start = nullptr, *counts = nullptr, *clk = nullptr;
    uint32_t *iq_job = nullptr, *iq_q0 = nullptr;
    EngArgs base{};
    // host
    EngProgress *pin[2] = {nullptr, nullptr};
    hipEvent_t pev[2] = {nullptr, nullptr};
    bool pend[2] = {false, false};
    unsigned long long seq[2] = {0, 0}, seq_next = 0;
    int pk = 0;
    EngProgress last{};
    unsigned long long last_seq = 0;    // (last is the snapshot of this number, if any was taken)
    HostJob hj[LR_JOBS];
    std::map<size_t, size_t> free_blocks;      // arena: offset -> bytes
    std::map<int64_t, int> by_id;
    std::deque<IssueRec> recs;
    int64_t next_id = 1;
    unsigned long long issue_end = 0, iq_hi = 0;
    int running = 0;
    uint64_t jobs_done = 0;
    LrhTune tune{256, 16, 256, 8, 1, 8, 0, 0};   // the best measured on the batched workload (MI355X)
    bool counting = false;
    // profiling: iterations launched one kernel at a time between events (no graph); 2: the walks in one launch
    int profiling = 0;
    std::vector<hipEvent_t> pevs;
    double kms[4] = {0, 0, 0, 0};
    uint64_t klaunch[4] = {0, 0, 0, 0};
    // light tracing: the queue of light paths that go on past their first vertex (made on the
    // first job with light tracing: LR_LIGHT_CHUNK entries of 64 bytes, and its count), its
    // launches and paths, and with profiling on its device time
    float4 *lq = nullptr;
    uint32_t *lqn = nullptr;
    hipEvent_t lev[2] = {nullptr, nullptr};
    uint64_t light_paths = 0, light_launches = 0;
    double light_ms = 0;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    bool graph_ok = false;
    bool two_level = false;     // a two-level scene has been submitted: the walks that take both
    bool apart = false;         // a job of a scene whose eps (its rays' tmin) the one launch's walks do not
                                // take runs (keys_ok): the walks' own kernels
    bool multi = false;         // a scene with more than one light has been submitted: shade and
                                // shadow that take up to three shadow rays a vertex
    double clk_khz = 100000.0, clk_host0 = 0.0;
    unsigned long long clk_dev0 = 0;
};

namespace {

int eng_fail_dev(const char *what, hipError_t e)
{
    return lr_fail(LRH_EDEVICE, "engine: %s: %s", what, hipGetErrorString(e));
}
#define ENG_HIP(call)                                          \
    do {                                                       \
        hipError_t e_ = (call);                                \
        if (e_ != hipSuccess) return eng_fail_dev(#call, e_);  \
    } while (0)

bool tune_valid(const LrhTune &t)
{
    return lr_blk_index(t.block_trace) >= 0 && lr_blk_index(t.block_shade) >= 0 && lr_stk_index(t.stack) >= 0 &&
           t.blocks_per_cu >= 1 && t.blocks_per_cu <= 16 && (t.tile == 1 || t.tile == 2 || t.tile == 4 || t.tile == 8) &&
           t.iters_per_graph >= 1 && t.iters_per_graph <= 64 && t.refill >= 0 && t.refill <= 64 && t.refill_shadow >= 0 &&
           t.refill_shadow <= 64;
}

// the kernels' arguments for a launch whose walk kernels run `threads` threads
EngArgs args_for(const LrhEngine *e, int stack, size_t threads, int mult, int refill = 0, int refill_shadow = 0)
{
    EngArgs A = e->base;
    A.spill_per = e->max_tree_depth + 2 - stack > 0 ? e->max_tree_depth + 2 - stack : 0;
    A.spill_stride = threads;
    A.mult = mult;
    A.refill = refill;
    A.refill_shadow = refill_shadow;
    return A;
}

bool refilled(const LrhEngine *e, int refill) { return !e->two_level && refill > 0; }
// the walks go in one launch (not where they are counted or a walk's lanes refilled, nor with an eps that
// their keys do not take)
bool walks_joint(const LrhEngine *e, const LrhTune &t)
{
    return !e->counting && !e->apart && !refilled(e, t.refill) && !(refilled(e, t.refill_shadow) && !e->multi);
}

// One iteration in the persistent grids of the batched form: regen, the walks, shade. ev (profiling):
// 5 events around regen, the extension walk, the shadow walk and shade, each a launch of its own (profiling
// 2: the walks' one launch in the extension walk's place, and none between the next two)
void launch_iteration(LrhEngine *e, const LrhTune &t, hipEvent_t *ev = nullptr)
{
    const LrEngTable &T = table();
    const int bt = lr_blk_index(t.block_trace), bs = lr_blk_index(t.block_shade), sk = lr_stk_index(t.stack);
    const dim3 gt(e->ncu * t.blocks_per_cu), gs(e->ncu * t.blocks_per_cu);
    const EngArgs At = args_for(e, t.stack, (size_t)gt.x * t.block_trace, t.tile, t.refill, t.refill_shadow);
    const EngArgs As = args_for(e, t.stack, 0, t.tile);
    const int tl = e->two_level ? 1 : 0, ml = e->multi ? 1 : 0, cnt = e->counting ? 1 : 0;
    const bool rf = refilled(e, t.refill), srf = !ml && refilled(e, t.refill_shadow);
    if (ev) (void)hipEventRecord(ev[0], e->stream);
    T.regen[bs](gs, e->stream, As);
    if (ev) (void)hipEventRecord(ev[1], e->stream);
    if ((!ev || e->profiling == 2) && walks_joint(e, t)) {
        T.walks[bt][sk][tl][ml](gt, e->stream, At);
        if (ev) (void)hipEventRecord(ev[2], e->stream);
    } else {
        if (rf) T.extend_rf[bt][sk][cnt](gt, e->stream, At);
        else (cnt ? T.extend_count : T.extend)[bt][sk][tl](gt, e->stream, At);
        if (ev) (void)hipEventRecord(ev[2], e->stream);
        if (srf) T.shadow_rf[bt][sk][cnt](gt, e->stream, At);
        else (cnt ? T.shadow_count : T.shadow)[bt][sk][tl][ml](gt, e->stream, At);
    }
    if (ev) (void)hipEventRecord(ev[3], e->stream);
    T.shade[bs][ml](gs, e->stream, As);
    if (ev) (void)hipEventRecord(ev[4], e->stream);
}

// profiling: one graph's worth of iterations, each kernel between events; waits for them
int launch_profiled(LrhEngine *e)
{
    const int G = e->tune.iters_per_graph;
    while ((int)e->pevs.size() < 5 * G) {
        hipEvent_t ev;
        ENG_HIP(hipEventCreate(&ev));
        e->pevs.push_back(ev);
    }
    for (int i = 0; i < G; i++) launch_iteration(e, e->tune, &e->pevs[5 * i]);
    ENG_HIP(hipGetLastError());
    ENG_HIP(hipEventSynchronize(e->pevs[5 * G - 1]));
    constexpr int stat[4] = {0, 1, 3, 2};   // (the stats' order: regen, extend, shade, shadow)
    const bool joint = e->profiling == 2 && walks_joint(e, e->tune);
    for (int i = 0; i < G; i++)
        for (int k = 0; k < 4; k++) {
            float ms = 0.0f;
            ENG_HIP(hipEventElapsedTime(&ms, e->pevs[5 * i + k], e->pevs[5 * i + k + 1]));
            if (k == 2 && joint) continue;
            e->kms[stat[k]] += ms;
            e->klaunch[stat[k]]++;
        }
    return 0;
}

int make_graph(LrhEngine *e)
{
    if (e->graph_ok) return 0;
    if (e->gexec) (void)hipGraphExecDestroy(e->gexec);
    if (e->graph) (void)hipGraphDestroy(e->graph);
    e->gexec = nullptr;
    e->graph = nullptr;
    ENG_HIP(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
    for (int i = 0; i < e->tune.iters_per_graph; i++) launch_iteration(e, e->tune);
    hipError_t le = hipGetLastError();
    hipError_t ce = hipStreamEndCapture(e->stream, &e->graph);
    if (le != hipSuccess) return eng_fail_dev("graph capture (launch)", le);
    if (ce != hipSuccess) return eng_fail_dev("graph capture", ce);
    ENG_HIP(hipGraphInstantiate(&e->gexec, e->graph, nullptr, nullptr, 0));
    e->graph_ok = true;
    return 0;
}

double dev_ms(const LrhEngine *e, unsigned long long clk)
{
    return e->clk_host0 + ((double)clk - (double)e->clk_dev0) / e->clk_khz;
}

// takes in a progress snapshot: jobs whose paths have all retired are done (a snapshot copied
// before a job's admission may still show the slot's previous job: it is not looked at)
// A pilot job's pass count from its first 4 passes' luminance sums, their means mu_k over the
// image: e4 = sqrt(var(mu) / 4) / mean(mu) the image mean's relative standard error after them,
// K = ceil(4 (e4 / target)^2) the passes that bring it to the target, within [4, spp] (a black
// image: 4). The rest of its paths are issued after this; the device's total follows first.
void pilot_decide(LrhEngine *e, int slot, const long long *sums)
{
    HostJob &h = e->hj[slot];
    const double npix = (double)h.desc.w * (double)h.desc.h;
    double mu[LR_PILOT_PASSES], mean = 0.0, var = 0.0;
    for (int k = 0; k < LR_PILOT_PASSES; k++) {
        mu[k] = (double)sums[k] / (double)(1u << LR_FIX_SHIFT) / npix;
        mean += mu[k] / LR_PILOT_PASSES;
    }
    for (int k = 0; k < LR_PILOT_PASSES; k++) var += (mu[k] - mean) * (mu[k] - mean) / (LR_PILOT_PASSES - 1);
    int K = h.desc.spp;
    double e4 = 0.0;
    if (var == 0.0) K = LR_PILOT_PASSES;
    else if (mean > 0.0) {
        e4 = sqrt(var / LR_PILOT_PASSES) / mean;
        const double t = h.desc.target_error;
        const double k = ceil(LR_PILOT_PASSES * (e4 / t) * (e4 / t));
        K = k < LR_PILOT_PASSES ? LR_PILOT_PASSES : (k > h.desc.spp ? h.desc.spp : (int)k);
    }
    h.pilot = false;
    h.spp_done = K;
    h.rel_error = (float)(e4 * sqrt((double)LR_PILOT_PASSES / K));
    h.total = (unsigned long long)npix * (unsigned long long)K;
    hipLaunchKernelGGL(k_job_total, dim3(1), dim3(1), 0, e->stream, e->jobs, slot, h.total);
}

void absorb(LrhEngine *e, const EngProgress &p, unsigned long long seq)
{
    e->last = p;
    e->last_seq = seq;
    for (int s = 0; s < LR_JOBS; s++) {
        HostJob &j = e->hj[s];
        if (j.state != LRH_JOB_RUNNING || seq < j.min_seq) continue;
        if (j.pilot && p.jret[s] >= j.total) pilot_decide(e, s, p.jpass[s]);
        if (p.jret[s] >= j.total && j.total > 0) {
            j.state = LRH_JOB_DONE;
            j.t_done = dev_ms(e, p.jdone[s]);
            e->running--;
            e->jobs_done++;
        }
    }
    while (!e->recs.empty() && e->recs.front().end <= p.ctl.next) e->recs.pop_front();
}

unsigned long long issue_lo(const LrhEngine *e) { return e->recs.empty() ? e->iq_hi : e->recs.front().rec; }

int progress_enqueue(LrhEngine *e)
{
    const int b = e->pk;
    ENG_HIP(hipMemcpyAsync(e->pin[b], e->prog, sizeof(EngProgress), hipMemcpyDeviceToHost, e->stream));
    ENG_HIP(hipEventRecord(e->pev[b], e->stream));
    e->pend[b] = true;
    e->seq[b] = e->seq_next++;
    e->pk ^= 1;
    return 0;
}

int progress_take(LrhEngine *e, int b)
{
    if (!e->pend[b]) return 0;
    ENG_HIP(hipEventSynchronize(e->pev[b]));
    e->pend[b] = false;
    absorb(e, *e->pin[b], e->seq[b]);
    return 0;
}

// every pending snapshot taken in, oldest first
int progress_flush(LrhEngine *e)
{
    int rc = progress_take(e, e->pk);
    if (!rc) rc = progress_take(e, e->pk ^ 1);
    return rc;
}

// the walks' overflow flags, as the last snapshot has them (taken after everything launched)
int check_overflow(LrhEngine *e)
{
    const uint32_t f = e->last.ctl.overflow;
    if (f & 2u) return lr_fail(LRH_EDEVICE, "engine: a two-level scene's ray reached a one-level walk");
    if (f) return lr_fail(LRH_EREFUSED, "engine: a walk needed more stack than the engine's tree depth allows");
    return 0;
}

size_t arena_first_fit(LrhEngine *e, size_t bytes)
{
    for (auto it = e->free_blocks.begin(); it != e->free_blocks.end(); ++it) {
        if (it->second < bytes) continue;
        const size_t off = it->first, left = it->second - bytes;
        e->free_blocks.erase(it);
        if (left) e->free_blocks[off + bytes] = left;
        return off;
    }
    return (size_t)-1;
}

// a new chunk of device memory in the offset space: false if it cannot be had
bool arena_grow(LrhEngine *e, size_t bytes)
{
    if (e->arena_bytes + bytes > e->arena_cap) return false;
    char *ptr = nullptr;
    if (hipMalloc((void **)&ptr, bytes) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    e->chunks.push_back({e->arena_next, bytes, ptr});
    e->free_blocks[e->arena_next] = bytes;
    e->arena_next += bytes + 256;
    e->arena_bytes += bytes;
    return true;
}

size_t arena_take(LrhEngine *e, size_t bytes)
{
    size_t off = arena_first_fit(e, bytes);
    if (off != (size_t)-1 || !e->arena_lazy) return off;
    // lazy: a chunk of at least 256 MiB (fewer, larger allocations), within the cap
    const size_t room = e->arena_cap - e->arena_bytes;
    size_t want = bytes > ((size_t)256 << 20) ? bytes : ((size_t)256 << 20);
    if (want > room) want = room & ~(size_t)255;
    if (want < bytes || !arena_grow(e, want)) return (size_t)-1;
    return arena_first_fit(e, bytes);
}

// the device address of an arena offset
char *arena_ptr(const LrhEngine *e, size_t off)
{
    for (const ArenaChunk &c : e->chunks)
        if (off >= c.base && off < c.base + c.bytes) return c.ptr + (off - c.base);
    return nullptr;
}

void arena_give(LrhEngine *e, size_t off, size_t bytes)
{
    auto it = e->free_blocks.emplace(off, bytes).first;
    auto nx = std::next(it);
    if (nx != e->free_blocks.end() && it->first + it->second == nx->first) {
        it->second += nx->second;
        e->free_blocks.erase(nx);
    }
    if (it != e->free_blocks.begin()) {
        auto pv = std::prev(it);
        if (pv->first + pv->second == it->first) {
            pv->second += it->second;
            e->free_blocks.erase(it);
        }
    }
}

int job_check(const LrhEngine *e, const LrhJob *j)
{
    if (!j || !j->scene || j->w <= 0 || j->h <= 0 || j->spp <= 0 || j->max_depth < 0)
        return lr_fail(LRH_EINVAL, "engine: bad job");
    const unsigned long long npix = (unsigned long long)j->w * (unsigned long long)j->h;
    if (npix * (unsigned long long)j->spp >= (1ull << 32))
        return lr_fail(LRH_EREFUSED, "engine: %d x %d x %d paths: at most 2^32 per job", j->w, j->h, j->spp);
    if (j->scene->depth > e->max_tree_depth)
        return lr_fail(LRH_EREFUSED, "engine: the scene's tree is %d deep, the engine's walks hold %d", j->scene->depth,
                       e->max_tree_depth);
    if (!(j->photons >= 0.0f) || (j->photons > 0.0f && j->target_error > 0.0f))
        return lr_fail(LRH_EINVAL, "engine: photons >= 0, and not with a target error");
    return 0;
}

// light tracing can add something: a lamp, and a mirror or glass to send its light on
// (scene_has_specular, tracer.c:546-551: a material whose roughness, as its preset makes it, is
// at most 0.02; not a lamp)
bool caustics_possible(const LrhPtScene *s)
{
    if (s->light < 0) return false;
    for (const LrhMaterial &m : s->hmats) {
        if (m.type == LRH_MAT_LIGHT || m.type == LRH_MAT_DIFFUSE) continue;
        if (m.type == LRH_MAT_MIRROR || m.type == LRH_MAT_GLASS) return true;
        const float r = m.roughness < 0.0f ? 0.0f : (m.roughness > 1.0f ? 1.0f : m.roughness);
        if (r <= 0.02f) return true;
    }
    return false;
}

// light paths a pass: photons per pixel (light_paths, trace_gpu.c:1589-1594)
uint32_t light_paths(const LrhJob *j)
{
    const double n = (double)j->photons * j->w * j->h;
    return n < 1.0 ? 1u : (n > 1.6e7 ? 16000000u : (uint32_t)n);
}

// admits a job: its descriptor and its image cleared; its paths are issued later, in chunks
int job_admit(LrhEngine *e, const LrhJob *j, int *slot_out)
{
    int rc = job_check(e, j);
    if (rc) return rc;
    int slot = -1;
    for (int s = 0; s < LR_JOBS; s++)
        if (e->hj[s].state == 0) {
            slot = s;
            break;
        }
    if (slot < 0) return lr_fail(LRH_EAGAIN, "engine: all %d job slots are in use", LR_JOBS);
    const bool caustics = j->photons > 0.0f && caustics_possible(j->scene);
    if (caustics && !e->lq) {
        // the light paths' queue, made on the first job that traces light paths
        if (hipMalloc(&e->lq, (size_t)LR_LIGHT_CHUNK * 64 + 256) != hipSuccess) {
            (void)hipGetLastError();
            e->lq = nullptr;
            return lr_fail(LRH_ENOMEM, "engine: the light paths' queue (%d MB) could not be had", LR_LIGHT_CHUNK >> 14);
        }
        e->lqn = reinterpret_cast<uint32_t *>(reinterpret_cast<char *>(e->lq) + (size_t)LR_LIGHT_CHUNK * 64);
    }
    const size_t npix = (size_t)j->w * (size_t)j->h;
    const size_t bytes = lr_engine_job_bytes(*j);
    const size_t off = arena_take(e, bytes);
    if (off == (size_t)-1) return lr_fail(LRH_EAGAIN, "engine: the image (%zu bytes) does not fit now", bytes);
    HostJob &h = e->hj[slot];
    h = HostJob();
    h.state = LRH_JOB_RUNNING;
    h.id = e->next_id++;
    h.desc = *j;
    h.off = off;
    h.bytes = bytes;
    // a denoised job: the guide (32 bytes a pixel), the moments (16), then the image (24)
    const size_t gbytes = j->denoise ? lr_align(npix * 32) : 0, mbytes = j->denoise ? lr_align(npix * 16) : 0;
    h.guide_off = off;
    h.mom_off = off + gbytes;
    h.acc_off = off + gbytes + mbytes;
    h.total = (unsigned long long)npix * (unsigned long long)j->spp;
    h.spp_done = j->spp;
    if (j->target_error > 0.0f && j->spp > LR_PILOT_PASSES) {
        // a target error: the first 4 passes alone until they decide the pass count
        h.pilot = true;
        h.spp_done = 0;
        h.total = (unsigned long long)npix * LR_PILOT_PASSES;
    }
    h.t_submit = now_ms();
    h.min_seq = e->seq_next;
    const LrhPtScene *s = j->scene;
    h.two_level = s->two_level;
    h.ordered = !s->two_level && s->nprims + s->ntris >= LR_ORDER_SHAPES;
    if (s->two_level && !e->two_level) {
        // from now on the walks that take two-level scenes too; the graphs already launched
        // run before this job's first paths are issued (the same stream)
        e->two_level = true;
        e->graph_ok = false;
    }
    h.odd_eps = !keys_ok(s->eps);
    bool apart = false;
    for (const HostJob &r : e->hj) apart = apart || (r.state == LRH_JOB_RUNNING && r.odd_eps);
    if (apart != e->apart) {   // likewise, the walks' own kernels (until none of those jobs runs)
        e->apart = apart;
        e->graph_ok = false;
    }
    if (lr_scene_multi_light(s) && !e->multi) {   // likewise, shade and shadow for several lights
        e->multi = true;
        e->graph_ok = false;
    }
    JobDev jd;
    memset(&jd, 0, sizeof(jd));
    lr_job_scene(jd, s);
    jd.accum = (long long *)arena_ptr(e, h.acc_off);
    if (j->denoise) {
        jd.guide = (const float4 *)arena_ptr(e, h.guide_off);
        jd.moments = (long long *)arena_ptr(e, h.mom_off);
    }
    jd.total = h.total;
    memcpy(jd.cam, j->cam, sizeof(jd.cam));
    jd.W = j->w;
    jd.H = j->h;
    jd.npix = (int)npix;
    jd.max_depth = j->max_depth;
    jd.mis = j->mis;
    jd.s0 = j->s0;
    jd.seed_lo = (uint32_t)j->seed;
    jd.seed_hi = (uint32_t)(j->seed >> 32);
    jd.clamp = j->clamp;
    jd.pilot = h.pilot ? 1 : 0;
    jd.skip_caustics = caustics ? 1 : 0;
    hipLaunchKernelGGL(k_job_put, dim3(1), dim3(1), 0, e->stream, e->jobs, e->prog->jret, e->prog->jdone, e->prog->jpass,
                       slot, jd);
    // the image cleared (and a denoised job's moments, just before it)
    long long *zero = j->denoise ? jd.moments : jd.accum;
    const size_t words = j->denoise ? (h.acc_off - h.mom_off) / 8 + npix * 3 : npix * 3;
    hipLaunchKernelGGL(k_zero64, dim3((unsigned)((words + SBLOCK - 1) / SBLOCK < 4096 ? (words + SBLOCK - 1) / SBLOCK : 4096)),
                       dim3(SBLOCK), 0, e->stream, zero, words);
    ENG_HIP(hipGetLastError());
    if (j->denoise) {
        // its guide, before any of its paths (the same stream; the walks' spill area is free
        // between the graphs' kernels)
        const size_t threads = std::min((npix + 255) / 256 * 256, (size_t)e->threads_cap / 256 * 256);
        table().guide[s->two_level ? 1 : 0](dim3((unsigned)(threads / 256)), e->stream, jd, (float4 *)jd.guide, e->base.spill,
                                             threads, e->spill_cap, e->base.tab, e->base.overflow);
        ENG_HIP(hipGetLastError());
    }
    if (caustics) {
        // the light paths of all its passes, added to its image now (integer sums: in any order
        // they come to the same), before any of its paths (the same stream)
        const uint32_t nlp = light_paths(j);
        const size_t paths = (size_t)nlp * (size_t)j->spp;
        if (e->profiling && !e->lev[0]) {
            ENG_HIP(hipEventCreate(&e->lev[0]));
            ENG_HIP(hipEventCreate(&e->lev[1]));
        }
        if (e->profiling) ENG_HIP(hipEventRecord(e->lev[0], e->stream));
        // in chunks of at most LR_LIGHT_CHUNK paths (and the engine's threads, for the spill stride)
        const uint64_t chunk = std::min<uint64_t>(LR_LIGHT_CHUNK, (uint64_t)e->threads_cap / 256 * 256);
        for (uint64_t g0 = 0; g0 < (uint64_t)paths; g0 += chunk) {
            const uint32_t n = (uint32_t)std::min<uint64_t>(chunk, (uint64_t)paths - g0);
            table().light[e->counting ? 1 : 0](e->stream, jd, nlp, g0, n, e->base.spill, e->spill_cap, e->base.tab, e->base.overflow,
                                                e->lq, e->lqn, e->counts + 10);
            ENG_HIP(hipGetLastError());
        }
        e->light_paths += paths;
        e->light_launches++;
        if (e->profiling) {
            // (profiling waits for its events, as the iterations' do)
            float ms = 0.0f;
            ENG_HIP(hipEventRecord(e->lev[1], e->stream));
            ENG_HIP(hipEventSynchronize(e->lev[1]));
            ENG_HIP(hipEventElapsedTime(&ms, e->lev[0], e->lev[1]));
            e->light_ms += ms;
        }
    }
    e->by_id[h.id] = slot;
    e->running++;
    *slot_out = slot;
    return 0;
}

// regen orders the bounce rays (LR_ORDER_SHAPES): by the jobs running as paths are issued, so that a
// queue of small scenes, or of large ones after instanced ones, is walked as in a new engine
uint32_t order_bounces(const LrhEngine *e)
{
    uint32_t order = 0;
    for (const HostJob &h : e->hj) {
        if (h.state != LRH_JOB_RUNNING) continue;
        if (h.two_level) return 0;
        order |= h.ordered ? 1u : 0u;
    }
    return order;
}

// issues the next n paths of job `slot` as one record
int issue_chunk(LrhEngine *e, int slot, unsigned long long n)
{
    HostJob &h = e->hj[slot];
    const unsigned long long rec = e->iq_hi++, start = e->issue_end;
    e->issue_end += n;
    e->recs.push_back(IssueRec{rec, start, start + n});
    hipLaunchKernelGGL(k_issue, dim3(1), dim3(1), 0, e->stream, &e->prog->ctl, e->iq_start, e->iq_job, e->iq_q0, rec,
                       start, (uint32_t)slot, (uint32_t)h.issued, e->issue_end, issue_lo(e), order_bounces(e));
    h.issued += n;
    ENG_HIP(hipGetLastError());
    return 0;
}

// Keeps enough paths issued ahead of the device for the next graphs (the host sees the device's
// progress one graph late), chunk by chunk, from the job with the fewest paths left to issue
// (shortest remaining first: small jobs finish early, the device stays full either way).
int top_up(LrhEngine *e)
{
    const unsigned long long target = (unsigned long long)(e->tune.iters_per_graph + 2) * e->C;
    while (e->issue_end - e->last.ctl.next < target && e->iq_hi - issue_lo(e) < LR_ISSUE - 2) {
        int best = -1;
        unsigned long long left = ~0ull;
        for (int s = 0; s < LR_JOBS; s++) {
            const HostJob &h = e->hj[s];
            if (h.state == LRH_JOB_RUNNING && h.issued < h.total && h.total - h.issued < left) {
                left = h.total - h.issued;
                best = s;
            }
        }
        if (best < 0) break;
        int rc = issue_chunk(e, best, left < e->C ? left : e->C);
        if (rc) return rc;
    }
    return 0;
}

// The iterations after which every admitted job is done, where that is known: all paths issued, none
// waiting for a place in the pool (the last snapshot's count of those not yet retired fits it), so
// each starts in the next iteration at the latest and has its max_depth + 1 vertices shaded in as many
// iterations (the last makes no shadow ray). 0: not known.
int tail_iterations(const LrhEngine *e)
{
    unsigned long long left = 0;
    int depth = 0;
    for (int s = 0; s < LR_JOBS; s++) {
        const HostJob &h = e->hj[s];
        if (h.state != LRH_JOB_RUNNING) continue;
        if (h.pilot || h.issued < h.total) return 0;
        left += h.total - (e->last_seq >= h.min_seq ? e->last.jret[s] : 0);
        depth = std::max(depth, std::min(h.desc.max_depth, 1 << 20));
    }
    return left <= e->C ? depth + 1 : 0;
}

int job_slot(const LrhEngine *e, int64_t id)
{
    auto it = e->by_id.find(id);
    return it == e->by_id.end() ? -1 : it->second;
}

}  // namespace

// lrh_engine_create, with an image arena made at once (lazy = false) or chunk by chunk as images
// need it, up to image_bytes in all (lazy = true: the server's, whose budget it must keep)
int lr_engine_create(LrhContext *c, int slots_log2, int max_tree_depth, size_t image_bytes, bool lazy, LrhEngine **out)
{
    if (!c || !out || slots_log2 < 10 || slots_log2 > LR_SLOT_BITS || max_tree_depth < 1 || max_tree_depth > 1024 ||
        image_bytes < 256)
        return lr_fail(LRH_EINVAL, "lrh_engine_create: bad arguments");
    *out = nullptr;
    LR_HIP(hipSetDevice(c->device));
    LrhEngine *e = new LrhEngine();
    e->ctx = c;
    e->device = c->device;
    e->C = 1u << slots_log2;
    e->max_tree_depth = max_tree_depth;
    int ncu = 0, khz = 0;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->device) != hipSuccess || ncu <= 0) ncu = 256;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, c->device) == hipSuccess && khz > 0) e->clk_khz = khz;
    e->ncu = ncu;
    // walk threads: every slot (the plain form's grids) or every persistent work-group's lane
    e->threads_cap = (size_t)e->C + 256;
    if ((size_t)ncu * 16 * 256 > e->threads_cap) e->threads_cap = (size_t)ncu * 16 * 256;
    e->spill_cap = max_tree_depth + 2 - 16 > 0 ? max_tree_depth + 2 - 16 : 0;
    const size_t C = e->C;
    const size_t sizes[] = {
        sizeof(EngProgress), LR_JOBS * sizeof(JobDev), LR_ISSUE * 8, LR_ISSUE * 4,   // 0..3
        2 * C * 16, 2 * C * 16, 2 * C * 8, 2 * C * 8, C * 4,                         // 4..8 thr rad rng meta (2 queues), sq
        C * 32, C * 32, C * 4, C * 4, C * 16,                                        // 9..13 qray qray qid qid hits
        C * 32, C * 4, C * 16,                                                       // 14..16 sray sid scon
        e->threads_cap * (size_t)(e->spill_cap > 0 ? e->spill_cap : 1) * 4,          // 17 spill
        2112 * 4, 4096 * 2, 256, 256, C * 4,                                         // 18..22 tab mask counts clk perm
        LR_ISSUE * 4, (C / 64 + 4) * 8, C * 16,                                      // 23 iq_q0, 24 ostat, 25 srad
        2 * C * 32, 2 * C * 16, C * 4};                                              // 26..28 xsray xscon sx
    constexpr int NS = sizeof(sizes) / sizeof(sizes[0]);
    size_t total = 0;
    for (size_t z : sizes) total += lr_align(z);
    e->arena_cap = image_bytes & ~(size_t)255;
    e->arena_lazy = lazy;
    if (hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) != hipSuccess || hipMalloc(&e->dmem, total) != hipSuccess ||
        (!lazy && !arena_grow(e, e->arena_cap))) {
        (void)hipGetLastError();
        lrh_engine_destroy(e);
        return lr_fail(LRH_ENOMEM, "lrh_engine_create: %zu + %zu bytes of device memory could not be had", total, image_bytes);
    }
    char *p[NS];
    char *at = (char *)e->dmem;
    for (int i = 0; i < NS; i++) {
        p[i] = at;
        at += lr_align(sizes[i]);
    }
    e->prog = (EngProgress *)p[0];
    e->jobs = (JobDev *)p[1];
    e->iq_start = (unsigned long long *)p[2];
    e->iq_job = (uint32_t *)p[3];
    e->iq_q0 = (uint32_t *)p[23];
    e->counts = (unsigned long long *)p[20];
    e->clk = (unsigned long long *)p[21];
    EngArgs &A = e->base;
    A.ctl = &e->prog->ctl;
    A.jobs = e->jobs;
    A.jret = e->prog->jret;
    A.jpass = e->prog->jpass;
    A.jdone = e->prog->jdone;
    A.iq_start = e->iq_start;
    A.iq_job = e->iq_job;
    A.iq_q0 = e->iq_q0;
    for (int b = 0; b < 2; b++) {
        A.thr[b] = (float4 *)p[4] + b * C;
        A.rad[b] = (float4 *)p[5] + b * C;
        A.rng[b] = (uint64_t *)p[6] + b * C;
        A.meta[b] = (uint2 *)p[7] + b * C;
    }
    A.sq = (uint32_t *)p[8];
    A.srad = (float4 *)p[25];
    for (int b = 0; b < 2; b++) {
        A.xsray[b] = (float4 *)p[26] + 2 * b * C;
        A.xscon[b] = (float4 *)p[27] + b * C;
    }
    A.sx = (uint32_t *)p[28];
    A.perm = (uint32_t *)p[22];
    A.qray[0] = (float4 *)p[9];
    A.qray[1] = (float4 *)p[10];
    A.qid[0] = (uint32_t *)p[11];
    A.qid[1] = (uint32_t *)p[12];
    A.hits = (float4 *)p[13];
    A.sray = (float4 *)p[14];
    A.sid = (uint32_t *)p[15];
    A.scon = (float4 *)p[16];
    A.spill = (uint32_t *)p[17];
    A.tab = (const float *)p[18];
    A.mask = (const uint16_t *)p[19];
    A.counts = e->counts;
    A.ostat = (unsigned long long *)p[24];
    A.overflow = &e->prog->ctl.overflow;
    A.mult = 1;
    std::vector<float> tab(2112);
    std::vector<uint16_t> mask(4096);
    lrs_brdf_tables(tab.data());
    lrs_blue_noise(mask.data());
    for (int b = 0; b < 2; b++) {
        if (hipHostMalloc((void **)&e->pin[b], sizeof(EngProgress), hipHostMallocDefault) != hipSuccess ||
            hipEventCreateWithFlags(&e->pev[b], hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            lrh_engine_destroy(e);
            return lr_fail(LRH_ENOMEM, "lrh_engine_create: pinned memory or events could not be had");
        }
    }
    int rc = 0;
    const double t0 = now_ms();
    if (hipMemsetAsync(e->dmem, 0, total, e->stream) != hipSuccess ||
        hipMemcpyAsync(p[18], tab.data(), 2112 * 4, hipMemcpyHostToDevice, e->stream) != hipSuccess ||
        hipMemcpyAsync(p[19], mask.data(), 4096 * 2, hipMemcpyHostToDevice, e->stream) != hipSuccess)
        rc = -1;
    if (!rc) {
        hipLaunchKernelGGL(k_eng_init, dim3(8), dim3(SBLOCK), 0, e->stream, e->prog, e->C);
        hipLaunchKernelGGL(k_clock, dim3(1), dim3(1), 0, e->stream, e->clk);
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(e->stream) != hipSuccess) rc = -1;
    }
    const double t1 = now_ms();
    if (!rc && hipMemcpy(&e->clk_dev0, e->clk, 8, hipMemcpyDeviceToHost) != hipSuccess) rc = -1;
    if (rc) {
        (void)hipGetLastError();
        lrh_engine_destroy(e);
        return lr_fail(LRH_EDEVICE, "lrh_engine_create: the engine's state could not be set up");
    }
    e->clk_host0 = 0.5 * (t0 + t1);
    memset(&e->last, 0, sizeof(e->last));
    e->last.ctl.tail = e->C;
    *out = e;
    return 0;
}

// a lazy arena's cap (chunks already made stay); the device memory its chunks hold
void lr_engine_arena_cap(LrhEngine *e, size_t cap) { e->arena_cap = cap & ~(size_t)255; }
size_t lr_engine_arena_held(const LrhEngine *e) { return e->arena_bytes; }

// frees the chunks of a lazy arena that hold no image
void lr_engine_arena_trim(LrhEngine *e)
{
    if (!e->arena_lazy) return;
    for (size_t k = 0; k < e->chunks.size();) {
        const ArenaChunk c = e->chunks[k];
        auto it = e->free_blocks.find(c.base);
        if (it == e->free_blocks.end() || it->second != c.bytes) {
            k++;
            continue;
        }
        (void)hipSetDevice(e->device);
        (void)hipStreamSynchronize(e->stream);
        (void)hipFree(c.ptr);
        e->free_blocks.erase(it);
        e->arena_bytes -= c.bytes;
        e->chunks.erase(e->chunks.begin() + (long)k);
    }
}

extern "C" {

double lrh_now_ms(void) { return now_ms(); }

void lrh_engine_destroy(LrhEngine *e)
{
    if (!e) return;
    (void)hipSetDevice(e->device);
    if (e->stream) (void)hipStreamSynchronize(e->stream);
    if (e->gexec) (void)hipGraphExecDestroy(e->gexec);
    if (e->graph) (void)hipGraphDestroy(e->graph);
    for (hipEvent_t ev : e->pevs) (void)hipEventDestroy(ev);
    for (hipEvent_t ev : e->lev)
        if (ev) (void)hipEventDestroy(ev);
    if (e->lq) (void)hipFree(e->lq);
    for (int b = 0; b < 2; b++) {
        if (e->pin[b]) (void)hipHostFree(e->pin[b]);
        if (e->pev[b]) (void)hipEventDestroy(e->pev[b]);
    }
    if (e->dmem) (void)hipFree(e->dmem);
    for (const ArenaChunk &ch : e->chunks) (void)hipFree(ch.ptr);
    if (e->stream) (void)hipStreamDestroy(e->stream);
    delete e;
}


int lrh_engine_create(LrhContext *c, int slots_log2, int max_tree_depth, size_t image_bytes, LrhEngine **out)
{
    return lr_engine_create(c, slots_log2, max_tree_depth, image_bytes, false, out);
}

int lrh_engine_tune_set(LrhEngine *e, const LrhTune *t)
{
    if (!e || !t || !tune_valid(*t)) return lr_fail(LRH_EINVAL, "lrh_engine_tune_set: bad launch shape");
    if (memcmp(&e->tune, t, sizeof(LrhTune)) != 0) {
        e->tune = *t;
        e->graph_ok = false;
    }
    return 0;
}

int lrh_engine_tune_get(const LrhEngine *e, LrhTune *t)
{
    if (!e || !t) return lr_fail(LRH_EINVAL, "lrh_engine_tune_get: bad arguments");
    *t = e->tune;
    return 0;
}

int lrh_engine_counting(LrhEngine *e, int on)
{
    if (!e) return lr_fail(LRH_EINVAL, "lrh_engine_counting: no engine");
    if ((bool)on != e->counting) {
        e->counting = on != 0;
        e->graph_ok = false;
    }
    return 0;
}

int lrh_engine_submit(LrhEngine *e, const LrhJob *job, int64_t *id)
{
    if (!e || !job || !id) return lr_fail(LRH_EINVAL, "lrh_engine_submit: bad arguments");
    (void)hipSetDevice(e->device);
    int slot;
    int rc = job_admit(e, job, &slot);
    if (rc) return rc;
    *id = e->hj[slot].id;
    return 0;
}

int lrh_engine_pump(LrhEngine *e, int graphs)
{
    if (!e || graphs < 0) return lr_fail(LRH_EINVAL, "lrh_engine_pump: bad arguments");
    (void)hipSetDevice(e->device);
    int rc = make_graph(e);
    if (rc) return rc;
    for (int g = 0; g < graphs && e->running > 0; g++) {
        rc = top_up(e);
        if (rc) return rc;
        if (e->profiling) rc = launch_profiled(e);
        else {
            hipError_t le = hipGraphLaunch(e->gexec, e->stream);
            if (le != hipSuccess) return eng_fail_dev("hipGraphLaunch", le);
        }
        if (!rc) rc = progress_enqueue(e);
        if (!rc) rc = progress_take(e, e->pk);   // the snapshot before this one
        if (rc) return rc;
    }
    return e->running;
}

int lrh_engine_drain(LrhEngine *e)
{
    if (!e) return lr_fail(LRH_EINVAL, "lrh_engine_drain: no engine");
    (void)hipSetDevice(e->device);
    unsigned long long seen = ~0ull;
    int still = 0;
    while (e->running > 0) {
        int rc = make_graph(e);
        if (!rc) rc = top_up(e);
        if (rc) return rc;
        const int G = e->tune.iters_per_graph, tail = e->profiling ? 0 : tail_iterations(e);
        if (tail > 0 && tail <= 4 * G) {
            // the end is in sight: as many iterations as it takes and no graph past them (whole graphs,
            // then kernels), instead of finding out from snapshots a graph or two late
            for (int g = 0; g < tail / G; g++) {
                hipError_t le = hipGraphLaunch(e->gexec, e->stream);
                if (le != hipSuccess) return eng_fail_dev("hipGraphLaunch", le);
            }
            for (int i = 0; i < tail % G; i++) launch_iteration(e, e->tune);
            ENG_HIP(hipGetLastError());
            rc = progress_enqueue(e);
            if (!rc) rc = progress_flush(e);
        } else rc = lrh_engine_pump(e, 1);
        if (rc < 0) return rc;
        // a stall (no path retired over many graphs) would be a defect: said, not waited on
        const unsigned long long t = e->last.ctl.tail;
        if (t == seen) {
            if (++still > 4096) return lr_fail(LRH_EDEVICE, "lrh_engine_drain: no progress");
        } else {
            seen = t;
            still = 0;
        }
    }
    int rc = progress_flush(e);
    if (!rc) rc = check_overflow(e);
    return rc;
}

int lrh_engine_plain(LrhEngine *e, const LrhJob *job, int64_t *id)
{
    if (!e || !job || !id) return lr_fail(LRH_EINVAL, "lrh_engine_plain: bad arguments");
    if (e->running > 0) return lr_fail(LRH_EINVAL, "lrh_engine_plain: the engine is busy");
    (void)hipSetDevice(e->device);
    const size_t npix = (size_t)job->w * (size_t)job->h;
    if (npix > e->C) return lr_fail(LRH_EREFUSED, "lrh_engine_plain: %zu pixels a pass, %u slots", npix, e->C);
    if (e->iq_hi - issue_lo(e) + (unsigned long long)job->spp >= LR_ISSUE - 2)
        return lr_fail(LRH_EAGAIN, "lrh_engine_plain: too many issue records in use");
    int slot;
    int rc = job_admit(e, job, &slot);
    if (rc) return rc;
    HostJob &h = e->hj[slot];
    const LrEngTable &T = table();
    const LrhTune &t = e->tune;
    const int bt = lr_blk_index(t.block_trace), bs = lr_blk_index(t.block_shade), sk = lr_stk_index(t.stack);
    const dim3 gt((unsigned)((npix + t.block_trace - 1) / t.block_trace)), gs((unsigned)((npix + t.block_shade - 1) / t.block_shade));
    const EngArgs At = args_for(e, t.stack, (size_t)gt.x * t.block_trace, 1);
    const EngArgs As = args_for(e, t.stack, 0, 1);
    const int tl = e->two_level ? 1 : 0, ml = e->multi ? 1 : 0;
    for (int s = 0; s < h.spp_done || h.pilot; s++) {
        if (h.pilot && s == LR_PILOT_PASSES) {
            // a target error: the first passes' sums decide how many passes the job takes
            ENG_HIP(hipStreamSynchronize(e->stream));
            long long sums[LR_PILOT_PASSES];
            ENG_HIP(hipMemcpy(sums, e->prog->jpass[slot], sizeof(sums), hipMemcpyDeviceToHost));
            pilot_decide(e, slot, sums);
            if (s >= h.spp_done) break;
        }
        // the pass: the job's paths s * npix .. (s + 1) * npix - 1, one per pixel
        rc = issue_chunk(e, slot, npix);
        if (rc) return rc;
        // (a vertex's shadow rays are walked with the next one's rays: once more past the last vertex)
        T.regen[bs](gs, e->stream, As);
        for (int d = 0; d <= job->max_depth + 1; d++) {
            if (e->counting || e->apart) {
                (e->counting ? T.extend_count : T.extend)[bt][sk][tl](gt, e->stream, At);
                (e->counting ? T.shadow_count : T.shadow)[bt][sk][tl][ml](gt, e->stream, At);
            } else T.walks[bt][sk][tl][ml](gt, e->stream, At);
            T.shade[bs][ml](gs, e->stream, As);
        }
    }
    ENG_HIP(hipGetLastError());
    ENG_HIP(hipStreamSynchronize(e->stream));    // the host waits for the job (gpu_wait)
    rc = progress_enqueue(e);
    if (!rc) rc = progress_flush(e);
    if (!rc) rc = check_overflow(e);
    if (rc) return rc;
    if (h.state != LRH_JOB_DONE) return lr_fail(LRH_EDEVICE, "lrh_engine_plain: the job did not finish");
    *id = h.id;
    return 0;
}

int lrh_engine_job(LrhEngine *e, int64_t id, LrhJobInfo *info)
{
    if (!e || !info) return lr_fail(LRH_EINVAL, "lrh_engine_job: bad arguments");
    const int s = job_slot(e, id);
    if (s < 0) return lr_fail(LRH_EINVAL, "lrh_engine_job: no job %lld", (long long)id);
    const HostJob &h = e->hj[s];
    info->state = h.state;
    info->w = h.desc.w;
    info->h = h.desc.h;
    info->spp = h.desc.spp;
    info->paths = h.total;
    info->spp_done = h.spp_done;
    info->rel_error = h.rel_error;
    info->t_submit_ms = h.t_submit;
    info->t_done_ms = h.state == LRH_JOB_DONE ? h.t_done : 0.0;
    return 0;
}

int lrh_engine_image(LrhEngine *e, int64_t id, float *d_out, int add)
{
    if (!e || !d_out) return lr_fail(LRH_EINVAL, "lrh_engine_image: bad arguments");
    const int s = job_slot(e, id);
    if (s < 0) return lr_fail(LRH_EINVAL, "lrh_engine_image: no job %lld", (long long)id);
    const HostJob &h = e->hj[s];
    if (h.state != LRH_JOB_DONE) return lr_fail(LRH_EAGAIN, "lrh_engine_image: job %lld is not done", (long long)id);
    const int npix = h.desc.w * h.desc.h;
    hipLaunchKernelGGL(k_resolve, dim3((npix + SBLOCK - 1) / SBLOCK), dim3(SBLOCK), 0, e->stream,
                       (const long long *)arena_ptr(e, h.acc_off), npix, (float)h.spp_done, (float4 *)d_out, add);
    ENG_HIP(hipGetLastError());
    ENG_HIP(hipStreamSynchronize(e->stream));
    return 0;
}

int lrh_engine_guide(LrhEngine *e, int64_t id, float *d_guide, float *d_moments)
{
    const int slot = job_slot(e, id);
    if (slot < 0 || !d_guide || !d_moments) return lr_fail(LRH_EINVAL, "lrh_engine_guide: unknown job %lld or no output", (long long)id);
    const HostJob &h = e->hj[slot];
    if (!h.desc.denoise) return lr_fail(LRH_EINVAL, "lrh_engine_guide: job %lld was not submitted with denoise = 1", (long long)id);
    if (h.state != LRH_JOB_DONE) return lr_fail(LRH_EAGAIN, "lrh_engine_guide: job %lld is not done", (long long)id);
    const int npix = h.desc.w * h.desc.h;
    ENG_HIP(hipSetDevice(e->device));
    ENG_HIP(hipMemcpyAsync(d_guide, arena_ptr(e, h.guide_off), (size_t)npix * 32, hipMemcpyDeviceToDevice, e->stream));
    hipLaunchKernelGGL(k_moments, dim3((npix + SBLOCK - 1) / SBLOCK), dim3(SBLOCK), 0, e->stream,
                       (const long long *)arena_ptr(e, h.mom_off), npix, (float2 *)d_moments);
    ENG_HIP(hipGetLastError());
    ENG_HIP(hipStreamSynchronize(e->stream));
    return 0;
}

int lrh_engine_denoise(LrhEngine *e, int64_t id, int passes, float *d_out)
{
    const int slot = job_slot(e, id);
    if (slot < 0 || !d_out || passes < 1 || passes > 5)
        return lr_fail(LRH_EINVAL, "lrh_engine_denoise: unknown job %lld, no output, or passes not in 1..5", (long long)id);
    const HostJob &h = e->hj[slot];
    if (!h.desc.denoise) return lr_fail(LRH_EINVAL, "lrh_engine_denoise: job %lld was not submitted with denoise = 1", (long long)id);
    if (h.state != LRH_JOB_DONE) return lr_fail(LRH_EAGAIN, "lrh_engine_denoise: job %lld is not done", (long long)id);
    const int W = h.desc.w, H = h.desc.h, npix = W * H;
    ENG_HIP(hipSetDevice(e->device));
    // the image (float4 sums and counts) and the moments (float2) beside the filter's own buffers
    const size_t fa = lr_align((size_t)npix * 16), fm = lr_align((size_t)npix * 8);
    char *tmp = nullptr;
    if (hipMalloc((void **)&tmp, fa + fm + lr_denoise_scratch_bytes(W, H)) != hipSuccess) {
        (void)hipGetLastError();
        return lr_fail(LRH_ENOMEM, "lrh_engine_denoise: device memory for the filter could not be had");
    }
    hipLaunchKernelGGL(k_resolve, dim3((npix + SBLOCK - 1) / SBLOCK), dim3(SBLOCK), 0, e->stream,
                       (const long long *)arena_ptr(e, h.acc_off), npix, (float)h.spp_done, (float4 *)tmp, 0);
    hipLaunchKernelGGL(k_moments, dim3((npix + SBLOCK - 1) / SBLOCK), dim3(SBLOCK), 0, e->stream,
                       (const long long *)arena_ptr(e, h.mom_off), npix, (float2 *)(tmp + fa));
    int rc = hipGetLastError() == hipSuccess ? 0 : lr_fail(LRH_EDEVICE, "lrh_engine_denoise: a launch failed");
    if (!rc)
        rc = lr_denoise_launch(e->stream, (const float *)tmp, (const float *)(tmp + fa), (const float *)arena_ptr(e, h.guide_off),
                               W, H, passes, tmp + fa + fm, d_out);
    if (hipStreamSynchronize(e->stream) != hipSuccess && !rc) rc = lr_fail(LRH_EDEVICE, "lrh_engine_denoise: the filter failed");
    (void)hipFree(tmp);
    return rc;
}

int lrh_engine_release(LrhEngine *e, int64_t id)
{
    if (!e) return lr_fail(LRH_EINVAL, "lrh_engine_release: no engine");
    const int s = job_slot(e, id);
    if (s < 0) return lr_fail(LRH_EINVAL, "lrh_engine_release: no job %lld", (long long)id);
    HostJob &h = e->hj[s];
    if (h.state != LRH_JOB_DONE) return lr_fail(LRH_EAGAIN, "lrh_engine_release: job %lld is running", (long long)id);
    arena_give(e, h.off, h.bytes);
    e->by_id.erase(id);
    h = HostJob();
    return 0;
}

int lrh_engine_stats(LrhEngine *e, LrhEngineStats *st)
{
    if (!e || !st) return lr_fail(LRH_EINVAL, "lrh_engine_stats: bad arguments");
    int rc = progress_flush(e);
    if (rc) return rc;
    unsigned long long cnt[14] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    ENG_HIP(hipMemcpyAsync(cnt, e->counts, sizeof cnt, hipMemcpyDeviceToHost, e->stream));
    ENG_HIP(hipStreamSynchronize(e->stream));
    st->rays_ext = e->last.ctl.rays_ext;
    st->rays_shadow = e->last.ctl.rays_shadow;
    st->iterations = e->last.ctl.iter;
    st->jobs_done = e->jobs_done;
    st->node_fetches = cnt[0];
    st->shape_tests = cnt[1];
    st->wave_node_steps = cnt[2];
    st->wave_shape_steps = cnt[3];
    st->shadow_node_fetches = cnt[4];
    st->shadow_shape_tests = cnt[5];
    st->shadow_wave_node_steps = cnt[6];
    st->shadow_wave_shape_steps = cnt[7];
    st->uniform_node_steps = cnt[8];
    st->shadow_uniform_node_steps = cnt[9];
    st->light_paths = e->light_paths;
    st->light_rays = cnt[10];
    st->light_shadow_rays = cnt[11];
    st->light_node_fetches = cnt[12];
    st->light_shape_tests = cnt[13];
    st->light_launches = e->light_launches;
    st->light_ms = e->light_ms;
    for (int k = 0; k < 4; k++) {
        st->kernel_ms[k] = e->kms[k];
        st->kernel_launches[k] = e->klaunch[k];
    }
    return 0;
}

int lrh_engine_profiling(LrhEngine *e, int on)
{
    if (!e) return lr_fail(LRH_EINVAL, "lrh_engine_profiling: no engine");
    e->profiling = on == 2 ? 2 : (on ? 1 : 0);
    return 0;
}

int lrh_engine_autotune(LrhEngine *e, const LrhJob *sample, int n, LrhTune *best, double *mrays)
{
    if (!e || !sample || n <= 0) return lr_fail(LRH_EINVAL, "lrh_engine_autotune: bad arguments");
    if (e->running > 0) return lr_fail(LRH_EINVAL, "lrh_engine_autotune: the engine is busy");
    hipEvent_t ev[2];
    ENG_HIP(hipEventCreate(&ev[0]));
    ENG_HIP(hipEventCreate(&ev[1]));
    // one timed run of the sample jobs under launch shape t: rays per microsecond
    auto run_once = [&](const LrhTune &t, double &score) -> int {
        int rc = lrh_engine_tune_set(e, &t);
        if (!rc) rc = make_graph(e);
        if (rc) return rc;
        const unsigned long long r0 = e->last.ctl.rays_ext + e->last.ctl.rays_shadow;
        std::vector<int64_t> ids;
        ENG_HIP(hipEventRecord(ev[0], e->stream));
        for (int i = 0; i < n; i++) {
            int64_t id;
            rc = lrh_engine_submit(e, &sample[i], &id);
            if (rc == LRH_EAGAIN) break;
            if (rc) return rc;
            ids.push_back(id);
        }
        if (ids.empty()) return lr_fail(LRH_EREFUSED, "lrh_engine_autotune: no sample job fits the engine");
        rc = lrh_engine_drain(e);
        if (rc) return rc;
        ENG_HIP(hipEventRecord(ev[1], e->stream));
        ENG_HIP(hipEventSynchronize(ev[1]));
        float ms = 0.0f;
        ENG_HIP(hipEventElapsedTime(&ms, ev[0], ev[1]));
        for (int64_t id : ids) lrh_engine_release(e, id);
        const unsigned long long r1 = e->last.ctl.rays_ext + e->last.ctl.rays_shadow;
        score = ms > 0.0f ? (double)(r1 - r0) / (ms * 1e3) : 0.0;
        return 0;
    };
    // the better of two runs (one run of a short sample is at the mercy of clocks and caches)
    auto measure = [&](const LrhTune &t, double &score) -> int {
        double a = 0.0, b = 0.0;
        int rc = run_once(t, a);
        if (!rc) rc = run_once(t, b);
        score = a > b ? a : b;
        return rc;
    };
    LrhTune cur = e->tune, win = cur;
    double top = 0.0, s = 0.0;
    int rc = measure(cur, s);   // a first run warms the caches and the code up
    if (!rc) rc = measure(cur, top);
    const int blks[3] = {64, 128, 256}, stks[3] = {16, 24, 32}, bpcs[5] = {1, 2, 4, 8, 16}, tiles[4] = {1, 2, 4, 8};
    auto consider = [&](const LrhTune &t) {
        if (rc || memcmp(&t, &win, sizeof(LrhTune)) == 0) return;
        double sc = 0.0;
        rc = measure(t, sc);
        if (!rc && sc > top) {
            top = sc;
            win = t;
        }
    };
    for (int b : blks)
        for (int k : stks) {
            LrhTune t = win;
            t.block_trace = b;
            t.stack = k;
            consider(t);
        }
    for (int v : bpcs) {
        LrhTune t = win;
        t.blocks_per_cu = v;
        consider(t);
    }
    for (int v : tiles) {
        LrhTune t = win;
        t.tile = v;
        consider(t);
    }
    for (int b : blks) {
        LrhTune t = win;
        t.block_shade = b;
        consider(t);
    }
    for (int v : {0, 8, 16, 32}) {
        LrhTune t = win;
        t.refill = v;
        consider(t);
    }
    for (int v : {0, 8, 16, 32}) {
        LrhTune t = win;
        t.refill_shadow = v;
        consider(t);
    }
    (void)hipEventDestroy(ev[0]);
    (void)hipEventDestroy(ev[1]);
    if (rc) return rc;
    rc = lrh_engine_tune_set(e, &win);
    if (rc) return rc;
    if (best) *best = win;
    if (mrays) *mrays = top;
    return 0;
}

// lrh_pt_render_job: a one-job batch on the context's own engine (made, or made larger, on demand)
int lrh_pt_render_job(LrhContext *c, const LrhJob *j, float *d_accum)
{
    if (!c || !j || !j->scene || !d_accum || j->w <= 0 || j->h <= 0 ||
        (unsigned long long)j->w * (unsigned long long)j->h >= (1ull << 32))
        return lr_fail(LRH_EINVAL, "lrh_pt_render_job: bad arguments");
    if (j->denoise) return lr_fail(LRH_EINVAL, "lrh_pt_render_job: a denoised job needs an engine (lrh_engine_denoise)");
    const LrhPtScene *s = j->scene;
    const size_t need = lr_align((size_t)j->w * j->h * 24);
    LrhEngine *e = c->engine;
    if (e && (e->max_tree_depth < s->depth || e->arena_bytes < need)) {
        lrh_engine_destroy(e);
        c->engine = e = nullptr;
    }
    if (!e) {
        const size_t img = need > ((size_t)64 << 20) ? need : ((size_t)64 << 20);
        int rc = lrh_engine_create(c, 20, s->depth > 64 ? s->depth : 64, img, &e);
        if (rc) return rc;
        c->engine = e;
    }
    // the caller's stream may still be writing d_accum or the scene
    LR_HIP(hipStreamSynchronize(c->stream));
    int64_t id;
    int rc = lrh_engine_submit(e, j, &id);
    if (!rc) rc = lrh_engine_drain(e);
    if (!rc) rc = lrh_engine_image(e, id, d_accum, 1);
    if (!rc) rc = lrh_engine_release(e, id);
    return rc;
}

// lrh_pt_render: lrh_pt_render_job of a plain job
int lrh_pt_render(LrhContext *c, const LrhPtScene *s, const float *cam, int W, int H, int spp, uint32_t s0, uint64_t seed,
                  int max_depth, int mis, float clamp, float *d_accum)
{
    if (!c || !s || !cam || W <= 0 || H <= 0 || spp <= 0 || max_depth < 0 || !d_accum)
        return lr_fail(LRH_EINVAL, "lrh_pt_render: bad arguments");
    LrhJob j{};   // (no denoiser inputs, no target error, no light tracing)
    j.scene = s;
    memcpy(j.cam, cam, sizeof(j.cam));
    j.w = W;
    j.h = H;
    j.spp = spp;
    j.s0 = s0;
    j.seed = seed;
    j.max_depth = max_depth;
    j.mis = mis;
    j.clamp = clamp;
    return lrh_pt_render_job(c, &j, d_accum);
}

}  // extern "C"
