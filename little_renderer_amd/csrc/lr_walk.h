// lr_walk.h - the BVH walk and the shape tests, shared by the trace kernels (lr_trace.hip)
// and the path tracer's extension and shadow kernels (lr_engine_k.h).
//
// The walk and its arithmetic are trace.wgsl traverse (:270-392), hit_tri (:159-173),
// hit_sphere / hit_quad (:130-157) and box_t (:175-184) with safe_inv (media.wgsl:45-48):
// the same f32 operations in the same order (the library is built without fused
// multiply-add), so hits equal the oracle's to the bit on the same tree. The stack differs
// from the reference's 40 entries that drop what does not fit: the first LR_LDS_STACK
// entries of each ray live in LDS (interleaved by lane: no bank conflicts) and deeper ones
// spill to device memory, sized from the tree's depth, so nothing is ever dropped. Sixteen
// LDS entries (8 KB for a work-group of 128) leave the walk kernels at their register-bound
// occupancy; the binary walk pushes only the farther child, so deep entries are rare (its entries in
// LDS: lr_trace.hip).
#pragma once

#include "lr_device.h"

#define LR_LDS_STACK 16

struct V3 {
    float x, y, z;
};
__device__ __forceinline__ V3 v3(float x, float y, float z) { return V3{x, y, z}; }
__device__ __forceinline__ V3 v3of(float4 a) { return V3{a.x, a.y, a.z}; }
__device__ __forceinline__ V3 vadd(V3 a, V3 b) { return v3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ V3 vsub(V3 a, V3 b) { return v3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ V3 vmul(V3 a, V3 b) { return v3(a.x * b.x, a.y * b.y, a.z * b.z); }
__device__ __forceinline__ V3 vscale(V3 a, float s) { return v3(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ V3 vneg(V3 a) { return v3(-a.x, -a.y, -a.z); }
__device__ __forceinline__ float vdot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ V3 vcross(V3 a, V3 b)
{
    return v3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}

__device__ __forceinline__ float safe_inv(float d) { return fabsf(d) > 1e-12f ? 1.0f / d : 1e30f; }

// box_t (trace.wgsl:175-184): the entry distance, -1 on a miss
__device__ __forceinline__ float box_t(float4 lo, float4 hi, V3 o, V3 inv, float tmin, float tmax)
{
    const float t0x = (lo.x - o.x) * inv.x, t0y = (lo.y - o.y) * inv.y, t0z = (lo.z - o.z) * inv.z;
    const float t1x = (hi.x - o.x) * inv.x, t1y = (hi.y - o.y) * inv.y, t1z = (hi.z - o.z) * inv.z;
    const float enter = wmax(wmax(wmin(t0x, t1x), wmin(t0y, t1y)), wmax(wmin(t0z, t1z), tmin));
    const float leave = wmin(wmin(wmax(t0x, t1x), wmax(t0y, t1y)), wmin(wmax(t0z, t1z), tmax));
    return leave < enter ? -1.0f : enter;
}

// box_t of two boxes for the binary walk, by minima and maxima that pass a NaN on (one instruction
// each, three operands, where wmin and wmax are a compare and a select): the same answers unless a NaN
// is in one of them, which shows in its entry or exit, and then box_t's own
__device__ __forceinline__ float nmin(float a, float b) { return __builtin_elementwise_minimum(a, b); }
__device__ __forceinline__ float nmax(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ void slab_(float4 lo, float4 hi, V3 o, V3 inv, float tmin, float tmax, float &enter, float &leave)
{
    const float t0x = (lo.x - o.x) * inv.x, t0y = (lo.y - o.y) * inv.y, t0z = (lo.z - o.z) * inv.z;
    const float t1x = (hi.x - o.x) * inv.x, t1y = (hi.y - o.y) * inv.y, t1z = (hi.z - o.z) * inv.z;
    enter = nmax(nmax(nmax(nmin(t0x, t1x), nmin(t0y, t1y)), nmin(t0z, t1z)), tmin);
    leave = nmin(nmin(nmin(nmax(t0x, t1x), nmax(t0y, t1y)), nmax(t0z, t1z)), tmax);
}
__device__ __forceinline__ void box_t2(float4 alo, float4 ahi, float4 blo, float4 bhi, V3 o, V3 inv, float tmin, float tmax,
                                       float &ta, float &tb)
{
    float ea, la, eb, lb;
    slab_(alo, ahi, o, inv, tmin, tmax, ea, la);
    slab_(blo, bhi, o, inv, tmin, tmax, eb, lb);
    ta = la < ea ? -1.0f : ea;
    tb = lb < eb ? -1.0f : eb;
    if (__builtin_isunordered(ea, la) || __builtin_isunordered(eb, lb)) {
        ta = box_t(alo, ahi, o, inv, tmin, tmax);
        tb = box_t(blo, bhi, o, inv, tmin, tmax);
    }
}

// hit_tri (trace.wgsl:159-173): t in (tmin, tmax) and the barycentrics
__device__ __forceinline__ bool hit_tri(float4 a, float4 b, float4 c, V3 o, V3 d, float tmin, float tmax, float &t_out,
                                        float &u_out, float &v_out)
{
    const V3 q = v3of(a), u = v3of(b), v = v3of(c);
    const V3 pvec = vcross(d, v);
    const float det = vdot(u, pvec);
    if (fabsf(det) < 1e-12f) return false;
    const float inv = 1.0f / det;
    const V3 tvec = vsub(o, q);
    const float b1 = vdot(tvec, pvec) * inv;
    if (b1 < 0.0f || b1 > 1.0f) return false;
    const V3 qvec = vcross(tvec, u);
    const float b2 = vdot(d, qvec) * inv;
    if (b2 < 0.0f || b1 + b2 > 1.0f) return false;
    const float t = vdot(v, qvec) * inv;
    if (t <= tmin || t >= tmax) return false;
    t_out = t;
    u_out = b1;
    v_out = b2;
    return true;
}

// a primitive's 96-byte record (trace.wgsl:3-10): c centre+radius, q corner (w: 0 sphere,
// 1 quad), u edge (w: material), v edge (w: area), n unit normal (w: plane_d), w = (u x v)/|u x v|^2
struct Prim {
    float4 c, q, u, v, n, w;
};

// hit_sphere (trace.wgsl:130-144)
__device__ __forceinline__ float hit_sphere(const Prim &p, V3 o, V3 d, float tmin, float tmax)
{
    const V3 oc = vsub(v3of(p.c), o);
    const float a = vdot(d, d), hh = vdot(d, oc), c = vdot(oc, oc) - p.c.w * p.c.w;
    const float disc = hh * hh - a * c;
    if (disc < 0.0f) return -1.0f;
    const float sq = sqrtf(disc);
    float t = (hh - sq) / a;
    if (t <= tmin || t >= tmax) {
        t = (hh + sq) / a;
        if (t <= tmin || t >= tmax) return -1.0f;
    }
    return t;
}

// hit_quad (trace.wgsl:146-157)
__device__ __forceinline__ float hit_quad(const Prim &p, V3 o, V3 d, float tmin, float tmax, float &a_out, float &b_out)
{
    const V3 n = v3of(p.n);
    const float denom = vdot(n, d);
    if (fabsf(denom) < 1e-12f) return -1.0f;
    const float t = (p.n.w - vdot(n, o)) / denom;
    if (t <= tmin || t >= tmax) return -1.0f;
    const V3 rel = vsub(vadd(o, vscale(d, t)), v3of(p.q));
    const float a = vdot(v3of(p.w), vcross(rel, v3of(p.v)));
    const float b = vdot(v3of(p.w), vcross(v3of(p.u), rel));
    if (a < 0.0f || a > 1.0f || b < 0.0f || b > 1.0f) return -1.0f;
    a_out = a;
    b_out = b;
    return t;
}

__device__ __forceinline__ Prim load_prim(const float4 *prims, uint32_t id)
{
    const float4 *p = prims + 6 * (size_t)id;
    return Prim{p[0], p[1], p[2], p[3], p[4], p[5]};
}

// hit_sphere / hit_quad on a record read as it is needed (the quad's edges only once its plane
// is hit): the same arithmetic, fewer registers held in the walks
__device__ __forceinline__ float hit_prim(const float4 *__restrict__ prims, uint32_t id, V3 o, V3 d, float tmin, float tmax,
                                          float &a_out, float &b_out)
{
    const size_t p = 6 * (size_t)id;
    const float4 q = ldg4(prims, p + 1);
    if (q.w < 0.5f) {
        Prim s;
        s.c = ldg4(prims, p);
        return hit_sphere(s, o, d, tmin, tmax);
    }
    const float4 nn = ldg4(prims, p + 4);
    const V3 n = v3of(nn);
    const float denom = vdot(n, d);
    if (fabsf(denom) < 1e-12f) return -1.0f;
    const float t = (nn.w - vdot(n, o)) / denom;
    if (t <= tmin || t >= tmax) return -1.0f;
    const float4 u = ldg4(prims, p + 2), v = ldg4(prims, p + 3), w = ldg4(prims, p + 5);
    const V3 rel = vsub(vadd(o, vscale(d, t)), v3of(q));
    const float a = vdot(v3of(w), vcross(rel, v3of(v)));
    const float b = vdot(v3of(w), vcross(v3of(u), rel));
    if (a < 0.0f || a > 1.0f || b < 0.0f || b > 1.0f) return -1.0f;
    a_out = a;
    b_out = b;
    return t;
}

struct WalkHit {
    float t;
    uint32_t id;
    float b1, b2;
};

// The stack of one ray: LDS slots stk[k * stride] for k < STK (the walk's template
// argument), then spill[(k - STK) * sstride] up to cap entries in all.
struct WalkStack {
    uint32_t *stk;
    int stride;
    uint32_t *spill;
    size_t sstride;
    int cap;
};

// entry sp of a walk's stack (LDS for the first STK, device memory past them). The LDS entry is
// read whatever sp is (at a clamped place) and the device one only past STK, as an atomic load
// (which the compiler does not merge with the other), so that the two stay an LDS read and a
// rare global one instead of becoming one flat read through a selected address (a vector
// memory instruction on every pop)
template <int STK>
__device__ __forceinline__ uint32_t stk_get(const WalkStack &S, int sp)
{
    uint32_t x = S.stk[(sp < STK ? sp : STK - 1) * S.stride];
    if (sp >= STK) x = __hip_atomic_load(&S.spill[(size_t)(sp - STK) * S.sstride], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    return x;
}

// The closest hit in (tmin, tmax), or (ANY) the first one, over shape ids taken from the
// leaves' aux entries: ids below nprims are primitives, the rest triangles (id - nprims).
//
// The nodes are visited in the reference's order (pop a node; test its two children's boxes;
// push the farther hit child, then the nearer, and pop again), but the nearer child is not
// pushed and popped: it stays in registers as the next entry, with its two child fields
// (lo.w, hi.w), which its parent's box test has already loaded. A farther child's two words go to
// the stack in its place in the first PAIRS entries (S.stk: PAIRS + STK words a ray, for STK entries);
// past them its index does, and the pop fetches them. The reference fetches the whole record of every
// node it pops. Same visits, same tests, same hits. Bound by the loads' data path (a wave's lanes are at
// different nodes, so a load takes 16 cycles or more whatever its width): without the pops' two loads,
// and with box_t2 (a third of it), 1920 x 1080 camera rays through a PLOC tree of 1M triangles take 2.02
// ms, before 2.26; with 14 two-word entries in LDS instead of 10, and fewer waves, 18 % more.
// COUNT adds the node records fetched (the root's, each inner node's two children, each popped node's
// past the PAIRS entries) and the shapes tested to cn, ct.
template <bool ANY, bool PRIMS, bool COUNT, int PAIRS, int STK>
__device__ __forceinline__ WalkHit walk(const float4 *__restrict__ nodes, uint32_t root, const uint32_t *__restrict__ aux,
                                        const float4 *__restrict__ tris, const float4 *__restrict__ prims, uint32_t nprims,
                                        V3 o, V3 d, float tmin, float tmax, const WalkStack &S, uint32_t *overflow,
                                        uint32_t &cn, uint32_t &ct)
{
    const V3 inv = v3(safe_inv(d.x), safe_inv(d.y), safe_inv(d.z));
    WalkHit best{tmax, LR_NONE, 0.0f, 0.0f};
    const float *words = reinterpret_cast<const float *>(nodes);
    // the entry being visited: its record's lo.w and hi.w (inner: the children; leaf: the
    // first aux entry, then LR_LEAF | count)
    uint32_t na = __float_as_uint(words[8 * (size_t)root + 3]), nb = __float_as_uint(words[8 * (size_t)root + 7]);
    if (COUNT) cn++;
    int sp = 0;
    auto pop = [&] {
        sp--;
        if (sp < PAIRS) {
            na = S.stk[2 * sp * S.stride];
            nb = S.stk[(2 * sp + 1) * S.stride];
        } else {
            const uint32_t ni = sp < STK ? S.stk[(PAIRS + sp) * S.stride] : S.spill[(size_t)(sp - STK) * S.sstride];
            na = __float_as_uint(words[8 * (size_t)ni + 3]);
            nb = __float_as_uint(words[8 * (size_t)ni + 7]);
            if (COUNT) cn++;
        }
    };
    for (;;) {
        while (nb & LR_LEAF) {
            const uint32_t cnt = nb & 0x7fffffffu;
            for (uint32_t k = 0; k < cnt; k++) {
                const uint32_t sid = aux[na + k];
                if (COUNT) ct++;
                if (PRIMS && sid < nprims) {
                    const Prim p = load_prim(prims, sid);
                    float a = 0.0f, b = 0.0f;
                    const float t = p.q.w < 0.5f ? hit_sphere(p, o, d, tmin, best.t) : hit_quad(p, o, d, tmin, best.t, a, b);
                    if (t > 0.0f) {
                        best = WalkHit{t, sid, a, b};
                        if (ANY) return best;
                    }
                    continue;
                }
                const uint32_t ti = PRIMS ? sid - nprims : sid;
                const float4 ta = tris[3 * (size_t)ti], tb = tris[3 * (size_t)ti + 1], tc = tris[3 * (size_t)ti + 2];
                float t, u, v;
                if (hit_tri(ta, tb, tc, o, d, tmin, best.t, t, u, v)) {
                    best = WalkHit{t, sid, u, v};
                    if (ANY) return best;
                }
            }
            if (sp == 0) return best;
            pop();
        }
        const float4 alo = nodes[2 * (size_t)na], ahi = nodes[2 * (size_t)na + 1];
        const float4 blo = nodes[2 * (size_t)nb], bhi = nodes[2 * (size_t)nb + 1];
        float tl, tr;
        box_t2(alo, ahi, blo, bhi, o, inv, tmin, best.t, tl, tr);
        if (COUNT) cn += 2;
        if (tl >= 0.0f && tr >= 0.0f) {
            if (sp + 1 > S.cap) {   // cannot happen with a correct depth: said, never silently dropped
                atomicOr(overflow, 1u);
                break;
            }
            const bool left_first = tl <= tr;
            if (sp < PAIRS) {
                S.stk[2 * sp * S.stride] = __float_as_uint(left_first ? blo.w : alo.w);
                S.stk[(2 * sp + 1) * S.stride] = __float_as_uint(left_first ? bhi.w : ahi.w);
            } else if (sp < STK) S.stk[(PAIRS + sp) * S.stride] = left_first ? nb : na;
            else S.spill[(size_t)(sp - STK) * S.sstride] = left_first ? nb : na;
            sp++;
            na = __float_as_uint(left_first ? alo.w : blo.w);
            nb = __float_as_uint(left_first ? ahi.w : bhi.w);
        } else if (tl >= 0.0f) {
            na = __float_as_uint(alo.w);
            nb = __float_as_uint(ahi.w);
        } else if (tr >= 0.0f) {
            na = __float_as_uint(blo.w);
            nb = __float_as_uint(bhi.w);
        } else {
            if (sp == 0) break;
            pop();
        }
    }
    return best;
}


// A walk's own counters (its counting variants): node records fetched and shapes tested by the
// lane, and the steps its wave took to do them (each counted once, by the wave's first lane at
// work in it), so that fetched / (64 x node steps) and tested / (64 x shape steps) are the shares
// of a wave's lanes at work in its node and shape steps.
struct WalkCnt {
    uint32_t n = 0, t = 0, wn = 0, wt = 0, wu = 0;   // wu: node steps whose lanes all fetch one node
};
__device__ __forceinline__ bool wave_first_lane() { return lane_id() == (uint32_t)__builtin_ctzll(__ballot(1)); }
__device__ __forceinline__ void count_node(WalkCnt &c)
{
    c.n++;
    if (wave_first_lane()) c.wn++;
}
// a node step at node k of the tree at w: counted as uniform when every lane at work in it is at
// the same node of the same tree
__device__ __forceinline__ void count_uniform(WalkCnt &c, const void *w, uint32_t k)
{
    const uint64_t p = (uint64_t)w;
    const uint32_t fk = __builtin_amdgcn_readfirstlane(k);
    const uint32_t flo = __builtin_amdgcn_readfirstlane((uint32_t)p), fhi = __builtin_amdgcn_readfirstlane((uint32_t)(p >> 32));
    const bool same = k == fk && (uint32_t)p == flo && (uint32_t)(p >> 32) == fhi;
    const uint64_t differ = __ballot(!same);
    if (wave_first_lane() && differ == 0) c.wu++;
}
__device__ __forceinline__ void count_shape(WalkCnt &c)
{
    c.t++;
    if (wave_first_lane()) c.wt++;
}

// ---- the engine's 4-wide walk ---------------------------------------------------------------
// The tree is an array of 48-byte slots (3 float4), each an inner node or a leaf, made by
// k_collapse (lr_pt_scene.hip) from the binary tree with the collapse rule of bvh.c:497-530; a
// node's 2 to 4 children lie side by side in child order. An entry (what the walks hold and
// stack) is a slot's first float4.
//   inner  corner.xyz, three axes' scale exponents (signed bytes 0..2) | children << 24
//          the children's lo.x, lo.y, lo.z as 8-bit steps from the corner (byte k: child k), the first child's entry
//          their hi.x, hi.y, hi.z, 0
//   leaf   q.xyz, LR_LEAF | u.xyz, shape id | v.xyz, 0 (a primitive: its record is read from prims; an
//          instance: kind and mesh root entry in q.x, q.y, its index for the shape id)
// The children's boxes are rounded outwards. What a slot is shows in its own word 3, so a wave's
// lanes load their nodes and leaves with the same three instructions and a child needs no reference
// of its own: nodes were 64 bytes with four references (a fourth load and four words to carry
// through the sort), a leaf's triangle and id two arrays more, the triangle's load waiting for the id.
// The walks are bound by their VALU instructions (a wave's lanes diverge) and the texture path: three
// loads a step and a place instead of a reference to carry took the extension walk of a 54M-path queue
// from 32.3 to 26.1 ms, its shadow walk from 22.6 to 18.1 ms, and 300,000 rays with nothing in common
// through 50,000 triangles from 273 to 160 us, with the children's distance and place sorted as one
// word. That cannot tell distances within 16 ulp, nor leave equal ones where they were, and so took
// another of the shapes that coincide (2 % of the rays at squares over one another in a plane). Whole
// distances, each with its place beside it, took 1.4 to 2.7 % longer; as keys of 64 bits (wide_next)
// they take what the one word did (the last 158 us), and every hit is the one it was. Two-level walks
// exchange distance and place: with the keys' pairs of registers they would lose one to two of their
// 6 waves a SIMD (two instanced frames 15.2 to 15.8 ms against 14.8).
constexpr uint32_t LR_SLOT_F4 = 3u;   // a slot's float4s

__device__ __forceinline__ const float4 *slot_at(const float4 *slots, uint32_t e) { return slots + e; }

// the slab test of an inner slot's children: t[k] is child k's entry distance, 3e38 where the child is
// missed or there is none (a hit's is at most tmax, at most 1e30: misses sort last). Each plane's t is
// one fused multiply-add of its step, fma(q, s * inv, (corner - o) * inv) (a culling test on boxes that
// hold the children's: its last bit decides no hit). The step s * inv has the sign of inv (s > 0), and
// a fused multiply-add is monotone in q, so along an axis whose inv is negative the high plane is the
// near one: each axis's near and far planes are picked once a node.
__device__ __forceinline__ void wide_test(float4 r0, float4 r1, float4 r2, V3 o, V3 inv, float tmin, float tmax, float t[4])
{
    const uint32_t w = __float_as_uint(r0.w);
    const float ax = ldexpf(inv.x, (int)(w << 24) >> 24), ay = ldexpf(inv.y, (int)(w << 16) >> 24);
    const float az = ldexpf(inv.z, (int)(w << 8) >> 24);
    const float bx = __builtin_fmaf(r0.x, inv.x, -(o.x * inv.x)), by = __builtin_fmaf(r0.y, inv.y, -(o.y * inv.y));
    const float bz = __builtin_fmaf(r0.z, inv.z, -(o.z * inv.z));
    const uint32_t lx = __float_as_uint(r1.x), ly = __float_as_uint(r1.y), lz = __float_as_uint(r1.z);
    const uint32_t hx = __float_as_uint(r2.x), hy = __float_as_uint(r2.y), hz = __float_as_uint(r2.z);
    const bool fx = inv.x < 0.0f, fy = inv.y < 0.0f, fz = inv.z < 0.0f;   // (flipped: high plane near)
    const uint32_t nx = fx ? hx : lx, ny = fy ? hy : ly, nz = fz ? hz : lz;
    const uint32_t gx = fx ? lx : hx, gy = fy ? ly : hy, gz = fz ? lz : hz;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int sh = 8 * k;
        const float t0x = __builtin_fmaf((float)((nx >> sh) & 0xffu), ax, bx);
        const float t0y = __builtin_fmaf((float)((ny >> sh) & 0xffu), ay, by);
        const float t0z = __builtin_fmaf((float)((nz >> sh) & 0xffu), az, bz);
        const float t1x = __builtin_fmaf((float)((gx >> sh) & 0xffu), ax, bx);
        const float t1y = __builtin_fmaf((float)((gy >> sh) & 0xffu), ay, by);
        const float t1z = __builtin_fmaf((float)((gz >> sh) & 0xffu), az, bz);
        const float enter = fmaxf(fmaxf(t0x, t0y), fmaxf(t0z, tmin));
        const float leave = fminf(fminf(t1x, t1y), fminf(t1z, tmax));
        const bool none = k >= 2 && w < ((uint32_t)(k + 1) << 24);   // (a node has at least two children)
        t[k] = none || leave < enter ? 3e38f : enter;
        // one child after the other: interleaving the four holds all 24 planes at once
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The children's order: a sorting network of five exchanges, each only of a smaller distance for a larger
// one. Equal distances stay where they are (which of them is visited first decides between shapes hit
// at one distance), and so the order is not the places' where exchanges moved others past them.
__device__ __forceinline__ void order_(float &ta, uint32_t &pa, float &tb, uint32_t &pb)
{
    const bool s = tb < ta;
    const float t = s ? tb : ta;
    const uint32_t p = s ? pb : pa;
    tb = s ? ta : tb;
    pb = s ? pa : pb;
    ta = t;
    pa = p;
}

// The first four exchanges by keys of 64 bits, a distance's bits above its place's: as doubles they order as
// the distances do (from +0 up: every pattern is a finite double), and equal distances by their places,
// which is to stay where they are: up to there the first of two positions holds the lower place. The
// last exchange compares the distances. Two instructions an exchange instead of five; the order is
// the same to the bit. For rays whose tmin is from +0 up (then so is every entry): keys_ok. A 54M-path
// queue 49.4 -> 48.5 ms, a 1280 x 720 x 8 still 8.18 -> 7.97, 300,000 scene rays 165 -> 158 us.
__device__ __forceinline__ double key_(float t, uint32_t p) { return __hiloint2double(__float_as_int(t), (int)p); }
__device__ __forceinline__ void order_keys_(double &a, double &b)
{
    double lo, hi;
    asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
    asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    a = lo;
    b = hi;
}
// The children hit, nearest first: the farther ones stacked (farthest first), the nearest the next
// entry; false when none was hit. While three more entries fit in LDS each is written at the top
// whether it is one or not, and the top moves past it if it is.
template <int STK, bool KEYS>
__device__ __forceinline__ bool wide_next(float t[4], uint32_t base, const WalkStack &S, int &sp, uint32_t &cur,
                                          uint32_t *overflow)
{
    uint32_t p[4] = {0u, LR_SLOT_F4, 2u * LR_SLOT_F4, 3u * LR_SLOT_F4};
    if constexpr (KEYS) {
        double k[4] = {key_(t[0], p[0]), key_(t[1], p[1]), key_(t[2], p[2]), key_(t[3], p[3])};
        order_keys_(k[0], k[1]);
        order_keys_(k[2], k[3]);
        order_keys_(k[0], k[2]);
        order_keys_(k[1], k[3]);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            t[q] = __int_as_float(__double2hiint(k[q]));
            p[q] = (uint32_t)__double2loint(k[q]);
        }
    } else {
        order_(t[0], p[0], t[1], p[1]);
        order_(t[2], p[2], t[3], p[3]);
        order_(t[0], p[0], t[2], p[2]);
        order_(t[1], p[1], t[3], p[3]);
    }
    order_(t[1], p[1], t[2], p[2]);
    if (sp + 3 <= STK) {
#pragma unroll
        for (int k = 3; k >= 1; k--) {
            S.stk[sp * S.stride] = base + p[k];
            sp += t[k] < 3e38f ? 1 : 0;
        }
    } else {
#pragma unroll
        for (int k = 3; k >= 1; k--) {
            if (!(t[k] < 3e38f)) continue;
            if (sp >= S.cap) {   // cannot happen with a correct depth: said, never silently dropped
                atomicOr(overflow, 1u);
                return false;
            }
            const uint32_t x = base + p[k];
            if (sp < STK) S.stk[sp * S.stride] = x;
            else S.spill[(size_t)(sp - STK) * S.sstride] = x;
            sp++;
        }
    }
    cur = base + p[0];
    return t[0] < 3e38f;
}

// One step: the entry's slot loaded, an inner node's children tested (those hit stacked farthest
// first) or a leaf's shape; leaves and nodes are thus visited near to far. Lanes at leaves and at
// nodes take their steps in one pass of the loop. False when the walk has ended.
template <bool ANY, bool COUNT, int STK, bool KEYS>
__device__ __forceinline__ bool walk4_step(const float4 *__restrict__ slots, const float4 *__restrict__ prims, uint32_t nprims, V3 o,
                                           V3 d, V3 inv, float tmin, WalkHit &best, int &sp, uint32_t &cur, const WalkStack &S,
                                           uint32_t *overflow, WalkCnt &c)
{
    const float4 *p = slot_at(slots, cur);
    const float4 r0 = ldg4(p, 0), r1 = ldg4(p, 1), r2 = ldg4(p, 2);
    bool more;   // the next entry is in cur (else: the stack's)
    if (__float_as_uint(r0.w) & LR_LEAF) {
        const uint32_t sid = __float_as_uint(r1.w);
        if (COUNT) count_shape(c);
        float t, u = 0.0f, v = 0.0f;
        bool hit;
        if (sid < nprims) {
            t = hit_prim(prims, sid, o, d, tmin, best.t, u, v);
            hit = t > 0.0f;
        } else hit = hit_tri(r0, r1, r2, o, d, tmin, best.t, t, u, v);
        if (hit) {
            best = WalkHit{t, sid, u, v};
            if (ANY) return false;
        }
        more = false;
    } else {
        if (COUNT) {
            count_node(c);
            count_uniform(c, slots, cur);
        }
        float t[4];
        wide_test(r0, r1, r2, o, inv, tmin, best.t, t);
        more = wide_next<STK, KEYS>(t, __float_as_uint(r1.w), S, sp, cur, overflow);
    }
    if (!more) {
        if (sp == 0) return false;
        sp--;
        cur = stk_get<STK>(S, sp);
    }
    return true;
}

template <bool ANY, bool COUNT, int STK, bool KEYS = false>
__device__ __forceinline__ WalkHit walk4(const float4 *__restrict__ slots, const float4 *__restrict__ prims, uint32_t nprims, V3 o,
                                         V3 d, float tmin, float tmax, const WalkStack &S, uint32_t *overflow, WalkCnt &c)
{
    const V3 inv = v3(safe_inv(d.x), safe_inv(d.y), safe_inv(d.z));
    WalkHit best{tmax, LR_NONE, 0.0f, 0.0f};
    int sp = 0;
    uint32_t cur = 0u;   // the entry being visited (the root's slot first)
    while (walk4_step<ANY, COUNT, STK, KEYS>(slots, prims, nprims, o, d, inv, tmin, best, sp, cur, S, overflow, c)) {
    }
    return best;
}
