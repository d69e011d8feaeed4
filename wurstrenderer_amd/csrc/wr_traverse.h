// wr_traverse.h -- BVH4 traversal with a per-lane LDS stack and the
// watertight ray/triangle test (Woop, Benthin, Wald, JCGT 2013), FP32 with the
// paper's FP64 recomputation of the edge functions on edge hits.
//
// Semantics follow rtcIntersect1 / rtcOccluded1 as the reference calls them
// (src/accel/embreeaccel.h:336-422): double-sided triangles, hits accepted
// for t in (tmin, tmax], closest hit for extension rays, any hit for shadow
// rays.  Node boxes are tested conservatively (exit distances widened by the
// bound on the slab arithmetic's rounding error) so that no watertight hit is
// lost to rounding in the box test.
#pragma once
#include <type_traits>

#include "wr_device.h"

namespace wr {

constexpr uint32_t kInvalid = 0xFFFFFFFFu;

struct RaySetup {
    float3 o;
    float tmin;
    float ix, iy, iz;          // 1/d with zero components replaced by +-1e-20
    float nnx, nny, nnz;       // per axis -(o/d), lowered (near planes) and raised (far planes) by
    float nfx, nfy, nfz;       // 2^-22 |o/d|: a plane p is crossed at fma(p, 1/d, nn) or fma(p, 1/d, nf)
    int kz;                    // watertight test: the axis of the largest direction component
    float Sx, Sy, Sz;
    uint32_t onx, ony, onz;    // byte offsets of the near-plane rows in a Node4 (the far row is at offset ^ 16)
    uint32_t snx, sny, snz;    // byte selectors of the near planes in a NodeQ plane word (kSelLow / kSelHigh)
};

// v_perm_b32 selectors that spread two planes of a NodeQ plane word (child a's
// low, child b's low, child a's high, child b's high) into the low bytes of two
// 16-bit halves: the low planes, or the high ones.  They differ by kSelSwap.
constexpr uint32_t kSelLow = 0x0c010c00u, kSelHigh = 0x0c030c02u, kSelSwap = kSelLow ^ kSelHigh;

// (v[kz + 1], v[kz + 2], v[kz]), indices modulo 3.  Woop et al. also exchange the
// first two where the direction is negative along kz, to keep the winding; that
// only negates the edge functions, the determinant and the scaled distance
// together, and none of the tests or t depends on that sign.
__device__ __forceinline__ float3 rotate_axes(float3 v, int kz) {
    const bool k0 = kz == 0, k1 = kz == 1;
    return f3(k0 ? v.y : (k1 ? v.z : v.x), k0 ? v.z : (k1 ? v.x : v.y), k0 ? v.x : (k1 ? v.y : v.z));
}

// Reciprocals use the hardware v_rcp_f32 (about 1 ulp): box exit distances are
// widened by 4 ulp, and the watertight shear only has to be the same for every
// triangle a ray meets, not correctly rounded.
__device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// One v_min3_f32 / v_max3_f32 (fminf and fmaxf first quieten an operand of
// unknown origin); a NaN operand loses, as with fminf and fmaxf.
__device__ __forceinline__ float min3(float a, float b, float c) {
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

__device__ __forceinline__ RaySetup setup_ray(float3 o, float3 d, float tmin) {
    RaySetup r;
    r.o = o; r.tmin = tmin;
    auto safe = [](float x) { return fabsf(x) < 1e-20f ? copysignf(1e-20f, x) : x; };
    r.ix = rcp(safe(d.x)); r.iy = rcp(safe(d.y)); r.iz = rcp(safe(d.z));
    const float mx = o.x * r.ix, my = o.y * r.iy, mz = o.z * r.iz;
    const float ex = 2.38418579e-7f * fabsf(mx), ey = 2.38418579e-7f * fabsf(my), ez = 2.38418579e-7f * fabsf(mz);
    r.nnx = -mx - ex; r.nny = -my - ey; r.nnz = -mz - ez;
    r.nfx = -mx + ex; r.nfy = -my + ey; r.nfz = -mz + ez;
    // a Node4 holds rows lo_x, hi_x, lo_y, hi_y, lo_z, hi_z of 16 bytes: the near
    // plane of an axis is its lo row for a positive direction, its hi row otherwise
    r.onx = r.ix < 0.f ? 16u : 0u;
    r.ony = r.iy < 0.f ? 48u : 32u;
    r.onz = r.iz < 0.f ? 80u : 64u;
    r.snx = r.ix < 0.f ? kSelHigh : kSelLow;
    r.sny = r.iy < 0.f ? kSelHigh : kSelLow;
    r.snz = r.iz < 0.f ? kSelHigh : kSelLow;
    float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    r.kz = (ax >= ay) ? ((ax >= az) ? 0 : 2) : ((ay >= az) ? 1 : 2);
    const float3 dr = rotate_axes(d, r.kz);
    r.Sz = rcp(dr.z);
    r.Sx = dr.x * r.Sz; r.Sy = dr.y * r.Sz;
    return r;
}

// Watertight FP32 test; returns true and t for a hit in (tmin, tmax].
__device__ __forceinline__ bool tri_test(const RaySetup &r, float4 va, float4 vb, float4 vc, float tmax, float &t_out) {
    const float3 A = rotate_axes(xyz(va) - r.o, r.kz), B = rotate_axes(xyz(vb) - r.o, r.kz),
                 C = rotate_axes(xyz(vc) - r.o, r.kz);
    const float Akz = A.z, Bkz = B.z, Ckz = C.z;
    const float Ax = fmaf(-r.Sx, Akz, A.x), Ay = fmaf(-r.Sy, Akz, A.y);
    const float Bx = fmaf(-r.Sx, Bkz, B.x), By = fmaf(-r.Sy, Bkz, B.y);
    const float Cx = fmaf(-r.Sx, Ckz, C.x), Cy = fmaf(-r.Sy, Ckz, C.y);
    float U, V, W;
    {
        // The per-vertex projections above may fuse (a vertex then projects to
        // the same value in every triangle that holds it), but the edge
        // functions must not: Cx*By - Cy*Bx with one product fused is not the
        // exact negation of the same edge's value in the neighbouring triangle,
        // Bx*Cy - By*Cx, and a ray through the shared edge could miss both.
#pragma clang fp contract(off)
        U = Cx * By - Cy * Bx;
        V = Ax * Cy - Ay * Cx;
        W = Bx * Ay - By * Ax;
    }
    if (min3(fabsf(U), fabsf(V), fabsf(W)) == 0.f) {
        // An edge function rounded to zero: recompute the three in FP64 from the
        // same projected coordinates (Woop et al., section 3.3).  A product of
        // two floats is exact in FP64, so each difference has the exact sign,
        // and a shared edge still gives its two triangles opposite values.
        double Ud, Vd, Wd;
        {
#pragma clang fp contract(off)
            Ud = double(Cx) * double(By) - double(Cy) * double(Bx);
            Vd = double(Ax) * double(Cy) - double(Ay) * double(Cx);
            Wd = double(Bx) * double(Ay) - double(By) * double(Ax);
        }
        if ((Ud < 0.0 || Vd < 0.0 || Wd < 0.0) && (Ud > 0.0 || Vd > 0.0 || Wd > 0.0)) return false;
        U = float(Ud);
        V = float(Vd);
        W = float(Wd);
    } else if (min3(U, V, W) < 0.f && max3(U, V, W) > 0.f) {
        return false;
    }
    const float det = U + V + W;
    if (det == 0.f) return false;
    const float T = r.Sz * (U * Akz + V * Bkz + W * Ckz);
    const float t = T * rcp(det);
    if (!(t > r.tmin && t <= tmax)) return false;
    t_out = t;
    return true;
}

// Far limit against which a closest-hit traversal culls boxes and stack
// entries: the best t so far widened by 2^-21 (4 ulp).  A triangle that ties
// with the best hit in t may sit in a box whose FP32 entry distance rounds a
// few ulp above that t; culling such a box would make the equal-t rule (lower
// leaf-order index wins) depend on the order in which leaves are reached.
__device__ __forceinline__ float cull_limit(float t) { return fmaf(fabsf(t), 4.76837158e-7f, t); }

// Per-lane traversal stack.  Closest hit keeps 64-bit entries (node ref in
// the low half, entry distance bits in the high half), any hit node refs only.
// Slot k of a lane lives in LDS at [k * kBlock + lane] for k < kLdsSlots
// (bank-conflict free, one 64-bit or 32-bit access per push and pop); deeper
// slots spill to the block's slice of a global region, at
// [(k - kLdsSlots) * kBlock + lane].  Slot 0 holds the end mark, an entry that
// every pop accepts, so a pop needs no test for an empty stack.  `top` is the
// LDS address of the next free slot and simply runs on past the LDS slots.
// A SIMD issues about one instruction per 2.4 clocks whatever its kind, and a
// node step used to spend half of them on branches and exec-mask updates.  So
// pushes and pops test once per wave whether any lane is near the end of its
// LDS slots (10 slots: one node step in three on the 1.31M-triangle frame),
// and only such waves run the code that looks at each lane's depth.  The BVH
// builder guarantees at most kStackDepth live entries.
typedef __attribute__((address_space(1))) uint64_t GlobalU64;
// Node refs: inner nodes 0 .. 2^31 - 1; leaves kLeafBit | (count - 1) << 28 |
// first with count <= 4, so 0x80000000 .. 0xBFFFFFFF; above that, marks.
constexpr uint32_t kEndRef = 0xFFFFFFFFu;   // the stack's end mark; cur of a lane that is done
constexpr uint32_t kPopRef = 0xFFFFFFFEu;   // cur of a lane that takes its next node from the stack
__device__ __forceinline__ bool is_inner(uint32_t ref) { return int32_t(ref) >= 0; }
__device__ __forceinline__ bool is_leaf(uint32_t ref) { return int32_t(ref) < int32_t(0xC0000000u); }
static_assert(kMaxLeafTris <= 4, "leaf refs stay below the marks");
__device__ __forceinline__ bool wave_any(bool p) { return __builtin_amdgcn_ballot_w64(p) != 0; }

// A closest-hit entry: node ref, entry distance bits.
typedef uint32_t StackEntry __attribute__((ext_vector_type(2)));
__device__ __forceinline__ StackEntry stack_entry(uint32_t ref, uint32_t tn_bits) { return StackEntry{ref, tn_bits}; }

template <int kBlock, bool ANY>
struct LaneStack {
    typedef typename std::conditional<ANY, uint32_t, StackEntry>::type Entry;
    typedef __attribute__((address_space(3))) Entry Lds;
    typedef __attribute__((address_space(1))) Entry Global;
    static constexpr int kSlots = ANY ? 2 * kLdsSlots : kLdsSlots;  // the same LDS bytes
    Lds *base;          // slot 0 of this lane
    Lds *top;           // next free slot
    GlobalU64 *spill;   // this block's spill slice (kSpillDepth * kBlock entries)
    // lds: kLdsSlots * kBlock 64-bit words; spill_region: kSpillDepth * kBlock entries per block of the grid
    __device__ __forceinline__ LaneStack(uint64_t *lds, uint2 *spill_region)
        : base((Lds *)lds + __lane_id()), top(base),
          spill((GlobalU64 *)spill_region + size_t(blockIdx.x) * (kSpillDepth * kBlock)) {}
    // an empty stack
    __device__ __forceinline__ void reset() {
        if constexpr (ANY) *base = kEndRef;
        else *base = stack_entry(kEndRef, 0xFF800000u);  // distance -inf
        top = base + kBlock;
    }
    __device__ __forceinline__ bool beyond(const Lds *p, int slots) const { return p > base + slots * kBlock; }
    __device__ __forceinline__ Global *deep(const Lds *p) const {
        return (Global *)(spill + (uint32_t(p - base) / kBlock - kSlots) * kBlock + __lane_id());
    }
    __device__ __forceinline__ Entry load(const Lds *p) const { return beyond(p, kSlots - 1) ? *deep(p) : *p; }
    __device__ __forceinline__ void store(Lds *p, Entry e) {
        if (beyond(p, kSlots - 1)) *deep(p) = e;
        else *p = e;
    }
    // pushes a if pa, then b if pb, then c if pc
    __device__ __forceinline__ void push3(Entry a, bool pa, Entry b, bool pb, Entry c, bool pc) {
        if (!wave_any(beyond(top, kSlots - 3))) {
            // every lane has three slots left: store all, keep those that count
            *top = a;
            top += pa ? kBlock : 0;
            *top = b;
            top += pb ? kBlock : 0;
            *top = c;
            top += pc ? kBlock : 0;
        } else {
            if (pa) { store(top, a); top += kBlock; }
            if (pb) { store(top, b); top += kBlock; }
            if (pc) { store(top, c); top += kBlock; }
        }
    }
};

// Entry and exit distances of the ray through the four child boxes of inner
// node `cur`, and the child refs.  The node is a NodeQ: four 16-byte loads.
// Plane q of an axis lies at origin + q * spacing, at or outside the child's
// exact plane (k_quantize_nodes), so the ray crosses it at
//   t = (origin - o) / d + q * spacing / d = b + q * g,
// one fused multiply-add per plane: v_perm_b32 spreads two planes of a word
// into two 16-bit halves, which read as half-precision denormals q * 2^-24,
// and v_fma_mix_f32 takes them as they are (the node stores spacing * 2^24).
//
// Errors: b (one subtraction, one product, v_rcp_f32) is off by less than
// 2^-22 |b|, a computed plane by less than 2^-21 (|b| + 255 |g|), and the
// watertight test places a hit along the axis to about 2^-22 of the same sum.
// b is therefore lowered for near planes and raised for far planes by
// 2^-20 (|b| + 255 |g|), so a box the ray touches always has entry <= exit.
// Where g or the stored spacing overflows, that margin is infinite and every
// plane of the axis becomes -inf / +inf or NaN, which max and min pass over: the
// axis culls nothing, and an exit that is NaN, on all three axes, does not
// either.  An empty slot is rejected by its ref (kEmptyChild).
// Returns the refs; tn holds the entry distances and hit[i] marks the
// children whose box is entered before `far_limit`.
//
// Measured with the branchless pushes and the FP64 sort (sort_push), all hits
// unchanged: instructions per wave and node step, everything included, 350 ->
// about 290; 1.31M-triangle frame 48.3 -> 46.6 ms, gap room at 961 x 541 and
// 24 spp 49.9 -> 47.4 ms.  What bounds it now is the L1, which serves a lane's
// four 16-byte rows as four requests (0.78 accesses per clock and CU, stalled
// on pending misses and tag conflicts for another 38% of the time).  Letting
// the four lanes of a quad fetch each other's nodes as 64-byte requests halves
// the accesses, but the transpose through LDS leaves room for 4 to 5 waves per
// SIMD, too few to cover the misses: 53 ms and 56 ms.
typedef _Float16 Half2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint4 node_test(uint4 r0, uint4 r1, uint4 r2, uint4 r3, const RaySetup &r, float far_limit,
                                           float tn[4], bool hit[4]) {
    const uint4 ch = make_uint4(r2.x, r2.z, r3.x, r3.z);
    const uint32_t c[4] = {ch.x, ch.y, ch.z, ch.w};
    float n[3][4], f[3][4];
    auto axis = [&](int k, uint32_t org, uint32_t scale, float o, float inv, uint32_t w01, uint32_t w23, uint32_t sel) {
        constexpr float kMargin = 0x1p-20f;
        const float b = (__uint_as_float(org) - o) * inv, g = __uint_as_float(scale) * inv;
        const float m = fmaf(fabsf(g), 255.f * 0x1p-24f, fabsf(b));
        const float bn = fmaf(m, -kMargin, b), bf = fmaf(m, kMargin, b);
        const uint32_t far_sel = sel ^ kSelSwap;
        auto two = [&](uint32_t w, uint32_t s) { return __builtin_bit_cast(Half2, __builtin_amdgcn_perm(w, w, s)); };
        const Half2 n01 = two(w01, sel), n23 = two(w23, sel), f01 = two(w01, far_sel), f23 = two(w23, far_sel);
        n[k][0] = fmaf(float(n01.x), g, bn);
        n[k][1] = fmaf(float(n01.y), g, bn);
        n[k][2] = fmaf(float(n23.x), g, bn);
        n[k][3] = fmaf(float(n23.y), g, bn);
        f[k][0] = fmaf(float(f01.x), g, bf);
        f[k][1] = fmaf(float(f01.y), g, bf);
        f[k][2] = fmaf(float(f23.x), g, bf);
        f[k][3] = fmaf(float(f23.y), g, bf);
    };
    axis(0, r0.x, r0.w, r.o.x, r.ix, r1.x, r1.y, r.snx);
    axis(1, r0.y, r3.y, r.o.y, r.iy, r1.z, r1.w, r.sny);
    axis(2, r0.z, r3.w, r.o.z, r.iz, r2.y, r2.w, r.snz);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        tn[i] = max3(n[0][i], n[1][i], fmaxf(n[2][i], r.tmin));
        hit[i] = (c[i] != kEmptyChild) & !(tn[i] > min3(f[0][i], f[1][i], f[2][i])) & (tn[i] <= far_limit);
    }
    return ch;
}

__device__ __forceinline__ uint4 node_test(const NodeQ *nodes, const RaySetup &r, uint32_t cur, float far_limit,
                                           float tn[4], bool hit[4]) {
    uint32_t stride = sizeof(NodeQ);
    asm("" : "+s"(stride));  // one 64-bit multiply-add instead of a shift and an add
    const uint4 *nb = reinterpret_cast<const uint4 *>(reinterpret_cast<const char *>(nodes) + uint64_t(cur) * stride);
    return node_test(nb[0], nb[1], nb[2], nb[3], r, far_limit, tn, hit);
}

// The same test on a full-precision Node4: seven loads (the near and far rows
// at the ray's per-axis byte offsets, and the refs), no decoding.  The kernels
// that trace one coherent or register-heavy path per lane (k_visualize,
// k_bdpt) use it, since their traversal is not bound by load requests.  Empty
// slots hold inverted boxes (lo = FLT_MAX, hi = -FLT_MAX), which fail the test.
__device__ __forceinline__ uint4 node_test(const Node4 *nodes, const RaySetup &r, uint32_t cur, float far_limit,
                                           float tn[4], bool hit[4]) {
    const char *nb = reinterpret_cast<const char *>(nodes);
    const uint32_t base = cur * uint32_t(sizeof(Node4));
    auto row = [&](uint32_t off) { return *reinterpret_cast<const float4 *>(nb + (base + off)); };
    const float4 nx_ = row(r.onx), fx_ = row(r.onx ^ 16u);
    const float4 ny_ = row(r.ony), fy_ = row(r.ony ^ 16u);
    const float4 nz_ = row(r.onz), fz_ = row(r.onz ^ 16u);
    const uint4 ch = *reinterpret_cast<const uint4 *>(nb + (base + 96u));
    const float nx[4] = {nx_.x, nx_.y, nx_.z, nx_.w}, fx[4] = {fx_.x, fx_.y, fx_.z, fx_.w};
    const float ny[4] = {ny_.x, ny_.y, ny_.z, ny_.w}, fy[4] = {fy_.x, fy_.y, fy_.z, fy_.w};
    const float nz[4] = {nz_.x, nz_.y, nz_.z, nz_.w}, fz[4] = {fz_.x, fz_.y, fz_.z, fz_.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        tn[i] = fmaxf(fmaxf(fmaf(nx[i], r.ix, r.nnx), fmaf(ny[i], r.iy, r.nny)), fmaxf(fmaf(nz[i], r.iz, r.nnz), r.tmin));
        const float tf = fminf(fminf(fmaf(fx[i], r.ix, r.nfx), fmaf(fy[i], r.iy, r.nfy)), fmaf(fz[i], r.iz, r.nfz));
        hit[i] = tn[i] <= fminf(tf * 1.00000095f, far_limit);
    }
    return ch;
}
template <class G>
__device__ __forceinline__ uint4 node_test(const G &s, const RaySetup &r, uint32_t cur, float far_limit, float tn[4],
                                           bool hit[4]) {
    return node_test(s.nodes, r, cur, far_limit, tn, hit);
}

struct TraversalCounters {
    uint32_t nodes = 0, tris = 0;
};

// Resumable traversal state of one lane.
struct TravState {
    RaySetup r;
    float t;          // current far limit (closest hit so far, or the shadow ray's tmax)
    uint32_t hit;     // leaf-order triangle or kInvalid
    uint32_t cur;     // node reference to process next
};

__device__ __forceinline__ void trav_begin(TravState &ts, const RaySetup &r, float tmax) {
    ts.r = r;
    // A ray that is not a number gets that as its far limit, so that no box is
    // entered and it misses at the root: NaN planes alone cull nothing and would
    // take it through the whole tree.
    ts.t = fmaf(r.ix, 0.f, fmaf(r.iy, 0.f, fmaf(r.iz, 0.f, fmaf(r.o.x, 0.f, fmaf(r.o.y, 0.f, fmaf(r.o.z, 0.f, tmax))))));
    ts.hit = kInvalid;
    ts.cur = 0;  // root (internal node 0)
}

// Orders the children near to far, pushes the entered ones but the nearest,
// farthest first, and returns the nearest (kPopRef if none is entered).  A
// key is the 64-bit stack entry (child ref low, entry distance bits high), its
// high word kNoEntry for a child whose box is not entered.  Read as doubles,
// keys order by their high words (an FP32 pattern up to infinity is the high
// word of a finite double), so a comparator is one v_min_f64 and one
// v_max_f64, which pass the winner's 64 bits on unchanged: two operations
// where a compare and four selects took five.  A push is one 64-bit LDS store.
constexpr uint32_t kNoEntry = 0x7FE00000u;  // above the bits of +inf, below those of a double infinity
template <int kBlock>
__device__ __forceinline__ uint32_t sort_push(StackEntry key[4], LaneStack<kBlock, false> &st) {
    auto cswap = [&](int a, int b) {
        StackEntry lo, hi;
        asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(key[a]), "v"(key[b]));
        asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(key[a]), "v"(key[b]));
        key[a] = lo;
        key[b] = hi;
    };
    cswap(0, 1); cswap(2, 3); cswap(0, 2); cswap(1, 3); cswap(1, 2);
    // the entered children are now a prefix of the four
    auto entered = [](StackEntry k) { return k.y != kNoEntry; };
    st.push3(key[3], entered(key[3]), key[2], entered(key[2]), key[1], entered(key[1]));
    return entered(key[0]) ? key[0].x : kPopRef;
}

// Closest hit, one speculative while-while round (Aila and Laine, "Understanding
// the Efficiency of Ray Traversal on GPUs", HPG 2009): each lane descends inner
// nodes and postpones the first leaf it meets, continuing speculatively with
// the next node, until no lane of the wave has an inner node to visit (or
// kSpecSteps steps have run); then the wave tests its postponed leaves
// together, so the box-test and triangle-test code each run with dense lanes.
// A lane whose cur is a leaf while one is postponed waits; a lane that is done
// or has no ray has cur = kEndRef and takes part in nothing.  All lanes of the
// wave must call it (it takes ballots).  The lane's ray is finished when cur
// is kEndRef on return.
#ifndef WR_SPEC_STEPS
#define WR_SPEC_STEPS 4
#endif
constexpr int kSpecSteps = WR_SPEC_STEPS;

// The next node of a lane whose cur is kPopRef, or a leaf it may postpone:
// pops until an entry is near enough and is not a leaf to postpone.
template <int kBlock>
__device__ __forceinline__ void next_node(TravState &ts, uint32_t &leaf, LaneStack<kBlock, false> &st) {
    auto take = [&]() {  // postpones cur if it is a leaf and none waits
        if (is_leaf(ts.cur) && leaf == kInvalid) {
            leaf = ts.cur;
            ts.cur = kPopRef;
        }
    };
    take();
    if (ts.cur == kPopRef) {
        const float lim = cull_limit(ts.t);
        auto pop = [&](bool deep) {
            do {
                st.top -= kBlock;
                const StackEntry e = deep ? st.load(st.top) : *st.top;
                if (!(__uint_as_float(e.y) > lim)) {
                    ts.cur = e.x;
                    take();
                }
            } while (ts.cur == kPopRef);
        };
        if (!wave_any(st.beyond(st.top, st.kSlots))) pop(false);
        else pop(true);
    }
}
template <bool COUNT, int kBlock, class G>
__device__ __forceinline__ void trav_round(const G &s, TravState &ts, LaneStack<kBlock, false> &st, TraversalCounters &cnt) {
    const RaySetup &r = ts.r;
    uint32_t leaf = kInvalid;  // postponed leaf
    if (is_leaf(ts.cur)) next_node(ts, leaf, st);  // one that waited for the last round's
    for (int it = 0; it < kSpecSteps; it++) {
        const bool inner = is_inner(ts.cur);
        if (!wave_any(inner)) break;
        if (inner) {
            float tn[4];
            bool h[4];
            const uint4 ch = node_test(s, r, ts.cur, cull_limit(ts.t), tn, h);
            if (COUNT) cnt.nodes++;
            StackEntry key[4] = {stack_entry(ch.x, h[0] ? __float_as_uint(tn[0]) : kNoEntry),
                               stack_entry(ch.y, h[1] ? __float_as_uint(tn[1]) : kNoEntry),
                               stack_entry(ch.z, h[2] ? __float_as_uint(tn[2]) : kNoEntry),
                               stack_entry(ch.w, h[3] ? __float_as_uint(tn[3]) : kNoEntry)};
            ts.cur = sort_push(key, st);
            next_node(ts, leaf, st);
        }
    }
    if (leaf != kInvalid) {
        const uint32_t first = leaf & 0x0FFFFFFFu;
        const uint32_t count = ((leaf >> 28) & 0x7u) + 1u;
        if (COUNT) cnt.tris += count;
        for (uint32_t k = 0; k < count; k++) {
            const float4 *tp = s.tris + 3 * size_t(first + k);
            float t;
            if (tri_test(r, tp[0], tp[1], tp[2], ts.t, t) && (t < ts.t || first + k < ts.hit)) {  // ties: lower index
                ts.t = t;
                ts.hit = first + k;
            }
        }
    }
}

// Any hit, the same round: children in slot order (no sort), a stack of node
// refs only, and the postponed leaf ends the ray at its first hit.
template <int kBlock>
__device__ __forceinline__ void next_node_any(TravState &ts, uint32_t &leaf, LaneStack<kBlock, true> &st) {
    auto take = [&]() {
        if (is_leaf(ts.cur) && leaf == kInvalid) {
            leaf = ts.cur;
            ts.cur = kPopRef;
        }
    };
    take();
    if (ts.cur == kPopRef) {
        auto pop = [&](bool deep) {
            do {
                st.top -= kBlock;
                ts.cur = deep ? st.load(st.top) : *st.top;
                take();
            } while (ts.cur == kPopRef);
        };
        if (!wave_any(st.beyond(st.top, st.kSlots))) pop(false);
        else pop(true);
    }
}
template <bool COUNT, int kBlock, class G>
__device__ __forceinline__ void trav_round_any(const G &s, TravState &ts, LaneStack<kBlock, true> &st, TraversalCounters &cnt) {
    const RaySetup &r = ts.r;
    uint32_t leaf = kInvalid;
    if (is_leaf(ts.cur)) next_node_any(ts, leaf, st);
    for (int it = 0; it < kSpecSteps; it++) {
        const bool inner = is_inner(ts.cur);
        if (!wave_any(inner)) break;
        if (inner) {
            float tn[4];
            bool h[4];
            const uint4 ch = node_test(s, r, ts.cur, cull_limit(ts.t), tn, h);
            if (COUNT) cnt.nodes++;
            st.push3(ch.w, h[3], ch.z, h[2], ch.y, h[1]);
            ts.cur = h[0] ? ch.x : kPopRef;
            next_node_any(ts, leaf, st);
        }
    }
    if (leaf != kInvalid) {
        const uint32_t first = leaf & 0x0FFFFFFFu;
        const uint32_t count = ((leaf >> 28) & 0x7u) + 1u;
        if (COUNT) cnt.tris += count;
        for (uint32_t k = 0; k < count; k++) {
            const float4 *tp = s.tris + 3 * size_t(first + k);
            float t;
            if (tri_test(r, tp[0], tp[1], tp[2], ts.t, t)) {
                ts.t = t;
                ts.hit = first + k;
                ts.cur = kEndRef;  // occluded: finished
                break;
            }
        }
    }
}

// Whole traversal of one ray in speculative rounds (trav_round / trav_round_any):
// ties in t go to the lower leaf-order index.  The rounds' ballots count the lanes that are active, so lanes of a
// wave may enter and leave it at different times.
template <bool ANY, int kBlock, class G>
__device__ __forceinline__ uint32_t traverse_rounds(const G &s, const RaySetup &r, float &t_best, uint64_t *lds, uint2 *spill,
                                                    TraversalCounters &cnt) {
    LaneStack<kBlock, ANY> st(lds, spill);
    TravState ts;
    trav_begin(ts, r, t_best);
    st.reset();
    do {
        if constexpr (ANY) trav_round_any<false, kBlock>(s, ts, st, cnt);
        else trav_round<false, kBlock>(s, ts, st, cnt);
    } while (ts.cur != kEndRef);
    t_best = ts.t;
    return ts.hit;
}

}  // namespace wr
