// wr_render.hip -- wavefront NEE + MIS path tracer for gfx950 and the C-ABI.
//
// Reference: PathNeeRenderer (src/renderer/pathnextevent.h:15-196) and the
// random walk of GeneralSubpathSampler (src/pathsampler/generalsubpathsampler.h:13-160).
// The reference's recursive per-sample loop over tiles becomes a wavefront
// over a fixed pool of paths, one iteration per path vertex:
//
//   regen     start the next unclaimed samples behind the continuing paths:
//             light vertex, camera ray, light->camera (t = 1) connection
//   trace     closest hit for every active path, and any hit for the NEE and
//             t = 1 rays of the iteration before; visible ones add their
//             contribution (quantised BVH4 traversal)
//   shade     emitter hit with MIS, NEE with MIS, BSDF sample; continuing paths
//             are compacted into the next state, a finished path stores its
//             radiance under its sample index; the last block to finish ends
//             the iteration (the next state becomes current)
//   (per pass) accumulate: per-pixel FP64 sums of the samples' radiance
//
// Refilling the pool as paths end keeps every kernel's queue full until the
// last samples drain.  Path state is stored in queue order, so every kernel
// reads and writes it contiguously; compaction is one atomic per block of up to
// 512 threads.  Every kernel reads its work count from device memory, and the
// host follows a pass through a pinned progress word that the device writes.
// Small passes take one kernel from start to end instead (k_small_pass).
// Radiance is gathered in FP32 per path and summed per pixel in FP64 in sample
// order (reproducible); t = 1 splats go to the FP64 splat film with atomics.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/wurst_amd.h"
#include "wr_device.h"
#include "wr_layout.h"
#include "wr_traverse.h"
#include "wr_guide.h"

using namespace wr;

#include "wr_host.h"

// Path state, hits and shadow rays are gigabytes that one kernel writes and the
// next reads once: non-temporal accesses keep them from displacing the scene in
// the caches.  1.31M-triangle frame 44.5 -> 44.1 ms, gap room 46.3 -> 45.7 ms,
// fog 32.8 -> 32.4 ms (stores alone give two thirds of it, loads alone little).
typedef float StreamRow __attribute__((ext_vector_type(4)));
typedef uint32_t StreamPair __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float4 load_once(const float4 *p) {
    const StreamRow v = __builtin_nontemporal_load(reinterpret_cast<const StreamRow *>(p));
    return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint2 load_once(const uint2 *p) {
    const StreamPair v = __builtin_nontemporal_load(reinterpret_cast<const StreamPair *>(p));
    return make_uint2(v.x, v.y);
}
__device__ __forceinline__ void store_once(float4 *p, float4 v) {
    __builtin_nontemporal_store(StreamRow{v.x, v.y, v.z, v.w}, reinterpret_cast<StreamRow *>(p));
}
__device__ __forceinline__ void store_once(uint2 *p, uint2 v) {
    __builtin_nontemporal_store(StreamPair{v.x, v.y}, reinterpret_cast<StreamPair *>(p));
}

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

__device__ __forceinline__ uint32_t mbcnt64(unsigned long long mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// Block-aggregated append: one atomic per block of up to kShadeBlock threads.
// All threads of the block must call it (it synchronises the block).
constexpr int kShadeBlock = 512;
constexpr int kWavesPerShadeBlock = kShadeBlock / 64;
__device__ __forceinline__ uint32_t block_append(uint32_t *counter, bool pred, uint32_t *lds /* kWavesPerShadeBlock+1 */) {
    const unsigned long long mask = __ballot(pred);
    const uint32_t wave = threadIdx.x / 64;
    if (lane_id() == 0) lds[wave] = (uint32_t)__popcll(mask);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t total = 0;
        for (uint32_t w = 0; w < blockDim.x / 64; w++) {
            const uint32_t k = lds[w];
            lds[w] = total;
            total += k;
        }
        lds[kWavesPerShadeBlock] = total ? atomicAdd(counter, total) : 0u;
    }
    __syncthreads();
    const uint32_t pos = lds[kWavesPerShadeBlock] + lds[wave] + mbcnt64(mask);
    __syncthreads();  // lds is reused by the next call
    return pred ? pos : kInvalid;
}

// The shade kernels' two appends at once: continuing paths (a) and shadow rays
// (b) share one 64-bit counter, paths in the low word, so a block does one
// atomic and one round of barriers for both.  Atomics on one address are served
// one after the other, across all XCDs: with two per 256 threads they, not
// memory, set k_shade's time on the 1.31M-triangle frame (two per 128 threads:
// +83%).  `flip` alternates between calls, so that a call's LDS words are not
// overwritten before every wave has read them.
struct Append2 {
    uint32_t a, b;  // positions (valid where the predicate is)
};
__device__ __forceinline__ Append2 block_append2(uint32_t *counter, bool pa, bool pb,
                                                 uint32_t (*lds)[kWavesPerShadeBlock + 2], uint32_t flip) {
    uint32_t *l = lds[flip & 1u];
    const unsigned long long ma = __ballot(pa), mb = __ballot(pb);
    const uint32_t wave = threadIdx.x / 64;
    if (lane_id() == 0) l[wave] = (uint32_t)__popcll(ma) | (uint32_t)__popcll(mb) << 16;  // block sums stay below 2^16
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t total = 0;
        for (uint32_t w = 0; w < blockDim.x / 64; w++) {
            const uint32_t k = l[w];
            l[w] = total;
            total += k;
        }
        unsigned long long base = 0;
        if (total)
            base = atomicAdd(reinterpret_cast<unsigned long long *>(counter),
                             (unsigned long long)(total & 0xFFFFu) | (unsigned long long)(total >> 16) << 32);
        l[kWavesPerShadeBlock] = uint32_t(base);
        l[kWavesPerShadeBlock + 1] = uint32_t(base >> 32);
    }
    __syncthreads();
    const uint32_t before = l[wave];
    return {l[kWavesPerShadeBlock] + (before & 0xFFFFu) + mbcnt64(ma),
            l[kWavesPerShadeBlock + 1] + (before >> 16) + mbcnt64(mb)};
}

__device__ __forceinline__ void wave_add_stat(unsigned long long *dst, uint32_t v) {
    uint32_t s = v;
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (lane_id() == 0 && s) atomicAdd(dst, (unsigned long long)s);
}

__device__ __forceinline__ uint32_t active_count(const uint32_t *c) { return c[kQ] + c[kFresh]; }

// ============================================================== control kernels
// Number of new samples the next iteration starts: the free room of the pool
// or what is left of the pass.  Written here so regen needs no atomics.
__device__ __forceinline__ void plan_fresh(uint32_t *c, const RenderArgs &a) {
    const uint32_t head = c[kQ];
    const uint32_t left = a.total - min(c[kClaimed], a.total);
    const uint32_t fresh = min(a.capacity - head, left);
    c[kBase] = c[kClaimed];
    c[kFresh] = fresh;
    c[kClaimed] += fresh;
}
__global__ void k_init(PathBuffers pb, RenderArgs a) {
    if (threadIdx.x < kNumCounterLines) {
        pb.counters[threadIdx.x * kCounterStride] = 0u;
        pb.counters[threadIdx.x * kCounterStride + 1] = 0u;  // kQn's high word, the iterations ended
    }
    __syncthreads();
    if (threadIdx.x == 0) plan_fresh(pb.counters, a);
}
// End of an iteration: the next state becomes current, work counters restart,
// the shadow queue traced in this iteration is emptied (the one the shade
// kernel filled stays for the next traversal launch), the next refill is
// planned, and the host is told how far the pass is.  Every block of the
// iteration's last kernel calls it when it has finished; the last one to do so
// does the work (a kernel of one thread for it took 4.7 us of each iteration,
// launch gap aside).  Thread 0 did its block's appends and holds their
// results, so they are done when it takes a ticket, and no fence (which would
// write back and invalidate the XCD's L2) is needed: what the last block reads
// is either older than this kernel or read with an atomic.  The barrier keeps
// the block's other waves ahead of its ticket: each wave reads the number of
// active paths, two words that the last block rewrites, when it starts, and in a
// block without work no append's barrier follows that read.
__device__ __forceinline__ void end_iteration(const PathBuffers &pb, const RenderArgs &a) {
    __syncthreads();
    if (threadIdx.x != 0) return;
    uint32_t *c = pb.counters;
    if (atomicAdd(&c[kTicket], 1u) != gridDim.x - 1) return;
    const unsigned long long appended = atomicAdd(reinterpret_cast<unsigned long long *>(&c[kQn]), 0ull);
    const uint32_t traced = pb.next.shadow_count, shadow = uint32_t(appended >> 32);
    pb.stats[0] += active_count(c);
    pb.stats[1] += c[traced];
    c[kQ] = uint32_t(appended);
    c[pb.cur.shadow_count] = shadow;
    c[kQn] = c[kQn + 1] = 0;
    c[traced] = 0;
    c[kTicket] = 0;
    for (int x = 0; x < kXcds; x++) {
        c[kFetchExtX + x * kCounterStride] = 0;
        c[kFetchShdX + x * kCounterStride] = 0;
    }
    plan_fresh(c, a);
    const uint32_t ended = ++c[kTicket + 1];
    if (a.progress) {
        const bool drained = c[kQ] == 0 && c[kFresh] == 0 && shadow == 0;
        __hip_atomic_store(a.progress, (unsigned long long)a.tag << 32 | ended << 1 | (drained ? 1u : 0u),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}
// The traversal copy of the BVH4 (NodeQ), one node per thread.  Per axis the
// grid starts at the smallest lo of the node's children and its spacing is
// (largest hi - origin) / 255, raised by ulps until plane 255 reaches the
// largest hi.  A child's low plane is the largest q whose plane is <= its lo,
// its high plane the smallest q whose plane is >= its hi: plane 0 is the origin
// (<= every lo) and plane 255 is at or above the largest hi, so both exist and
// the planes contain the child's box.  Planes are compared in FP64 as offsets
// from the origin: q * spacing is exact there, and a plane - origin difference
// is rounded by at most 2^-53 of itself, far inside the traversal's margin.
__global__ void k_quantize_nodes(const Node4 *__restrict__ in, NodeQ *__restrict__ out, uint32_t n) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const Node4 &nd = in[k];
    const float *lo[3] = {nd.lo_x, nd.lo_y, nd.lo_z}, *hi[3] = {nd.hi_x, nd.hi_y, nd.hi_z};
    NodeQ q;
    float scale[3];
    uint32_t pl[6];
    for (int a = 0; a < 3; a++) {
        float org = FLT_MAX, top = -FLT_MAX;
        for (int c = 0; c < 4; c++)
            if (nd.child[c] != kEmptyChild) {
                org = fminf(org, lo[a][c]);
                top = fmaxf(top, hi[a][c]);
            }
        if (!(org <= top)) org = top = 0.f;  // no child
        const double ext = double(top) - double(org);
        float sc = fmaxf(float(ext / 255.0), FLT_MIN);
        while (255.0 * double(sc) < ext) sc = nextafterf(sc, INFINITY);
        uint32_t w[2] = {0u, 0u};  // children 0 and 1, 2 and 3
        for (int c = 0; c < 4; c++) {
            uint32_t ql = 255, qh = 0;  // empty slot
            if (nd.child[c] != kEmptyChild) {
                const double l = double(lo[a][c]) - double(org), h = double(hi[a][c]) - double(org), s = double(sc);
                int a0 = int(fmin(255.0, fmax(0.0, floor(l / s))));
                while (a0 > 0 && a0 * s > l) a0--;
                while (a0 < 255 && (a0 + 1) * s <= l) a0++;
                int b0 = int(fmin(255.0, fmax(0.0, ceil(h / s))));
                while (b0 < 255 && b0 * s < h) b0++;
                while (b0 > 0 && (b0 - 1) * s >= h) b0--;
                ql = uint32_t(a0);
                qh = uint32_t(b0);
            }
            w[c >> 1] |= (ql << (8 * (c & 1))) | (qh << (16 + 8 * (c & 1)));
        }
        q.org[a] = org;
        scale[a] = sc * 0x1p24f;
        pl[2 * a] = w[0];
        pl[2 * a + 1] = w[1];
    }
    q.scale_x = scale[0];
    q.scale_y = scale[1];
    q.scale_z = scale[2];
    q.x01 = pl[0]; q.x23 = pl[1]; q.y01 = pl[2]; q.y23 = pl[3]; q.z01 = pl[4]; q.z23 = pl[5];
    q.child0 = nd.child[0]; q.child1 = nd.child[1]; q.child2 = nd.child[2]; q.child3 = nd.child[3];
    out[k] = q;
}

__global__ void k_fill_u32(uint32_t *p, uint32_t v, size_t n) {
    for (size_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) p[i] = v;
}
__global__ void k_fill_f64(double *p, double *q, size_t n) {
    for (size_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) p[i] = q[i] = 0.0;
}

// ============================================================== batches
// A batch renders several (scene, film, parameters) jobs through one path pool
// and one launch of every kernel per iteration: the pass's samples are the
// jobs' samples laid end to end (job-major), a path carries its job in the
// high bits of rad.w (bounce in the low 8), and every per-path lookup reads
// the job's scene.  Single-scene kernels (BATCH = false) take the scene as a
// kernel argument instead, and their job is always 0.
struct BatchJob {
    DScene s;
    uint32_t offset;        // first pass sample of the job
    uint32_t count;         // samples of the job in this pass = k * wh
    uint32_t wh, k;         // pixels, samples per pixel in this pass
    uint32_t first_sample;  // sample index of the pass's first spp
    uint32_t seed;
    int N, use_mis;
    double *film_base, *film_splat;
};
constexpr uint32_t kBounceBits = 8;
constexpr uint32_t kBounceMask = (1u << kBounceBits) - 1;
constexpr int kMaxBatchJobs = 1 << 16;
// The job a pass sample belongs to: the last job whose offset is <= g.
__device__ __forceinline__ uint32_t find_job(const BatchJob *jobs, uint32_t n_jobs, uint32_t g) {
    uint32_t lo = 0, hi = n_jobs;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (jobs[mid].offset <= g) lo = mid; else hi = mid;
    }
    return lo;
}
// Geometry of one lane's scene for traversal.
struct Geo {
    const NodeQ *nodes;
    const float4 *tris;
};
// The same over the full-precision BVH4 (per-pixel kernels, see node_test).
struct Geo4 {
    const Node4 *nodes;
    const float4 *tris;
};

// Camera sample of path `key`: lens point and primary direction from its
// lens and pixel-jitter dimensions (lens_point_u / primary_dir_u).
__device__ __forceinline__ float3 lens_point(const DCamera &cam, uint32_t key) {
    return lens_point_u(cam, u01(key, kDimLens), u01(key, kDimLens + 1));
}
__device__ __forceinline__ float3 primary_dir(const DCamera &cam, uint32_t key, uint32_t px, uint32_t py, float3 lens,
                                              float &pdfW) {
    return primary_dir_u(cam, u01(key, kDimPixel), u01(key, kDimPixel + 1), px, py, lens, pdfW);
}

// A path vertex's outcome: the shadow ray it sends (origin and length, direction
// and target, contribution and job) and the ray that continues the path.
struct Vertex {
    float4 so = make_float4(0, 0, 0, 0), sd = so, sc = so;
    float4 o = so, d = so, thr = so;
    bool shadow = false, cont = false;
};

// ============================================================== regenerate
// Fills the pool behind the continuing paths with the next unclaimed samples:
// createLightSubpath + createCameraSubpath up to the first ray, with the t = 1
// light->camera connection (pathnextevent.h:53-99; thinlens.h:121-166), which
// PrimitivePathRenderer (a.nee == 0) does not make.  For LightSplattingRenderer
// (a.light) an entry is a light subpath instead (lightsplatting.h:58-108,
// generalsubpathsampler.h:185-268): its light vertex connects to the camera
// with weight 1, and its first ray leaves the light in a cosine-distributed
// direction (DiffuseAreaLight::sampleLe1CosByPdf, contribution 1).
template <bool ENV>
__device__ __forceinline__ void start_path(const DScene &s, const RenderArgs &a, int use_mis, uint32_t key, uint32_t px,
                                           uint32_t py, uint32_t job, Vertex &out) {
    const DCamera &cam = s.cam;
    // camera vertex (sampleWe0ByPdf)
    const float3 lens = lens_point(cam, key);
    const float3 cpos = cam_to_world(cam, lens) + f3(cam.ox, cam.oy, cam.oz);
    const float3 cz = f3(cam.zx, cam.zy, cam.zz);
    // t = 1 connection
    const LightSample l = sample_light<ENV>(s, u01(key, kDimLight), u01(key, kDimLight + 1), key);
    if (ENV && a.nee && l.env) {
        // an envmap vertex: the camera looks along its direction; G = |cos| at
        // the camera only, Le1 = 1, visibility to infinity (path.h:64-76, scene.h:98-101)
        const float3 d = l.pos;
        const float G = fabsf(dot3(cz, d));
        float rx = 0.f, ry = 0.f;
        const float we1 = G != 0.f ? camera_we1(cam, lens, d, rx, ry) : 0.f;
        if (we1 != 0.f) {
            float mis = 1.f;
            if (use_mis) {
                const float c = cam_to_local(cam, d).z;
                const float camPdfA = cam.per_pixel_norm / (c * c * c);
                mis = l.pdfA / (l.pdfA + camPdfA);
            }
            const float3 c = l.contrib * (mis * we1 * G);
            if (!is_black(c)) {
                const uint32_t target = kToSplat | (uint32_t(ry) * uint32_t(cam.W) + uint32_t(rx));
                out.so = make_float4(cpos.x, cpos.y, cpos.z, INFINITY);
                out.sd = make_float4(d.x, d.y, d.z, __uint_as_float(target));
                out.sc = make_float4(c.x, c.y, c.z, __uint_as_float(job));
                out.shadow = true;
            }
        }
    } else if (a.nee || a.light) {
        const float3 uv = cpos - l.pos;
        const float len2 = dot3(uv, uv);
        const float len = sqrtf(len2);
        const float3 nuv = uv * (1.0f / len);
        const float cos_l = dot3(l.n, nuv);
        const float G = fabsf(cos_l) * fabsf(dot3(cz, nuv)) / len2;
        if (G != 0.f && cos_l >= 0.f) {
            float rx, ry;
            const float3 wcam = -nuv;
            const float we1 = camera_we1(cam, lens, wcam, rx, ry);
            if (we1 != 0.f) {
                float mis = 1.f;
                if (use_mis) {
                    const float c = cam_to_local(cam, wcam).z;
                    float camPdfA = cam.per_pixel_norm / (c * c * c) * fabsf(cos_l) / len2;
                    if (s.med.on) camPdfA *= pass_pdf(s.med, len);
                    mis = l.pdfA / (l.pdfA + camPdfA);
                }
                const float k = mis * we1 * G * kInvPi;
                float3 c = l.contrib * k;
                if (s.med.on) c = c * transmittance(s.med, len);  // attenuated connection
                const uint32_t target = kToSplat | (uint32_t(ry) * uint32_t(cam.W) + uint32_t(rx));
                out.so = make_float4(l.pos.x, l.pos.y, l.pos.z, len - kRayEps);
                out.sd = make_float4(nuv.x, nuv.y, nuv.z, __uint_as_float(target));
                out.sc = make_float4(c.x, c.y, c.z, __uint_as_float(job));
                out.shadow = true;
            }
        }
    }
    if (a.light) {
        // the light subpath's first ray (pdf not needed: no MIS)
        const float3 dir =
            to_world(make_frame(l.n), cosine_hemisphere(u01(key, kDimPixel), u01(key, kDimPixel + 1)));
        out.o = make_float4(l.pos.x, l.pos.y, l.pos.z, 0.f);
        out.d = make_float4(dir.x, dir.y, dir.z, 0.f);
        out.thr = make_float4(l.contrib.x, l.contrib.y, l.contrib.z, 0.f);
    } else {
        // primary ray (samplePerPixelWe1CosByPdf)
        float pdfW;
        const float3 dir = primary_dir(cam, key, px, py, lens, pdfW);
        out.o = make_float4(cpos.x, cpos.y, cpos.z, 0.f);
        out.d = make_float4(dir.x, dir.y, dir.z, 0.f);
        out.thr = make_float4(1.f, 1.f, 1.f, use_mis ? pdfW : 0.f);
    }
}
template <bool BATCH, bool ENV = false>
__global__ __launch_bounds__(kShadeBlock) void k_regen(DScene s1, const BatchJob *__restrict__ jobs, uint32_t n_jobs,
                                                       PathBuffers pb, RenderArgs a) {
    __shared__ uint32_t agg[kWavesPerShadeBlock + 1];
    const uint32_t head = pb.counters[kQ];
    const uint32_t fresh_n = pb.counters[kFresh];
    const uint32_t sbase = pb.counters[kBase];
    const PathState st = pb.cur;
    for (uint32_t base = blockIdx.x * blockDim.x; base < fresh_n; base += gridDim.x * blockDim.x) {
        const uint32_t i = base + threadIdx.x;
        const bool fresh = i < fresh_n;
        const uint32_t sidx = sbase + i;
        Vertex v;
        uint32_t job = 0;
        if (fresh) {
            uint32_t local = sidx, wh = a.wh, first = a.first_sample, seed = a.seed;
            int use_mis = a.use_mis;
            if (BATCH) {
                job = find_job(jobs, n_jobs, sidx);
                const BatchJob &J = jobs[job];
                local = sidx - J.offset;
                wh = J.wh;
                first = J.first_sample;
                seed = J.seed;
                use_mis = J.use_mis;
            }
            const DScene &s = BATCH ? jobs[job].s : s1;
            const DCamera &cam = s.cam;
            const uint32_t pixel = local % wh;
            const uint32_t sample = first + local / wh;
            const uint32_t px = pixel % uint32_t(cam.W), py = pixel / uint32_t(cam.W);
            const uint32_t key = path_key(seed, pixel, sample);
            start_path<ENV>(s, a, use_mis, key, px, py, job, v);
            v.o.w = __uint_as_float(key);
            v.d.w = __uint_as_float(sidx);
        }
        if (fresh) {
            const uint32_t e = head + i;
            store_once(&st.ray_o[e], v.o);
            store_once(&st.ray_d[e], v.d);
            store_once(&st.thr[e], v.thr);
            store_once(&st.rad[e], make_float4(0.f, 0.f, 0.f, __uint_as_float(job << kBounceBits)));
            if (a.guided) st.rec[e] = 0u;
        }
        // t = 1 connections join the previous shade kernel's shadow rays
        const uint32_t si = block_append(&pb.counters[pb.next.shadow_count], v.shadow, agg);
        if (v.shadow) {
            store_once(&pb.sh_o[si], v.so);
            store_once(&pb.sh_d[si], v.sd);
            store_once(&pb.sh_c[si], v.sc);
        }
    }
}

// ============================================================== extend
// Persistent traversal: a wave claims `chunk` consecutive entries per atomic
// and refills its lanes from that local range as soon as `refill` of them are
// idle, so a wave never waits for its slowest ray and atomics stay rare.
// Waves beyond the work exit at once.  Both are runtime parameters
// (TravTune).  With the quantised nodes (traversal bound by L1 requests),
// on the 1.31M-triangle frame chunk x refill 64x16 / 96x16 / 128x16 / 192x16 /
// 256x16 gave 7,312 / 7,377 / 7,387 / 7,418 / 7,442 Mrays/s and 96x8 / 96x24 /
// 96x32 / 96x48 7,355 / 7,326 / 7,205 / 6,911; in the gap room 256x16 7,938,
// 96x16 7,862, 96x32 7,655: a wave now refills once a quarter of its lanes
// are idle.  wr_autotune searches them per workload.
#ifndef WR_REFILL_LANES
#define WR_REFILL_LANES 16
#endif
#ifndef WR_FETCH_CHUNK
#define WR_FETCH_CHUNK 256
#endif
struct TravTune {
    uint32_t chunk = WR_FETCH_CHUNK;
    uint32_t refill = WR_REFILL_LANES;
};

// Waves per SIMD of the traversal kernels.  The plain one runs 7: its registers
// then fit without spills, and with the shorter node step the L1's rate of lane
// requests binds before latency does (1.31M-triangle frame 46.5 ms at 7 waves,
// 46.7 at 8, 47.5 at 6; gap room 47.4 / 48.4 / 48.6; fog 35.7 / 35.7 / 37.2).
// The batched instance, whose lanes read different scenes, runs 8 (16 scenes
// 16.8 ms, 18.0 at 7).
#ifndef WR_EXTEND_WAVES
#define WR_EXTEND_WAVES 7
#endif
#ifndef WR_BATCH_WAVES
#define WR_BATCH_WAVES 8
#endif
#define WR_EXTEND_ATTR(W) __attribute__((amdgpu_waves_per_eu(W, W)))

struct WaveRange {
    uint32_t lo = 0, hi = 0;  // wave-uniform
    uint32_t tried = 0;       // XCD shares found empty so far (wave-uniform)
    bool fixed = false;       // the range is all this wave gets
    // A queue that leaves each block at most one chunk is dealt without
    // counters: an atomic's round trip is about a microsecond, and a wave that has
    // emptied its range asks all eight shares in turn (64 x 64 preview at 4 spp:
    // 0.384 -> 0.320 ms).
    __device__ __forceinline__ WaveRange(uint32_t n, uint32_t block) {
        if (n <= gridDim.x * kBlock) {
            lo = min(block * kBlock, n);
            hi = min(lo + kBlock, n);
            fixed = true;
        }
    }
};
// Returns the entry for this lane (>= n when it got none).  The queue's n
// entries are split into kXcds contiguous shares, share x = [n x / 8,
// n (x + 1) / 8), each with its own work counter (`xcd_counters` + x lines):
// workgroups are dispatched to the XCDs round-robin, so block b runs on XCD
// b % 8, and its waves claim chunks of that XCD's share first -- queue order
// follows pixel order, so neighbouring rays, and the nodes they read, stay in
// one XCD's L2 -- then of the other shares in turn, so no XCD idles while work
// is left.  A new chunk is claimed only when the local range is empty;
// `exhausted` (wave-uniform) is set when no share has a chunk left.  (Reading
// the eight counters at once to go straight to an open share sends all waves
// to the same one: 1080p frame 43.9 -> 45.4 ms, Cornell box 4.6 -> 5.4 ms.)
// All lanes of the wave must call it.
__device__ __forceinline__ uint32_t refill(uint32_t *xcd_counters, uint32_t n, bool idle, unsigned long long idle_mask,
                                           WaveRange &wr, bool &exhausted, uint32_t chunk) {
    if (wr.lo == wr.hi) {
        if (wr.fixed) {
            exhausted = true;
            return n;
        }
        for (;;) {
            const uint32_t x = (blockIdx.x + wr.tried) % kXcds;
            const uint32_t lo = uint32_t(uint64_t(n) * x / kXcds), hi = uint32_t(uint64_t(n) * (x + 1) / kXcds);
            uint32_t got = 0;
            if (lane_id() == 0) got = atomicAdd(&xcd_counters[x * kCounterStride], chunk);
            got = __builtin_amdgcn_readfirstlane(got);  // every lane is active here, so this reads lane 0
            if (got < hi - lo) {
                wr.lo = lo + got;
                wr.hi = min(lo + got + chunk, hi);
                break;
            }
            if (++wr.tried == kXcds) {
                exhausted = true;
                return n;
            }
        }
    }
    const uint32_t k = (uint32_t)__popcll(idle_mask);
    const uint32_t avail = wr.hi - wr.lo;
    const uint32_t r = mbcnt64(idle_mask);
    const uint32_t e = (idle && r < avail) ? wr.lo + r : n;
    wr.lo += min(k, avail);
    return e;
}

// Chunk size for a queue of n entries.  Blocks past n / kBlock exit at once,
// so a short queue (the last bounces of a frame) is worked by ceil(n / 64)
// waves: a chunk of 64 then gives every lane one ray to start at once,
// where a larger chunk leaves fewer waves with work and queues the rest of
// each chunk behind their lanes' first rays.  Long queues keep `chunk`.
__device__ __forceinline__ uint32_t spread_chunk(uint32_t n, uint32_t chunk) {
    const uint32_t per_wave = n / gridDim.x + (n % gridDim.x != 0);
    // wave-uniform; kept in a scalar register (the division runs on the VALU)
    return __builtin_amdgcn_readfirstlane(min(chunk, max(uint32_t(kBlock), per_wave)));
}

// Closest hit for the n active paths of the current state.  `st_ent` is the
// block's LDS stack (kLdsSlots x kBlock entries).
template <bool COUNT, bool BATCH>
__device__ __forceinline__ void extend_rays(DScene s1, const BatchJob *__restrict__ jobs, PathBuffers pb, uint2 *spill,
                                            TravTune tune, uint32_t n, uint64_t *st_ent) {
    const uint32_t chunk = spread_chunk(n, tune.chunk);
    LaneStack<kBlock, false> st(st_ent, spill);
    TraversalCounters cnt;
    TravState ts;
    ts.cur = kEndRef;
    uint32_t p = 0;
    WaveRange wr(n, blockIdx.x);
    Geo geo{s1.nodes, s1.tris};
    bool active = false, exhausted = false;
    for (;;) {
        const unsigned long long idle = __ballot(!active);
        if (!exhausted && __popcll(idle) >= tune.refill) {
            const uint32_t i = refill(&pb.counters[kFetchExtX], n, !active, idle, wr, exhausted, chunk);
            if (!active && i < n) {
                p = i;
                const float4 o = load_once(&pb.cur.ray_o[p]), d = load_once(&pb.cur.ray_d[p]);
                if (BATCH) {
                    const DScene &sj = jobs[__float_as_uint(pb.cur.rad[p].w) >> kBounceBits].s;
                    geo = Geo{sj.nodes, sj.tris};
                }
                trav_begin(ts, setup_ray(xyz(o), xyz(d), kRayEps), INFINITY);
                st.reset();
                active = true;
            }
        }
        if (__ballot(active) == 0) {
            if (exhausted) break;
            continue;
        }
        if (BATCH) trav_round<COUNT, kBlock>(geo, ts, st, cnt);
        else trav_round<COUNT, kBlock>(s1, ts, st, cnt);
        if (active && ts.cur == kEndRef) {
            store_once(&pb.hit[p], make_uint2(ts.hit, __float_as_uint(ts.t)));
            active = false;
        }
    }
    if (COUNT) {
        wave_add_stat(&pb.stats[2], cnt.nodes);
        wave_add_stat(&pb.stats[3], cnt.tris);
    }
}

// ============================================================== shade
// One vertex of randomWalk with the PathNeeRenderer callback
// (generalsubpathsampler.h:34-130, pathnextevent.h:100-149): the hit h of the
// ray with direction rd, the radiance and bounce in rad, and origin and
// throughput from load_o and load_thr, which are called only where they are needed.
template <bool ENV, class LoadO, class LoadThr>
__device__ __forceinline__ void shade_vertex(const DScene &s, const RenderArgs &a, int N, int use_mis, uint2 h, float3 rd,
                                             uint32_t sidx, float4 &rad, LoadO &&load_o, LoadThr &&load_thr, Vertex &out) {
    const uint32_t bounce = __float_as_uint(rad.w) & kBounceMask;
    const int cNum = int(bounce) + 2;  // camera is vertex 1
    if (ENV && h.x == kInvalid && s.env_select > 0.f) {
        // a miss is the envmap vertex (scene.h:82-88): an emitter hit with Le1 = 1,
        // Le0 = the lookup, and area pdfs equal to the solid-angle ones
        const float4 thr = load_thr();
        float mis = a.nee ? 0.f : 1.f;
        if (use_mis) {
            const float lightPdfA = s.env_select * env_pdf_dir(s, rd);
            mis = thr.w / (lightPdfA + thr.w);
        }
        const float3 c = xyz(thr) * env_eval(s, rd) * mis;
        rad.x += c.x;
        rad.y += c.y;
        rad.z += c.z;
    }
    if (h.x != kInvalid) {
        const float t = __uint_as_float(h.y);
        const float4 ray_o = load_o();
        const float3 ro = xyz(ray_o);
        const uint32_t key = __float_as_uint(ray_o.w);
        const float4 v0 = s.tris[3 * size_t(h.x) + 0];
        const float4 v1 = s.tris[3 * size_t(h.x) + 1];
        const float4 v2 = s.tris[3 * size_t(h.x) + 2];
        const float3 pos = ro + rd * t;
        const float3 ng = normalize3(cross3(xyz(v1) - xyz(v0), xyz(v2) - xyz(v0)));
        const int2 gi = s.geom_info[__float_as_uint(v1.w)];
        const float4 thr = load_thr();
        const float3 T = xyz(thr);
        if (gi.y >= 0) {
            // emitter hit: MIS against light sampling (pathnextevent.h:128-146);
            // without NEE it is the only estimate (weight 1, primitivepath.h:52-56)
            const float cos_l = -dot3(ng, rd);
            if (cos_l >= 0.f) {
                const DLight &L = s.lights[gi.y];
                float mis = a.nee ? 0.f : 1.f;
                if (use_mis) {
                    const float cPdfA = thr.w * fabsf(cos_l) / (t * t);
                    const float lightPdfA = L.pdf_select * L.inv_area;
                    mis = cPdfA / (lightPdfA + cPdfA);
                }
                rad.x += mis * T.x * L.L[0];
                rad.y += mis * T.y * L.L[1];
                rad.z += mis * T.z * L.L[2];
            }
        } else if (cNum != N) {
            const DMat m = s.mats[gi.x];
            const Frame f = make_frame(ng);
            const float3 wi = to_local(f, -rd);
            // NEE with MIS (pathnextevent.h:106-127)
            const LightSample l = sample_light<ENV>(s, u01(key, kDimLight), u01(key, kDimLight + 1), key);
            if (ENV && a.nee && l.env) {
                // toward an envmap vertex: G = |cos| at the surface, visibility to infinity
                const float3 nuv = l.pos;
                const float G = fabsf(dot3(ng, nuv));
                const float3 wo = to_local(f, nuv);
                const float3 fs = G != 0.f ? bsdf_eval(m, wi, wo) : f3(0.f, 0.f, 0.f);
                if (!is_black(fs)) {
                    const float mis = use_mis ? l.pdfA / (l.pdfA + bsdf_pdf(m, wi, wo)) : 1.f;
                    const float3 c = T * fs * l.contrib * (mis * G);
                    if (!is_black(c)) {
                        out.so = make_float4(pos.x, pos.y, pos.z, INFINITY);
                        out.sd = make_float4(nuv.x, nuv.y, nuv.z, 0.f);
                        out.sc = make_float4(c.x, c.y, c.z, 0.f);
                        out.shadow = true;
                    }
                }
            }
            const float3 uv = l.pos - pos;
            const float len2 = dot3(uv, uv);
            const float len = sqrtf(len2);
            const float3 nuv = uv * (1.0f / len);
            const float cos_lv = -dot3(l.n, nuv);
            const float G = fabsf(dot3(ng, nuv)) * fabsf(cos_lv) / len2;
            if (a.nee && !(ENV && l.env) && G != 0.f && cos_lv >= 0.f) {
                const float3 wo = to_local(f, nuv);
                const float3 fs = bsdf_eval(m, wi, wo);
                if (!is_black(fs)) {
                    float mis = 1.f;
                    if (use_mis) {
                        const float bsdfPdfA = bsdf_pdf(m, wi, wo) * fabsf(cos_lv) / len2;
                        mis = l.pdfA / (l.pdfA + bsdfPdfA);
                    }
                    const float k = mis * G * kInvPi;
                    const float3 c = T * fs * l.contrib * k;
                    if (!is_black(c)) {
                        out.so = make_float4(pos.x, pos.y, pos.z, len - kRayEps);
                        out.sd = make_float4(nuv.x, nuv.y, nuv.z, 0.f);
                        out.sc = make_float4(c.x, c.y, c.z, 0.f);
                        out.shadow = true;
                    }
                }
            }
            // BSDF sampling (generalsubpathsampler.h:81-130); here cNum < N
            const uint32_t dim = kDimBounce0 + kDimsPerBounce * bounce + kBdBsdf;
            float3 wo;
            float pdf = 0.f;
            const float3 w = bsdf_sample(m, wi, u01(key, dim), u01(key, dim + 1), wo, pdf);
            if (!is_black(w)) {
                const float3 nd = to_world(f, wo);
                out.o = make_float4(pos.x, pos.y, pos.z, __uint_as_float(key));
                out.d = make_float4(nd.x, nd.y, nd.z, __uint_as_float(sidx));
                out.thr = make_float4(w.x * T.x, w.y * T.y, w.z * T.z, use_mis ? pdf : 0.f);
                out.cont = true;
            }
        }
    }
}
// The vertices of all active paths.  Continuing paths are compacted into the
// next state; a finished path stores its radiance in its sample's slot of the pass.
template <bool BATCH, bool ENV = false>
__global__ __launch_bounds__(kShadeBlock) void k_shade(DScene s1, const BatchJob *__restrict__ jobs, PathBuffers pb,
                                                       RenderArgs a) {
    __shared__ uint32_t agg[2][kWavesPerShadeBlock + 2];
    const uint32_t n = active_count(pb.counters);
    const PathState cs = pb.cur, ns = pb.next;
    uint32_t flip = 0;
    for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += gridDim.x * blockDim.x, flip++) {
        const uint32_t i = base + threadIdx.x;
        const bool valid = i < n;
        Vertex v;
        float4 rad = make_float4(0, 0, 0, 0);
        uint32_t job = 0, sidx = 0;
        if (valid) {
            const float4 ray_d = load_once(&cs.ray_d[i]);
            const float3 rd = xyz(ray_d);
            sidx = __float_as_uint(ray_d.w);
            rad = load_once(&cs.rad[i]);
            job = __float_as_uint(rad.w) >> kBounceBits;
            const DScene &s = BATCH ? jobs[job].s : s1;
            const int N = BATCH ? jobs[job].N : a.N;
            const int use_mis = BATCH ? jobs[job].use_mis : a.use_mis;
            const uint2 h = load_once(&pb.hit[i]);
            shade_vertex<ENV>(s, a, N, use_mis, h, rd, sidx, rad, [&] { return load_once(&cs.ray_o[i]); },
                              [&] { return load_once(&cs.thr[i]); }, v);
        }
        const Append2 at = block_append2(&pb.counters[kQn], v.cont, v.shadow, agg, flip);
        const uint32_t qi = at.a, si = at.b;
        if (v.cont) {
            store_once(&ns.ray_o[qi], v.o);
            store_once(&ns.ray_d[qi], v.d);
            store_once(&ns.thr[qi], v.thr);
            rad.w = __uint_as_float(__float_as_uint(rad.w) + 1u);  // the next bounce
            store_once(&ns.rad[qi], rad);
        } else if (valid) {
            store_once(&pb.sample_rad[sidx], rad);
        }
        const uint32_t target = v.cont ? (kToNextPath | qi) : (kToSample | sidx);
        v.sd.w = __uint_as_float(target);
        v.sc.w = __uint_as_float(job);
        if (v.shadow) {
            store_once(&pb.sh_o[si], v.so);
            store_once(&pb.sh_d[si], v.sd);
            store_once(&pb.sh_c[si], v.sc);
        }
    }
    end_iteration(pb, a);
}

// ============================================================== light subpaths
// One vertex of a light subpath (LightSplattingRenderer, lightsplatting.h:91-105;
// randomWalk, generalsubpathsampler.h:34-160).  Vertex k of the subpath (the
// light vertex is 1; the first hit is bounce 0, vertex 2) exists for k <= N - 1.
// A surface vertex connects to the camera: G We1 f T with f evaluated from the
// previous vertex toward the camera, splatted at the camera raster through a
// shadow ray; then, before vertex N - 1, the BSDF samples the next direction.
// An emitter hit ends the subpath.  No medium (the reference's sampler here
// is not volumetric).
__global__ __launch_bounds__(kShadeBlock) void k_shade_light(DScene s, PathBuffers pb, RenderArgs a) {
    __shared__ uint32_t agg[2][kWavesPerShadeBlock + 2];
    const uint32_t n = active_count(pb.counters);
    const PathState cs = pb.cur, ns = pb.next;
    const DCamera &cam = s.cam;
    uint32_t flip = 0;
    for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += gridDim.x * blockDim.x, flip++) {
        const uint32_t i = base + threadIdx.x;
        bool push_shadow = false, cont = false;
        const bool valid = i < n;
        float4 so = make_float4(0, 0, 0, 0), sd = so, sc = so;
        float4 new_o = so, new_d = so, new_thr = so, rad = so;
        uint32_t sidx = 0;
        if (valid) {
            const float4 ray_d = load_once(&cs.ray_d[i]);
            sidx = __float_as_uint(ray_d.w);
            rad = load_once(&cs.rad[i]);
            const uint32_t bounce = __float_as_uint(rad.w) & kBounceMask;
            const int k = int(bounce) + 2;  // vertex of the light subpath
            const uint2 h = load_once(&pb.hit[i]);
            if (h.x != kInvalid && k <= a.N - 1) {
                const float t = __uint_as_float(h.y);
                const float4 ray_o = load_once(&cs.ray_o[i]);
                const float3 ro = xyz(ray_o), rd = xyz(ray_d);
                const float4 v0 = s.tris[3 * size_t(h.x) + 0];
                const float4 v1 = s.tris[3 * size_t(h.x) + 1];
                const float4 v2 = s.tris[3 * size_t(h.x) + 2];
                const int2 gi = s.geom_info[__float_as_uint(v1.w)];
                if (gi.y < 0) {
                    const float3 pos = ro + rd * t;
                    const float3 ng = normalize3(cross3(xyz(v1) - xyz(v0), xyz(v2) - xyz(v0)));
                    const float3 T = xyz(cs.thr[i]);
                    const uint32_t key = __float_as_uint(ray_o.w);
                    const DMat m = s.mats[gi.x];
                    const Frame f = make_frame(ng);
                    const float3 wi = to_local(f, -rd);
                    // connection to the camera vertex
                    const float3 lens = lens_point(cam, key);
                    const float3 cpos = cam_to_world(cam, lens) + f3(cam.ox, cam.oy, cam.oz);
                    const float3 uv = cpos - pos;
                    const float len2 = dot3(uv, uv);
                    const float len = sqrtf(len2);
                    const float3 nuv = uv * (1.0f / len);
                    const float G = fabsf(dot3(ng, nuv)) * fabsf(dot3(f3(cam.zx, cam.zy, cam.zz), nuv)) / len2;
                    float rx = 0.f, ry = 0.f;
                    const float we1 = G != 0.f ? camera_we1(cam, lens, -nuv, rx, ry) : 0.f;
                    if (we1 != 0.f) {
                        const float3 fs = bsdf_eval(m, wi, to_local(f, nuv));
                        const float3 c = T * fs * (G * we1);
                        if (!is_black(c)) {
                            const uint32_t target = kToSplat | (uint32_t(ry) * uint32_t(cam.W) + uint32_t(rx));
                            so = make_float4(pos.x, pos.y, pos.z, len - kRayEps);
                            sd = make_float4(nuv.x, nuv.y, nuv.z, __uint_as_float(target));
                            sc = make_float4(c.x, c.y, c.z, 0.f);
                            push_shadow = true;
                        }
                    }
                    if (k < a.N - 1) {
                        const uint32_t dim = kDimBounce0 + kDimsPerBounce * bounce + kBdBsdf;
                        float3 wo;
                        float pdf = 0.f;
                        const float3 w = bsdf_sample(m, wi, u01(key, dim), u01(key, dim + 1), wo, pdf);
                        if (!is_black(w)) {
                            const float3 nd = to_world(f, wo);
                            new_o = make_float4(pos.x, pos.y, pos.z, ray_o.w);
                            new_d = make_float4(nd.x, nd.y, nd.z, ray_d.w);
                            new_thr = make_float4(w.x * T.x, w.y * T.y, w.z * T.z, 0.f);
                            cont = true;
                        }
                    }
                }
            }
        }
        const Append2 at = block_append2(&pb.counters[kQn], cont, push_shadow, agg, flip);
        const uint32_t qi = at.a, si = at.b;
        if (cont) {
            store_once(&ns.ray_o[qi], new_o);
            store_once(&ns.ray_d[qi], new_d);
            store_once(&ns.thr[qi], new_thr);
            rad.w = __uint_as_float(__float_as_uint(rad.w) + 1u);  // the next bounce
            store_once(&ns.rad[qi], rad);
        } else if (valid) {
            store_once(&pb.sample_rad[sidx], rad);
        }
        if (push_shadow) {
            store_once(&pb.sh_o[si], so);
            store_once(&pb.sh_d[si], sd);
            store_once(&pb.sh_c[si], sc);
        }
    }
    end_iteration(pb, a);
}

// ============================================================== extended shade
// k_shade with learned guiding and/or a homogeneous medium.
//
// Guiding: the direction at a vertex is drawn by one-sample MIS from the
// network's lobe mixture (probability alpha) or the BSDF / phase function, and
// weighted by f / (alpha q + (1 - alpha) p); the same combined density enters
// the NEE and emitter-hit MIS weights, so the estimator stays unbiased for any
// network.  k_guide_infer draws the direction and evaluates q.  Selected paths
// append a training record at every scattering vertex; the record is closed
// when the path's next vertex is shaded (radiance snapshot).
//
// Medium (homogeneous.h:11-66, generalsubpathsampler.h:40-53,131-154): each
// segment first samples a free flight on one colour channel; a flight that ends
// before the surface makes a medium vertex (throughput sigma_s Tr / pdf, NEE
// through the HG phase function, phase sampling), otherwise the surface is
// reached with throughput Tr / P(pass).  Shadow contributions carry the
// transmittance of their segment, and the MIS densities the pass probability.
__device__ __forceinline__ float guide_alpha(const DMat &m, float frac) {
    // sharp Phong lobes are sampled well by the BSDF itself
    return m.type == kPhong ? frac * fminf(1.f, fmaxf(0.1f, 30.f / m.n)) : frac;
}

// Network inference for the current state, for every vertex that k_shade_ext
// samples a direction at -- a surface that is not an emitter or the last
// vertex, or (with a medium) a scattering event before the last vertex -- one
// forward pass per wave of 64 entries on MFMA.  With the lobes on chip it also
// evaluates what shading needs of them: it draws the vertex's direction (the
// network with probability alpha, else the BSDF or phase function, from the
// same random numbers k_shade would use) and returns q at that direction and
// at the direction of the vertex's light sample.  The free-flight decision
// repeats k_shade_ext's.
// Network outputs reach their record's lane through v_permlane32_swap, so LDS
// holds only the weights (37 KB BF16, 18 KB e4m3) and the kernel runs 3 waves
// per SIMD (155-166 VGPRs): 2/3/4 waves took 91.7/82.4/81.4 ms of guided
// shading per 32 spp at 1080p (4 spills registers), 88.7 with the former
// 42 KB LDS stage at 2 waves.
#ifndef WR_INFER_WAVES
#define WR_INFER_WAVES 3
#endif
#ifndef WR_INFER_LDS_WEIGHTS
#define WR_INFER_LDS_WEIGHTS 1
#endif
constexpr int kInferBlock = 256;  // 4 waves share one LDS copy of the weights
// FP8: the e4m3 variant of the network (guide::forward8).
template <bool MEDIUM, bool FP8>
__global__ __launch_bounds__(kInferBlock) __attribute__((amdgpu_waves_per_eu(WR_INFER_WAVES, WR_INFER_WAVES))) void k_guide_infer(
    DScene s, PathState cs, const uint2 *__restrict__ hit, const uint32_t *__restrict__ counters, int N, guide::Net gnet,
    float frac, uint32_t max_bounce, guide::Draw out) {
    using OpT = typename std::conditional<FP8, guide::u32x2, guide::u32x4>::type;
#if WR_INFER_LDS_WEIGHTS
    __shared__ OpT w_ops[guide::kFwdOps];
#endif
    __shared__ float w_bias[guide::kBiasPacked];
    __shared__ float w_scale[guide::kLayers];
    const uint32_t n = active_count(counters);
    if (blockIdx.x * kInferBlock >= n) return;
#if WR_INFER_LDS_WEIGHTS
    const OpT *src;
    if constexpr (FP8) src = gnet.fwd8;
    else src = gnet.fwd;
    for (int j = threadIdx.x; j < guide::kFwdOps; j += kInferBlock) w_ops[j] = src[j];
#endif
    for (int j = threadIdx.x; j < guide::kBiasPacked; j += kInferBlock) w_bias[j] = gnet.bias[j];
    if (FP8 && threadIdx.x < guide::kLayers) w_scale[threadIdx.x] = gnet.wscale[threadIdx.x];
    __syncthreads();
    guide::Net net = gnet;
    if constexpr (FP8) {
#if WR_INFER_LDS_WEIGHTS
        net.fwd8 = w_ops;
#endif
        net.wscale = w_scale;
    } else {
#if WR_INFER_LDS_WEIGHTS
        net.fwd = w_ops;
#endif
    }
    net.bias = w_bias;
    for (uint32_t base = blockIdx.x * kInferBlock; base < n; base += gridDim.x * kInferBlock) {
        const uint32_t i = base + threadIdx.x;
        bool need = false, med = false;
        float3 pos = f3(0.f, 0.f, 0.f), ng = f3(0.f, 1.f, 0.f), nf = ng, rd = f3(0.f, 0.f, 1.f);
        int mat = 0;
        uint32_t key = 0, bounce = 0;
        if (i < n) {
            const uint2 h = hit[i];
            bounce = __float_as_uint(cs.rad[i].w);
            if (int(bounce) + 2 != N && bounce < max_bounce) {
                const float4 ray_o = load_once(&cs.ray_o[i]);
                key = __float_as_uint(ray_o.w);
                float tf = 0.f;
                med = MEDIUM && free_flight(s.med, key, bounce, h.x != kInvalid ? __uint_as_float(h.y) : INFINITY, tf);
                if (med) {
                    need = true;
                    rd = xyz(cs.ray_d[i]);
                    pos = xyz(ray_o) + rd * tf;
                    nf = -rd;  // no surface: the incoming direction stands in for the normal
                } else if (h.x != kInvalid) {
                    const float4 v0 = s.tris[3 * size_t(h.x) + 0];
                    const float4 v1 = s.tris[3 * size_t(h.x) + 1];
                    const float4 v2 = s.tris[3 * size_t(h.x) + 2];
                    const int2 gi = s.geom_info[__float_as_uint(v1.w)];
                    if (gi.y < 0) {
                        need = true;
                        mat = gi.x;
                        rd = xyz(cs.ray_d[i]);
                        pos = xyz(ray_o) + rd * __uint_as_float(h.y);
                        ng = normalize3(cross3(xyz(v1) - xyz(v0), xyz(v2) - xyz(v0)));
                        nf = dot3(ng, rd) > 0.f ? -ng : ng;
                    }
                }
            }
        }
        if (__ballot(need)) {
            float L[guide::kOut];  // this lane's record's raw outputs, then its decoded lobes
            if constexpr (FP8) guide::forward8(net, guide::encode(pos, nf, -rd, net.box), L);
            else guide::forward(net, guide::encode(pos, nf, -rd, net.box), L);
            if (need) {
                float wl[guide::kLobes];
                guide::decode(L, wl);
                const LightSample l = sample_light(s, u01(key, kDimLight), u01(key, kDimLight + 1), key);
                const float3 dl = normalize3(l.pos - pos);
                const uint32_t dim = kDimBounce0 + kDimsPerBounce * bounce + kBdBsdf;
                const float u0 = u01(key, dim), u1 = u01(key, dim + 1), us = u01(key, dim + 2);
                float alpha = frac;
                DMat m{};
                if (!med) {
                    m = s.mats[mat];
                    alpha = guide_alpha(m, frac);
                }
                // At a surface the mixture is folded onto the hemisphere of nf (the
                // BSDFs reflect only): a draw below the surface is mirrored across
                // the tangent plane, so the density is q(w) + q(R w) above and 0
                // below -- normalised, and no network draw is lost to f = 0.
                auto q = [&](float3 w) {
                    if (med) return guide::pdf(L, w);
                    const float c = dot3(w, nf);
                    return c < 0.f ? 0.f : guide::pdf(L, w) + guide::pdf(L, w - nf * (2.f * c));
                };
                float3 d;
                if (us < alpha) {
                    d = guide::sample(L, wl, us * guide::frcp(alpha), u0, u1);
                    const float c = dot3(d, nf);
                    if (!med && c < 0.f) d = d - nf * (2.f * c);
                } else if (med) {
                    d = hg_sample(s.med.g, rd, u0, u1);
                } else {
                    const Frame f = make_frame(ng);
                    float3 wo = f3(0.f, 0.f, 0.f);
                    float pb = 0.f;
                    bsdf_sample(m, to_local(f, -rd), u0, u1, wo, pb);
                    d = normalize3(to_world(f, wo));
                }
                out.dir[i] = make_float4(d.x, d.y, d.z, q(d));
                out.q_nee[i] = q(dl);
            }
        }
    }
}

template <bool GUIDED, bool MEDIUM>
__global__ __launch_bounds__(kShadeBlock) void k_shade_ext(DScene s, PathBuffers pb, RenderArgs a, guide::Shade g) {
    __shared__ uint32_t agg[2][kWavesPerShadeBlock + 2];
    __shared__ uint32_t rec_agg[kWavesPerShadeBlock + 1];
    const uint32_t n = active_count(pb.counters);
    const PathState cs = pb.cur, ns = pb.next;
    const float3 zero = f3(0.f, 0.f, 0.f);
    uint32_t flip = 0;
    for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += gridDim.x * blockDim.x, flip++) {
        const uint32_t i = base + threadIdx.x;
        const bool valid = i < n;
        // ---- the vertex
        float4 ray_o = make_float4(0, 0, 0, 0), ray_d = ray_o, rad = ray_o;
        uint2 h = make_uint2(kInvalid, 0u);
        float3 pos = zero, ng = f3(0.f, 1.f, 0.f), rd = f3(0.f, 0.f, 1.f);
        int2 gi = make_int2(0, -1);
        bool in_medium = false;
        float seg_t = 0.f;
        if (valid) {
            ray_o = load_once(&cs.ray_o[i]);
            ray_d = load_once(&cs.ray_d[i]);
            rad = load_once(&cs.rad[i]);
            h = load_once(&pb.hit[i]);
            rd = xyz(ray_d);
            seg_t = h.x != kInvalid ? __uint_as_float(h.y) : INFINITY;
            if (MEDIUM) {
                float tf = 0.f;
                in_medium = free_flight(s.med, __float_as_uint(ray_o.w), __float_as_uint(rad.w), seg_t, tf);
                if (in_medium) seg_t = tf;
            }
            if (in_medium) {
                pos = xyz(ray_o) + rd * seg_t;
            } else if (h.x != kInvalid) {
                pos = xyz(ray_o) + rd * seg_t;
                const float4 v0 = s.tris[3 * size_t(h.x) + 0];
                const float4 v1 = s.tris[3 * size_t(h.x) + 1];
                const float4 v2 = s.tris[3 * size_t(h.x) + 2];
                ng = normalize3(cross3(xyz(v1) - xyz(v0), xyz(v2) - xyz(v0)));
                gi = s.geom_info[__float_as_uint(v1.w)];
            }
        }
        const bool hit_vertex = valid && !in_medium && h.x != kInvalid;
        const uint32_t key = __float_as_uint(ray_o.w), sidx = __float_as_uint(ray_d.w), bounce = __float_as_uint(rad.w);
        const bool last = int(bounce) + 2 == a.N;
        const bool surf = hit_vertex && gi.y < 0 && !last;
        const bool med = valid && in_medium && !last;
        const float3 nf = in_medium ? -rd : (dot3(ng, rd) > 0.f ? -ng : ng);  // faces the incoming ray
        const bool need = GUIDED && (surf || med) && g.alpha > 0.f && bounce < g.max_bounce;
        float4 gdir = make_float4(0.f, 0.f, 0.f, 0.f);  // k_guide_infer's direction and q there
        float q_nee = 0.f;
        if (GUIDED && need) {
            gdir = g.draw.dir[i];
            q_nee = g.draw.q_nee[i];
        }
        // ---- shading
        bool push_shadow = false, cont = false;
        float4 so = make_float4(0, 0, 0, 0), sd = so, sc = so;
        float4 new_o = so, new_d = so, new_thr = so;
        float3 wdir = zero, T = zero;
        float prev_pdfw = 0.f;
        if (valid) {
            if (GUIDED) {
                // radiance before this vertex closes the record of the previous one
                const uint32_t prev = cs.rec[i];
                if (prev) g.rec.rad[prev - 1] = rad;
            }
            const float4 thr = load_once(&cs.thr[i]);
            prev_pdfw = thr.w;
            T = xyz(thr);
            if (MEDIUM && (in_medium || h.x != kInvalid)) {
                // free-flight weight of the segment
                const float3 tr = transmittance(s.med, seg_t);
                if (in_medium) T = T * f3(s.med.sig_s[0], s.med.sig_s[1], s.med.sig_s[2]) * tr * (1.f / scatter_pdf(s.med, seg_t));
                else T = T * tr * (1.f / pass_pdf(s.med, seg_t));
            }
        }
        if (hit_vertex && gi.y >= 0) {
            // emitter hit: MIS against light sampling (pathnextevent.h:128-146)
            const float cos_l = -dot3(ng, rd);
            if (cos_l >= 0.f) {
                const DLight &L = s.lights[gi.y];
                float mis = a.nee ? 0.f : 1.f;
                if (a.use_mis) {
                    float cPdfA = prev_pdfw * fabsf(cos_l) / (seg_t * seg_t);
                    if (MEDIUM) cPdfA *= pass_pdf(s.med, seg_t);
                    const float lightPdfA = L.pdf_select * L.inv_area;
                    mis = cPdfA / (lightPdfA + cPdfA);
                }
                rad.x += mis * T.x * L.L[0];
                rad.y += mis * T.y * L.L[1];
                rad.z += mis * T.z * L.L[2];
            }
        }
        if (surf || med) {
            DMat m{};
            Frame f{};
            float3 wi = zero;
            if (surf) {
                m = s.mats[gi.x];
                f = make_frame(ng);
                wi = to_local(f, -rd);
            }
            const float alpha = need ? (surf ? guide_alpha(m, g.alpha) : g.alpha) : 0.f;
            // NEE with MIS against the density that samples directions here (pathnextevent.h:106-127)
            const LightSample l = sample_light(s, u01(key, kDimLight), u01(key, kDimLight + 1), key);
            const float3 uv = l.pos - pos;
            const float len2 = dot3(uv, uv);
            const float len = sqrtf(len2);
            const float3 nuv = uv * (1.0f / len);
            const float cos_lv = -dot3(l.n, nuv);
            const float G = (med ? 1.f : fabsf(dot3(ng, nuv))) * fabsf(cos_lv) / len2;
            if (a.nee && G != 0.f && cos_lv >= 0.f) {
                float3 fs;
                float p;
                if (med) {
                    const float ph = hg_pdf(s.med.g, dot3(rd, nuv));
                    fs = f3(ph, ph, ph);
                    p = ph;
                } else {
                    const float3 wo = to_local(f, nuv);
                    fs = bsdf_eval(m, wi, wo);
                    p = bsdf_pdf(m, wi, wo);
                }
                if (!is_black(fs)) {
                    float mis = 1.f;
                    if (a.use_mis) {
                        if (GUIDED && need) p = alpha * q_nee + (1.f - alpha) * p;
                        float dirPdfA = p * fabsf(cos_lv) / len2;
                        if (MEDIUM) dirPdfA *= pass_pdf(s.med, len);
                        mis = l.pdfA / (l.pdfA + dirPdfA);
                    }
                    const float k = mis * G * kInvPi;
                    float3 c = T * fs * l.contrib * k;
                    if (MEDIUM) c = c * transmittance(s.med, len);
                    if (!is_black(c)) {
                        so = make_float4(pos.x, pos.y, pos.z, len - kRayEps);
                        sd = make_float4(nuv.x, nuv.y, nuv.z, 0.f);
                        sc = make_float4(c.x, c.y, c.z, 0.f);
                        push_shadow = true;
                    }
                }
            }
            // direction: BSDF or phase function, one-sample MIS with the network when guided
            const uint32_t dim = kDimBounce0 + kDimsPerBounce * bounce + kBdBsdf;
            const float u0 = u01(key, dim), u1 = u01(key, dim + 1);
            float3 nd = zero, w = zero;
            float pdf = 0.f;
            if (GUIDED && need) {
                // the direction k_guide_infer drew from the mixture alpha q + (1 - alpha) p;
                // whichever component drew it, its weight is f cos / (alpha q + (1 - alpha) p)
                nd = xyz(gdir);
                float3 fv;
                float pd;
                if (med) {
                    pd = hg_pdf(s.med.g, dot3(rd, nd));
                    fv = f3(pd, pd, pd);
                } else {
                    const float3 wo = to_local(f, nd);
                    fv = bsdf_eval(m, wi, wo) * fabsf(wo.y);
                    pd = bsdf_pdf(m, wi, wo);
                }
                pdf = alpha * gdir.w + (1.f - alpha) * pd;
                if (pdf > 0.f && !is_black(fv)) w = fv * (1.f / pdf);
            } else if (med) {
                nd = hg_sample(s.med.g, rd, u0, u1);
                pdf = hg_pdf(s.med.g, dot3(rd, nd));
                w = f3(1.f, 1.f, 1.f);
            } else {
                float3 wo = zero;
                w = bsdf_sample(m, wi, u0, u1, wo, pdf);
                nd = to_world(f, wo);
            }
            if (!is_black(w) && pdf > 0.f) {
                wdir = nd;
                new_o = make_float4(pos.x, pos.y, pos.z, ray_o.w);
                new_d = make_float4(nd.x, nd.y, nd.z, ray_d.w);
                new_thr = make_float4(w.x * T.x, w.y * T.y, w.z * T.z, a.use_mis ? pdf : 0.f);
                cont = true;
            }
        }
        uint32_t rec_id = 0;
        if (GUIDED && g.collect) {
            const bool want = cont && bounce < g.max_bounce && float(mix32(key ^ 0x68bc21ebu) >> 8) * 0x1p-24f < g.record_prob;
            const uint32_t r = block_append(g.rec.count, want, rec_agg);
            if (want && r < g.rec.capacity) {
                g.rec.pos[r] = make_float4(pos.x, pos.y, pos.z, ray_d.w);
                g.rec.nrm[r] = make_float4(nf.x, nf.y, nf.z, 0.f);
                g.rec.wo[r] = make_float4(-rd.x, -rd.y, -rd.z, 0.f);
                g.rec.wi[r] = make_float4(wdir.x, wdir.y, wdir.z, 0.f);
                g.rec.thr[r] = make_float4(T.x, T.y, T.z, 0.f);
                g.rec.rad[r] = make_float4(0.f, 0.f, 0.f, 0.f);
                rec_id = r + 1;
            }
        }
        const Append2 at = block_append2(&pb.counters[kQn], cont, push_shadow, agg, flip);
        const uint32_t qi = at.a, si = at.b;
        if (cont) {
            store_once(&ns.ray_o[qi], new_o);
            store_once(&ns.ray_d[qi], new_d);
            store_once(&ns.thr[qi], new_thr);
            rad.w = __uint_as_float(bounce + 1u);
            store_once(&ns.rad[qi], rad);
            if (GUIDED) ns.rec[qi] = rec_id;
        } else if (valid) {
            store_once(&pb.sample_rad[sidx], rad);
        }
        const uint32_t target = cont ? (kToNextPath | qi) : (kToSample | sidx);
        sd.w = __uint_as_float(target);
        if (push_shadow) {
            store_once(&pb.sh_o[si], so);
            store_once(&pb.sh_d[si], sd);
            store_once(&pb.sh_c[si], sc);
        }
    }
    end_iteration(pb, a);
}

// ============================================================== shadow
// Any hit for the n entries of the shadow queue the previous shade kernel (and
// this iteration's regeneration) filled; a visible connection adds its
// contribution to the radiance of its path (continuing: by then in the
// current state; finished: its sample), or to the FP64 splat film for
// light->camera (t = 1) connections.  `st_ent` is the block's LDS stack, here of
// node refs (any hit keeps no entry distances).
template <bool COUNT, bool BATCH>
__device__ __forceinline__ void shadow_rays(DScene s1, const BatchJob *__restrict__ jobs, PathBuffers pb, uint2 *spill,
                                            TravTune tune, uint32_t n, uint32_t first_block, uint64_t *st_ent) {
    const uint32_t chunk = spread_chunk(n, tune.chunk);
    LaneStack<kBlock, true> st(st_ent, spill);
    TraversalCounters cnt;
    TravState ts;
    ts.cur = kEndRef;
    uint32_t i = 0;
    WaveRange wr(n, first_block);
    Geo geo{s1.nodes, s1.tris};
    bool active = false, exhausted = false;
    for (;;) {
        const unsigned long long idle = __ballot(!active);
        if (!exhausted && __popcll(idle) >= tune.refill) {
            const uint32_t j = refill(&pb.counters[kFetchShdX], n, !active, idle, wr, exhausted, chunk);
            if (!active && j < n) {
                i = j;
                const float4 o = load_once(&pb.sh_o[i]), d = load_once(&pb.sh_d[i]);
                if (BATCH) {
                    const DScene &sj = jobs[__float_as_uint(pb.sh_c[i].w)].s;
                    geo = Geo{sj.nodes, sj.tris};
                }
                trav_begin(ts, setup_ray(xyz(o), xyz(d), kRayEps), o.w);
                st.reset();
                active = true;
            }
        }
        if (__ballot(active) == 0) {
            if (exhausted) break;
            continue;
        }
        if (BATCH) trav_round_any<COUNT, kBlock>(geo, ts, st, cnt);
        else trav_round_any<COUNT, kBlock>(s1, ts, st, cnt);
        if (active && ts.cur == kEndRef) {
            active = false;
            if (ts.hit == kInvalid) {
                const float4 c = pb.sh_c[i];
                const uint32_t target = __float_as_uint(pb.sh_d[i].w);
                const uint32_t idx = target & kTargetMask;
                if ((target & ~kTargetMask) == kToSplat) {
                    double *dst = (BATCH ? jobs[__float_as_uint(c.w)].film_splat : pb.film_splat) + 3 * size_t(idx);
                    atomicAdd(dst + 0, double(c.x));
                    atomicAdd(dst + 1, double(c.y));
                    atomicAdd(dst + 2, double(c.z));
                } else {
                    // the three sums alone: other waves of this launch read a path's fourth word, its job
                    float *r = &((target & ~kTargetMask) == kToSample ? pb.sample_rad + idx : pb.cur.rad + idx)->x;
                    const float rx = r[0] + c.x, ry = r[1] + c.y, rz = r[2] + c.z;
                    r[0] = rx; r[1] = ry; r[2] = rz;
                }
            }
        }
    }
    if (COUNT) {
        wave_add_stat(&pb.stats[4], cnt.nodes);
        wave_add_stat(&pb.stats[5], cnt.tris);
    }
}

// ============================================================== traversal launch
// One launch per iteration traces the closest-hit rays of the current state
// and the shadow queue of the previous shade kernel: the two are independent
// (both read only what that shade kernel and this iteration's regeneration
// wrote), and in one launch each queue's last, slowest rays overlap the other
// queue's work instead of ending a launch of their own.  A block with
// closest-hit work traces it first; the shadow queue is dealt to the blocks
// from the first one without closest-hit work on (block index rotated by the
// number of blocks the closest-hit rays occupy), so short queues run side by
// side and long ones back to back.  Both share the block's LDS stack.
template <bool COUNT, bool BATCH>
__device__ __forceinline__ void trace_bounce(DScene s1, const BatchJob *__restrict__ jobs, PathBuffers pb, uint2 *spill,
                                             TravTune tune) {
    __shared__ uint64_t st_ent[kLdsSlots * kBlock];
    const uint32_t n_ext = active_count(pb.counters);
    const uint32_t n_shd = pb.counters[pb.next.shadow_count];
    const uint32_t g = gridDim.x;
    const uint32_t ext_blocks = min(g, n_ext / kBlock + (n_ext % kBlock != 0));
    if (blockIdx.x < ext_blocks) extend_rays<COUNT, BATCH>(s1, jobs, pb, spill, tune, n_ext, st_ent);
    const uint32_t sb = (blockIdx.x + g - ext_blocks) % g;
    if (sb * kBlock < n_shd)
        shadow_rays<COUNT, BATCH>(s1, jobs, pb, spill, tune, n_shd, sb, st_ent);
}
template <bool COUNT, bool BATCH>
__global__ __launch_bounds__(kBlock) WR_EXTEND_ATTR(WR_BATCH_WAVES) void k_trace_bounce(DScene s1, const BatchJob *__restrict__ jobs,
                                                                        PathBuffers pb, uint2 *spill, TravTune tune) {
    trace_bounce<COUNT, BATCH>(s1, jobs, pb, spill, tune);
}
// ============================================================== small passes
// A pass of few samples, start to end in one launch.  Its iterations are bound
// by the latency of their launches and queues (about 28 us each, of which a
// traversal over a short queue takes 12), so a block of two waves keeps 64 paths
// in registers: the first wave starts them, traces their closest hits and
// shades; the second traces the shadow rays that the first one left in LDS, at
// the same time.  The arithmetic and the order in which a sample's radiance is
// summed are those of k_regen, k_trace_bounce_fast and k_shade.
//
// A block has per_block consecutive samples: a tile of 64, or, where the pass
// has more tiles than the spill region has pairs of slices, an equal share of
// the pass for each resident block, which starts the next samples in the lanes
// whose paths have ended once kRestartLanes of them have.
//
// A wave steps at the pace of its slowest ray, where the queues refill lanes
// inside a traversal; with enough rays to fill the chip several times over they
// win, the earlier the more the lengths of the traversals differ.  Queues / this
// kernel, in ms, by samples of the pass (12 to 18 path vertices):
//                          16,384       131,044      262,144      1,048,576    4,194,304
//   Cornell box, 36         0.33 / 0.17  0.53 / 0.25  0.59 / 0.42  1.83 / 1.11  5.25 / 3.72
//   clutter, 1,000                                   0.75 / 0.55  2.05 / 1.36  5.47 / 4.61
//   clutter, 5,000                                   0.84 / 0.65  2.17 / 1.68  5.61 / 5.79
//   clutter, 40,000                                  0.97 / 0.70  2.31 / 1.95  5.71 / 6.79
//   clutter, 200,000                                 1.16 / 0.84  2.57 / 2.33  6.15 / 8.05
//   spheres, 1.31M         1.54 / 0.59  2.27 / 0.95  2.34 / 1.27  3.09 / 2.40
//   gap room, 1.0M         2.31 / 1.33  2.99 / 1.68  3.21 / 3.04  7.70 / 10.4
// (16,777,216 in the Cornell box 14.2 / 14.2), hence small_pass_samples.  Six
// waves per SIMD, at which 132 bytes a lane spill to scratch (192 with an envmap):
// 262,144 samples of the gap room take 3.04 ms, 3.6 at four.  Restarting at 1 / 8 / 16 / 32 idle lanes:
// 3.91 / 3.78 / 3.72 / 3.96 ms in the box at 4,194,304 samples.
constexpr uint32_t kRestartLanes = 16;
// Largest pass of k_small_pass in a scene of n_tris triangles; passes of at most
// a tile per pair of spill slices (2^18 samples; 2^15 in the fixed region, whose
// 512 blocks would leave most of the chip idle with more) always take it.
static uint32_t small_pass_samples(uint32_t n_tris) {
    return n_tris <= 1u << 11 ? 1u << 22 : n_tris <= 1u << 16 ? 1u << 20 : 0u;
}
template <bool ENV>
__global__ __launch_bounds__(2 * kBlock) WR_EXTEND_ATTR(6) void k_small_pass(DScene s, PathBuffers pb, RenderArgs a, uint32_t per_block, uint2 *spill) {
    __shared__ uint64_t st_ent[2][kLdsSlots * kBlock];
    __shared__ float4 sh_o[kBlock], sh_d[kBlock], sh_c[kBlock];
    __shared__ uint32_t sent[kBlock], seen[kBlock];  // a shadow ray of lane l; it adds to its path
    __shared__ uint32_t more;
    const uint32_t wave = threadIdx.x / kBlock, lane = lane_id();
    const DCamera &cam = s.cam;
    uint2 *my_spill = spill + size_t(blockIdx.x + wave) * (kSpillDepth * kBlock);  // slice 2 blockIdx.x + wave
    TraversalCounters cnt;
    uint32_t rays = 0;
    uint32_t next = min(blockIdx.x * per_block, a.total);  // wave 0: the block's next sample
    const uint32_t end = min(next + per_block, a.total);
    bool alive = false, pending = false;  // pending: ended, its last shadow ray is on its way
    bool shadow = false;                  // v.so, v.sd, v.sc is a shadow ray to trace
    uint32_t sidx = 0;
    Vertex v;
    float4 rad = make_float4(0, 0, 0, 0);
    for (;;) {
        if (wave == 0) {
            const unsigned long long idle = __ballot(!alive && !pending);
            const uint32_t k = (uint32_t)__popcll(idle);
            if (next < end && k >= kRestartLanes) {
                if (!alive && !pending) {
                    sidx = next + mbcnt64(idle);
                    alive = sidx < end;
                    v = Vertex{};
                    rad = make_float4(0, 0, 0, 0);
                    if (alive) {
                        const uint32_t pixel = sidx % a.wh;
                        const uint32_t key = path_key(a.seed, pixel, a.first_sample + sidx / a.wh);
                        start_path<ENV>(s, a, a.use_mis, key, pixel % uint32_t(cam.W), pixel / uint32_t(cam.W), 0u, v);
                        v.o.w = __uint_as_float(key);
                    }
                    shadow = v.shadow;
                }
                next = min(next + k, end);
            }
            sent[lane] = shadow;
            if (shadow) { sh_o[lane] = v.so; sh_d[lane] = v.sd; sh_c[lane] = v.sc; }
            const bool go = __ballot(alive || pending) != 0;
            if (lane == 0) more = go;
        }
        __syncthreads();  // the shadow rays and `more` are written
        if (!more) break;
        uint2 h = make_uint2(kInvalid, 0u);
        if (wave == 0) {
            if (alive) {
                float t = INFINITY;
                h.x = traverse_rounds<false, kBlock>(s, setup_ray(xyz(v.o), xyz(v.d), kRayEps), t, st_ent[0], my_spill, cnt);
                h.y = __float_as_uint(t);
                rays++;
            }
        } else {
            bool adds = false;
            if (sent[lane]) {
                const float4 o = sh_o[lane], d = sh_d[lane];
                float t = o.w;
                const bool visible = traverse_rounds<true, kBlock>(s, setup_ray(xyz(o), xyz(d), kRayEps), t, st_ent[1],
                                                                   my_spill, cnt) == kInvalid;
                const uint32_t target = __float_as_uint(d.w);
                const bool splat = (target & ~kTargetMask) == kToSplat;
                if (visible && splat) {
                    const float4 c = sh_c[lane];
                    double *dst = pb.film_splat + 3 * size_t(target & kTargetMask);
                    atomicAdd(dst + 0, double(c.x));
                    atomicAdd(dst + 1, double(c.y));
                    atomicAdd(dst + 2, double(c.z));
                }
                adds = visible && !splat;
                rays++;
            }
            seen[lane] = adds;
        }
        __syncthreads();  // the shadow rays are traced
        if (wave != 0) continue;
        if (seen[lane]) {
            const float4 c = sh_c[lane];
            rad.x += c.x; rad.y += c.y; rad.z += c.z;
        }
        bool ended = pending;
        pending = shadow = false;
        if (alive) {
            const float4 o = v.o, thr = v.thr;
            Vertex nv;
            shade_vertex<ENV>(s, a, a.N, a.use_mis, h, xyz(v.d), sidx, rad, [&] { return o; }, [&] { return thr; }, nv);
            nv.sd.w = __uint_as_float(kToSample);
            v = nv;
            shadow = v.shadow;
            alive = v.cont;
            ended = !alive && !shadow;
            pending = !alive && shadow;
            rad.w = __uint_as_float(__float_as_uint(rad.w) + 1u);  // the next bounce
        }
        if (ended) store_once(&pb.sample_rad[sidx], rad);
    }
    wave_add_stat(&pb.stats[wave], rays);
}

// The plain kernel of wr_render_nee / wr_render_guided and the other
// integrators' loops.
__global__ __launch_bounds__(kBlock) WR_EXTEND_ATTR(WR_EXTEND_WAVES) void k_trace_bounce_fast(DScene s1, PathBuffers pb, uint2 *spill,
                                                                             TravTune tune) {
    trace_bounce<false, false>(s1, nullptr, pb, spill, tune);
}

// ============================================================== accumulate
// Film::addSample for a pass (film.h:42-48): the samples of pixel p are
// p, p + wh, p + 2 wh, ...; their FP32 radiance is summed in FP64, in sample
// order, so the film is bit-reproducible.
__global__ void k_accumulate(const float4 *__restrict__ sample_rad, double *film_base, uint32_t wh, uint32_t spp) {
    for (uint32_t px = blockIdx.x * blockDim.x + threadIdx.x; px < wh; px += gridDim.x * blockDim.x) {
        double r = 0.0, g = 0.0, b = 0.0;
        for (uint32_t k = 0; k < spp; k++) {
            const float4 v = sample_rad[size_t(k) * wh + px];
            r += v.x; g += v.y; b += v.z;
        }
        double *dst = film_base + 3 * size_t(px);
        dst[0] += r; dst[1] += g; dst[2] += b;
    }
}

// Film::getImage (film.h:78-90, pathnextevent.h:154-157) of `n` film values:
// base / spp + splat / (spp W H), written straight to pinned host memory.
__global__ void k_film_image(const double *__restrict__ base, const double *__restrict__ splat, double base_div,
                             double splat_div, double *__restrict__ out, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = base[i] / base_div + splat[i] / splat_div;
}

// ============================================================== trace kernels (parity / benchmark)
// Hits leave as (leaf triangle, t) pairs, or, with IDS, as what the host API
// returns: the geometry, the triangle within it and t in three arrays of n
// (a triangle record holds its input index and geometry; geom_first is each
// geometry's first triangle).  A block takes tiles of 64 rays in a stride of the
// grid, which is what is resident (8M any-hit rays among 1.31M triangles: 228 us,
// 264 with 8,192 blocks of which 7,168 are).  Closest hit runs 8 waves per SIMD
// (8M rays in a 40,000-triangle clutter 742 us, 7 waves 850), any hit, whose
// registers fit 7 without spills, 7 (2M rays 104 us, 8 waves 116).
template <bool ANY, bool IDS = false>
__global__ __launch_bounds__(kBlock) WR_EXTEND_ATTR(ANY ? 7 : 8) void k_trace(DScene s, const float4 *__restrict__ rays, uint32_t n, uint2 *hits,
                                                  uint8_t *occ, const uint32_t *__restrict__ geom_first, uint2 *spill) {
    __shared__ uint64_t st_ent[kLdsSlots * kBlock];
    TraversalCounters cnt;
    for (uint32_t base = blockIdx.x * kBlock; base < n; base += gridDim.x * kBlock) {
        const uint32_t i = base + lane_id();
        if (i < n) {
            const float4 a = rays[2 * size_t(i)], b = rays[2 * size_t(i) + 1];
            const RaySetup r = setup_ray(xyz(a), xyz(b), a.w);
            float t = b.w;
            const uint32_t tri = traverse_rounds<ANY, kBlock>(s, r, t, st_ent, spill, cnt);
            if (ANY) occ[i] = tri != kInvalid;
            else if (IDS) {
                uint32_t *out = reinterpret_cast<uint32_t *>(hits);
                uint32_t geom = kInvalid, prim = kInvalid;
                if (tri != kInvalid) {
                    geom = __float_as_uint(s.tris[3 * size_t(tri) + 1].w);
                    prim = __float_as_uint(s.tris[3 * size_t(tri)].w) - geom_first[geom];
                }
                out[i] = geom;
                out[size_t(n) + i] = prim;
                out[2 * size_t(n) + i] = __float_as_uint(tri == kInvalid ? INFINITY : t);
            } else hits[i] = make_uint2(tri, __float_as_uint(tri == kInvalid ? INFINITY : t));
        }
    }
}

// VisualizeGeometryNormal::render (visualizegeomnormal.h:32-74): per sample
// the camera ray's first hit adds (1, 1, 1) on an emitter and the unit
// geometric normal (v1 - v0) x (v2 - v0), unflipped, as RGB on any other
// surface; a miss adds nothing.  The camera sample (lens point, pixel jitter)
// is the path tracers' one.  One lane per pixel sums its samples in sample
// order into the FP64 base film, so the film is bit-reproducible.
__global__ __launch_bounds__(kBlock) void k_visualize(DScene s, uint32_t wh, uint32_t spp, uint32_t first_sample,
                                                      uint32_t seed, double *film_base, uint2 *spill) {
    __shared__ uint64_t st_ent[kLdsSlots * kBlock];
    TraversalCounters cnt;
    const DCamera &cam = s.cam;
    for (uint32_t pixel = blockIdx.x * kBlock + lane_id(); pixel < wh; pixel += gridDim.x * kBlock) {
        const uint32_t px = pixel % uint32_t(cam.W), py = pixel / uint32_t(cam.W);
        double r = 0.0, g = 0.0, b = 0.0;
        for (uint32_t k = 0; k < spp; k++) {
            const uint32_t key = path_key(seed, pixel, first_sample + k);
            const float3 lens = lens_point(cam, key);
            const float3 cpos = cam_to_world(cam, lens) + f3(cam.ox, cam.oy, cam.oz);
            float pdfW;
            const float3 dir = primary_dir(cam, key, px, py, lens, pdfW);
            float t = INFINITY;
            const uint32_t tri = traverse_rounds<false, kBlock>(Geo4{s.fnodes, s.tris}, setup_ray(cpos, dir, kRayEps),
                                                                t, st_ent, spill, cnt);
            if (tri == kInvalid) {
                if (s.env_select > 0.f) { r += 1.0; g += 1.0; b += 1.0; }  // the envmap vertex is a light vertex
                continue;
            }
            const float4 v0 = s.tris[3 * size_t(tri) + 0], v1 = s.tris[3 * size_t(tri) + 1],
                         v2 = s.tris[3 * size_t(tri) + 2];
            if (s.geom_info[__float_as_uint(v1.w)].y >= 0) {
                r += 1.0; g += 1.0; b += 1.0;
            } else {
                const float3 ng = normalize3(cross3(xyz(v1) - xyz(v0), xyz(v2) - xyz(v0)));
                r += ng.x; g += ng.y; b += ng.z;
            }
        }
        double *dst = film_base + 3 * size_t(pixel);
        dst[0] += r; dst[1] += g; dst[2] += b;
    }
}

// ============================================================== bidirectional path tracing
// BidirPathRenderer::render (bidirpath.h:316-395) for one lane per pixel and
// its samples in sample order: a light subpath (traceLightSubpath,
// bidirpath.h:196-219) whose vertices go to a per-lane record array in HBM,
// then a camera subpath (traceCameraSubpath, bidirpath.h:221-257) whose every
// surface vertex connects to every stored light vertex (bdptConnect,
// bidirpath.h:79-123); t = 1 connections (light vertex -> camera vertex) are
// FP64 atomic splats, the rest sum into the pixel's FP64 base film.
//
// Balance-heuristic weights (computeMisWeight, bidirpath.h:125-194, power 1):
// 1 / w = 1 + sum of the light-side ratio products + sum of the camera-side
// ones.  With b_i = (camera-side pdf / light-side pdf) of light vertex i and
// a_j = (light-side pdf / camera-side pdf) of camera vertex j, the light sum of
// strategy (s, t) is b_s'(1 + b_{s-1}'(1 + E_{s-2})) with E_k = b_k (1 + E_{k-1}),
// E_0 = 0, and the camera sum a_t'(1 + a_{t-1}'(1 + D_{t-2})) with
// D_k = a_k (1 + D_{k-1}), D_1 = 0 (the camera vertex never enters); primes
// are the pdfs re-evaluated at the connection, the rest are fixed once the
// subpath has moved two vertices on.  Each connection therefore costs O(1)
// instead of the reference's loop over the path.
//
// Light vertex record (4 float4 per vertex, one plane per field, lane-major):
//   0: position, pdf with which the light subpath made it (area)
//   1: geometric normal, -
//   2: throughput (mPathContrib), E_{k-2}
//   3: direction to the previous light vertex, material (bits)
constexpr int kBdptMaxVertices = 64;
constexpr uint32_t kBdptKeySalt = 0x3c6ef372u;  // the light subpath's walk draws from its own stream

__device__ __forceinline__ float bd_conv(float3 from, float3 to, float3 to_n) {
    const float3 u = to - from;
    const float l2 = dot3(u, u);
    return fabsf(dot3(to_n, u)) / (sqrtf(l2) * l2);
}
__device__ __forceinline__ float bd_cam_pdfW(const DCamera &cam, float3 w) {
    const float c = cam_to_local(cam, w).z;
    return cam.per_pixel_norm / (c * c * c);
}
__device__ __forceinline__ float bd_weight(float inv) {
    const float w = 1.f / inv;
    return w >= 0.f && w <= 1.f ? w : 0.f;  // a zero forward pdf (grazing FP32 hit) weighs 0
}

// Capped at 128 VGPRs (4 waves per SIMD; 328 B/lane spill to scratch): 227 VGPRs
// and 2 waves measured 676 / 4,351 Mrays/s on the 1.31M-triangle frame at 4 spp /
// a 512^2 Cornell box at 16 spp, 4 waves 912-945 / 5,341, 6 waves 1,046 / 3,530,
// 8 waves 803 / 2,932; the film is bit-identical across all of them.
__global__ __launch_bounds__(kBlock, 4) void k_bdpt(DScene s, uint32_t wh, uint32_t spp, uint32_t first_sample,
                                                 uint32_t seed, int N, double *film_base, double *film_splat,
                                                 float4 *__restrict__ recs, unsigned long long *counts, uint2 *spill) {
    __shared__ uint64_t st_ent[kLdsSlots * kBlock];
    TraversalCounters cnt;
    const DCamera &cam = s.cam;
    const float3 cz = f3(cam.zx, cam.zy, cam.zz);
    const size_t lanes = size_t(gridDim.x) * kBlock, lane = size_t(blockIdx.x) * kBlock + lane_id();
    auto rec = [&](int k, int f) -> float4 & { return recs[(size_t(k - 1) * 4 + f) * lanes + lane]; };
    unsigned long long n_ext = 0, n_shd = 0;
    auto occluded = [&](float3 o, float3 d, float len) {
        n_shd++;
        float t = len - kRayEps;
        return traverse_rounds<true, kBlock>(Geo4{s.fnodes, s.tris}, setup_ray(o, d, kRayEps), t, st_ent, spill, cnt) != kInvalid;
    };
    auto closest = [&](float3 o, float3 d, float &t) {
        n_ext++;
        t = INFINITY;
        return traverse_rounds<false, kBlock>(Geo4{s.fnodes, s.tris}, setup_ray(o, d, kRayEps), t, st_ent, spill, cnt);
    };
    for (uint32_t pixel = blockIdx.x * kBlock + lane_id(); pixel < wh; pixel += gridDim.x * kBlock) {
        const uint32_t px = pixel % uint32_t(cam.W), py = pixel / uint32_t(cam.W);
        double acc_r = 0.0, acc_g = 0.0, acc_b = 0.0;
        for (uint32_t k = 0; k < spp; k++) {
            const uint32_t key = path_key(seed, pixel, first_sample + k);
            const uint32_t kl = mix32(key ^ kBdptKeySalt);
            const float3 lens = lens_point(cam, key);
            const float3 cpos = cam_to_world(cam, lens) + f3(cam.ox, cam.oy, cam.oz);
            // ---- light subpath
            const LightSample l = sample_light<false>(s, u01(key, kDimLight), u01(key, kDimLight + 1), key);
            rec(1, 0) = make_float4(l.pos.x, l.pos.y, l.pos.z, l.pdfA);
            rec(1, 1) = make_float4(l.n.x, l.n.y, l.n.z, 0.f);
            rec(1, 2) = make_float4(l.contrib.x, l.contrib.y, l.contrib.z, 0.f);
            int nL = 1;
            // t = 1 connection of vertex sN (light or surface) to the camera vertex
            auto splat_camera = [&](float3 p, float3 n, float3 T, float pf, bool is_light, const DMat &m, float3 wi_w,
                                    float3 q_p, float3 q_n, float q_pf, float E2, int sN) {
                const float3 uv = cpos - p;
                const float len2 = dot3(uv, uv), len = sqrtf(len2);
                const float3 nuv = uv * (1.f / len);
                const float G = fabsf(dot3(n, nuv)) * fabsf(dot3(cz, nuv)) / len2;
                if (G == 0.f) return;
                float rx = 0.f, ry = 0.f;
                const float we1 = camera_we1(cam, lens, -nuv, rx, ry);
                if (we1 == 0.f) return;
                float3 fl;
                const Frame fr = make_frame(n);
                if (is_light) {
                    if (to_local(fr, nuv).y < 0.f) return;
                    fl = f3(kInvPi, kInvPi, kInvPi);
                } else {
                    fl = bsdf_eval(m, to_local(fr, wi_w), to_local(fr, nuv));
                    if (is_black(fl)) return;
                }
                if (occluded(p, nuv, len)) return;
                // weight: light-side ratios only (t = 1)
                const float bs = bd_cam_pdfW(cam, -nuv) * fabsf(dot3(n, nuv)) / len2 / pf;
                float inv;
                if (sN == 1) {
                    inv = 1.f + bs;
                } else {
                    const float cq = bsdf_pdf(m, to_local(fr, nuv), to_local(fr, wi_w)) * bd_conv(p, q_p, q_n);
                    inv = 1.f + bs * (1.f + (cq / q_pf) * (1.f + E2));
                }
                const float c = bd_weight(inv) * G * we1;
                const float3 v = T * fl * c;
                double *dst = film_splat + 3 * (size_t(uint32_t(ry)) * uint32_t(cam.W) + uint32_t(rx));
                atomicAdd(dst + 0, double(v.x));
                atomicAdd(dst + 1, double(v.y));
                atomicAdd(dst + 2, double(v.z));
            };
            const DMat none{};
            splat_camera(l.pos, l.n, l.contrib, l.pdfA, true, none, f3(0, 0, 0), f3(0, 0, 0), f3(0, 0, 0), 1.f, 0.f, 1);
            if (N - 1 >= 2) {
                const Frame lf = make_frame(l.n);
                float3 ro = l.pos;
                float3 rd = to_world(lf, cosine_hemisphere(u01(kl, kDimPixel), u01(kl, kDimPixel + 1)));
                float pdfW = fmaxf(to_local(lf, rd).y, 0.f) * kInvPi;
                float3 w = f3(1.f, 1.f, 1.f), T = l.contrib;
                // the previous vertex q: position, normal, forward pdf
                float3 q_p = l.pos, q_n = l.n;
                float q_pf = l.pdfA;
                float E2 = 0.f;  // E_{k-2} for the vertex about to be made
                for (uint32_t bounce = 0;; bounce++) {
                    float t;
                    const uint32_t tri = closest(ro, rd, t);
                    if (tri == kInvalid) break;
                    const float4 v0 = s.tris[3 * size_t(tri) + 0], v1 = s.tris[3 * size_t(tri) + 1],
                                 v2 = s.tris[3 * size_t(tri) + 2];
                    const int2 gi = s.geom_info[__float_as_uint(v1.w)];
                    if (gi.y >= 0) break;  // a light ends the light subpath
                    const float3 p = ro + rd * t;
                    const float3 ng = normalize3(cross3(xyz(v1) - xyz(v0), xyz(v2) - xyz(v0)));
                    const float3 wiw = -rd;
                    T = T * w;
                    const float pf = pdfW * bd_conv(q_p, p, ng);
                    nL++;
                    rec(nL, 0) = make_float4(p.x, p.y, p.z, pf);
                    rec(nL, 1) = make_float4(ng.x, ng.y, ng.z, 0.f);
                    rec(nL, 2) = make_float4(T.x, T.y, T.z, E2);
                    rec(nL, 3) = make_float4(wiw.x, wiw.y, wiw.z, __int_as_float(gi.x));
                    const DMat m = s.mats[gi.x];
                    splat_camera(p, ng, T, pf, false, m, wiw, q_p, q_n, q_pf, E2, nL);
                    if (nL == N - 1) break;
                    const Frame f = make_frame(ng);
                    const float3 wi = to_local(f, wiw);
                    const uint32_t dim = kDimBounce0 + kDimsPerBounce * bounce + kBdBsdf;
                    float3 wo;
                    float pdf = 0.f;
                    w = bsdf_sample(m, wi, u01(kl, dim), u01(kl, dim + 1), wo, pdf);
                    if (is_black(w)) break;
                    // the previous vertex's camera-side pdf given this direction -> E_{k-1}
                    const float pr_q = bsdf_pdf(m, wo, wi) * bd_conv(p, q_p, q_n);
                    E2 = (pr_q / q_pf) * (1.f + E2);  // E_{k-1}, stored with the next vertex
                    q_p = p; q_n = ng; q_pf = pf;
                    pdfW = pdf;
                    ro = p;
                    rd = to_world(f, wo);
                }
            }
            // ---- camera subpath
            float pdfW;
            float3 rd = primary_dir(cam, key, px, py, lens, pdfW);
            float3 ro = cpos;
            float3 q_p = cpos, q_n = cz;  // previous camera-subpath vertex
            float q_pf = 1.f;
            float3 T = f3(1.f, 1.f, 1.f), w = f3(1.f, 1.f, 1.f);
            float D2 = 0.f;  // D_{t-2}
            float sr = 0.f, sg = 0.f, sb = 0.f;
            for (int tv = 2; tv <= N; tv++) {
                float th;
                const uint32_t tri = closest(ro, rd, th);
                if (tri == kInvalid) break;
                const float4 v0 = s.tris[3 * size_t(tri) + 0], v1 = s.tris[3 * size_t(tri) + 1],
                             v2 = s.tris[3 * size_t(tri) + 2];
                const int2 gi = s.geom_info[__float_as_uint(v1.w)];
                const float3 p = ro + rd * th;
                const float3 ng = normalize3(cross3(xyz(v1) - xyz(v0), xyz(v2) - xyz(v0)));
                const float3 wiw = -rd;
                T = T * w;
                const float pf = pdfW * bd_conv(q_p, p, ng);
                if (gi.y >= 0) {
                    // s = 0: the camera subpath ends on an emitter (Le1 * Le0 = L on its front)
                    const float cl = dot3(ng, wiw);
                    if (cl >= 0.f) {
                        const DLight &L = s.lights[gi.y];
                        const float at = L.pdf_select * L.inv_area / pf;
                        float inv;
                        if (tv == 2) {
                            inv = 1.f + at;
                        } else {
                            const float pr_q = cl * kInvPi * bd_conv(p, q_p, q_n);
                            inv = 1.f + at * (1.f + (pr_q / q_pf) * (1.f + D2));
                        }
                        const float c = bd_weight(inv) * (kInvPi * kPi);
                        sr += T.x * L.L[0] * c; sg += T.y * L.L[1] * c; sb += T.z * L.L[2] * c;
                    }
                    break;
                }
                if (tv == N) break;
                const DMat m = s.mats[gi.x];
                const Frame f = make_frame(ng);
                const float3 wi = to_local(f, wiw);
                // connections to the stored light vertices, s + t <= N
                const int smax = min(nL, N - tv);
                for (int sN = 1; sN <= smax; sN++) {
                    const float4 A = rec(sN, 0), B = rec(sN, 1), Cc = rec(sN, 2);
                    const float3 lp = xyz(A), ln = xyz(B);
                    const float3 uv = p - lp;  // light vertex -> camera vertex
                    const float len2 = dot3(uv, uv), len = sqrtf(len2);
                    const float3 nuv = uv * (1.f / len);
                    const float G = fabsf(dot3(ln, nuv)) * fabsf(dot3(ng, nuv)) / len2;
                    if (G == 0.f) continue;
                    const float3 wo_c = to_local(f, -nuv);
                    const float3 fc = bsdf_eval(m, wi, wo_c);
                    if (is_black(fc)) continue;
                    const Frame lfr = make_frame(ln);
                    float3 fl;
                    float lpdf_c;  // light-side pdf of the camera vertex (solid angle at the light vertex)
                    DMat lm{};
                    float3 lwi_l = f3(0, 0, 0);
                    if (sN == 1) {
                        const float cl = to_local(lfr, nuv).y;
                        if (cl < 0.f) continue;
                        fl = f3(kInvPi, kInvPi, kInvPi);
                        lpdf_c = cl * kInvPi;
                    } else {
                        const float4 Dd = rec(sN, 3);
                        lm = s.mats[__float_as_int(Dd.w)];
                        lwi_l = to_local(lfr, xyz(Dd));
                        const float3 lwo = to_local(lfr, nuv);
                        fl = bsdf_eval(lm, lwi_l, lwo);
                        if (is_black(fl)) continue;
                        lpdf_c = bsdf_pdf(lm, lwi_l, lwo);
                    }
                    if (occluded(lp, nuv, len)) continue;
                    // light-side sum
                    const float bs = bsdf_pdf(m, wi, wo_c) * fabsf(dot3(ln, nuv)) / len2 / A.w;
                    float lsum;
                    if (sN == 1) {
                        lsum = bs;
                    } else {
                        const float4 Aq = rec(sN - 1, 0), Bq = rec(sN - 1, 1);
                        const float cq = bsdf_pdf(lm, to_local(lfr, nuv), lwi_l) * bd_conv(lp, xyz(Aq), xyz(Bq));
                        lsum = bs * (1.f + (cq / Aq.w) * (1.f + Cc.w));
                    }
                    // camera-side sum
                    const float at = lpdf_c * fabsf(dot3(ng, nuv)) / len2 / pf;
                    float csum;
                    if (tv == 2) {
                        csum = at;
                    } else {
                        const float lq = bsdf_pdf(m, wo_c, wi) * bd_conv(p, q_p, q_n);
                        csum = at * (1.f + (lq / q_pf) * (1.f + D2));
                    }
                    const float c = bd_weight(1.f + lsum + csum) * G;
                    const float3 v = xyz(Cc) * fl * fc * T * c;
                    sr += v.x; sg += v.y; sb += v.z;
                }
                // continue the camera subpath
                const uint32_t dim = kDimBounce0 + kDimsPerBounce * uint32_t(tv - 2) + kBdBsdf;
                float3 wo;
                float pdf = 0.f;
                w = bsdf_sample(m, wi, u01(key, dim), u01(key, dim + 1), wo, pdf);
                if (is_black(w)) break;
                if (tv >= 3) {  // D_{t-1} from the previous vertex's light-side pdf given this direction
                    const float pr_q = bsdf_pdf(m, wo, wi) * bd_conv(p, q_p, q_n);
                    D2 = (pr_q / q_pf) * (1.f + D2);
                }
                q_p = p; q_n = ng; q_pf = pf;
                pdfW = pdf;
                ro = p;
                rd = to_world(f, wo);
            }
            acc_r += sr; acc_g += sg; acc_b += sb;
        }
        double *dst = film_base + 3 * size_t(pixel);
        dst[0] += acc_r; dst[1] += acc_g; dst[2] += acc_b;
    }
    atomicAdd(counts + 0, n_ext);
    atomicAdd(counts + 1, n_shd);
}

// Resident blocks per CU of a kernel (HIP occupancy API), cached per device.
static int occupancy(wr_device *d, const void *fn, int block) {
    std::lock_guard<std::mutex> lock(d->occ_mutex);  // scenes of one device may render in several threads
    auto it = d->occ_cache.find(fn);
    if (it != d->occ_cache.end()) return it->second;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, block, 0) != hipSuccess || nb <= 0) nb = 1;
    nb = std::min(nb, kMaxTraversalBlocksPerCU);
    d->occ_cache[fn] = nb;
    return nb;
}

// The entry points below inherit C linkage from their declarations in wurst_amd.h.

const char *wr_last_error(void) { return wr::error_string().c_str(); }
const char *wr_version(void) { return "wurst_amd 0.1 (gfx950, BVH4-128B, wavefront NEE+MIS)"; }

static int scratch_setup(wr_device *d);

int wr_device_create(int ordinal, wr_device **out) {
    if (!out) return set_error(WR_ERR_INVALID_ARGUMENT, "out is null");
    *out = nullptr;
    int count = 0;
    WR_HIP(hipGetDeviceCount(&count));
    if (ordinal < 0 || ordinal >= count) return set_error(WR_ERR_INVALID_ARGUMENT, "device ordinal out of range");
    WR_HIP(hipSetDevice(ordinal));
    hipDeviceProp_t prop;
    WR_HIP(hipGetDeviceProperties(&prop, ordinal));
    wr_device *d = new wr_device;
    d->ordinal = ordinal;
    d->n_cu = prop.multiProcessorCount;
    auto occ = [](const void *fn, int block, int &out_blocks) {
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, block, 0) == hipSuccess && nb > 0) out_blocks = nb;
        out_blocks = std::min(out_blocks, kMaxTraversalBlocksPerCU);
    };
    occ(reinterpret_cast<const void *>(&k_trace_bounce_fast), kBlock, d->occ_rays);
    occ(reinterpret_cast<const void *>(&k_regen<false>), kShadeBlock, d->occ_generate);
    if (int rc = scratch_setup(d)) {
        delete d;
        return rc;
    }
    *out = d;
    return WR_OK;
}

void wr_device_destroy(wr_device *dev) { delete dev; }

constexpr size_t align256(size_t b) { return (b + 255) / 256 * 256; }

void wr_scene_destroy(wr_scene *s) {
    if (!s) return;
    (void)hipSetDevice(s->dev->ordinal);
    if (s->stream) (void)hipStreamSynchronize(s->stream);
    // (freeing the geometry of 1.31M triangles, 170 MB, takes 1 ms)
    auto drop = [&](BlockPool::Block &b, void *p) {
        if (b.p) s->dev->geometry.give(b);
        else (void)hipFree(p);
    };
    drop(s->nodes_block, s->d_nodes);
    drop(s->qnodes_block, s->d_qnodes);
    drop(s->tris_block, s->d_tris);
    (void)hipFree(s->d_tables);
    (void)hipFree(s->d_env);
    (void)hipFree(s->d_env_cdf);
    s->dev->spills.give(s->spill);
    (void)hipFree(s->d_bdpt);
    (void)hipFree(s->pool);
    if (s->h_counters) (void)hipHostFree(s->h_counters);
    for (auto &e : s->ev)
        if (e) (void)hipEventDestroy(e);
    if (s->stream) (void)hipStreamDestroy(s->stream);
    delete s;
}

// `arrays`: also the checks over the vertex and triangle arrays, which the GPU
// build does on the device (mesh_check_gpu).
static int validate_desc(const wr_scene_desc *d, bool arrays = true) {
    if (!d) return set_error(WR_ERR_INVALID_ARGUMENT, "desc is null");
    if (d->n_tris > 0 && (!d->verts || !d->tris || !d->tri_geom))
        return set_error(WR_ERR_INVALID_ARGUMENT, "null geometry arrays");
    if (d->n_tris >= kMaxTriangles) return set_error(WR_ERR_UNSUPPORTED, "too many triangles (limit 2^28)");
    if (d->n_verts > 0 && !d->verts) return set_error(WR_ERR_INVALID_ARGUMENT, "null vertex array");
    for (size_t i = 0; arrays && i < 3 * size_t(d->n_verts); i++)
        if (!std::isfinite(d->verts[i])) return set_error(WR_ERR_INVALID_ARGUMENT, "non-finite vertex coordinate");
    if (d->camera.width <= 0 || d->camera.height <= 0) return set_error(WR_ERR_INVALID_ARGUMENT, "bad resolution");
    if ((uint64_t)d->camera.width * d->camera.height >= (1ull << 31))
        return set_error(WR_ERR_UNSUPPORTED, "resolution too large");
    if (!(d->camera.focal_distance > 0.f))
        return set_error(WR_ERR_INVALID_ARGUMENT, "focal distance must be > 0 (the JSON key \"radius\" sets it)");
    if (!(d->camera.fovy_deg > 0.f && d->camera.fovy_deg < 180.f))
        return set_error(WR_ERR_INVALID_ARGUMENT, "fovy must be in (0, 180) degrees");
    for (uint32_t i = 0; arrays && i < 3 * d->n_tris; i++)
        if (d->tris[i] >= d->n_verts) return set_error(WR_ERR_INVALID_ARGUMENT, "triangle vertex index out of range");
    uint32_t prev = 0;
    for (uint32_t t = 0; arrays && t < d->n_tris; t++) {
        if (d->tri_geom[t] >= d->n_geoms) return set_error(WR_ERR_INVALID_ARGUMENT, "tri_geom out of range");
        if (d->tri_geom[t] < prev) return set_error(WR_ERR_INVALID_ARGUMENT, "triangles of a geometry must be contiguous and ordered");
        prev = d->tri_geom[t];
    }
    for (uint32_t g = 0; g < d->n_geoms; g++) {
        const int m = d->geom_material[g], l = d->geom_light[g];
        if (l >= (int)d->n_lights) return set_error(WR_ERR_INVALID_ARGUMENT, "geom_light out of range");
        if (l < 0 && (m < 0 || m >= (int)d->n_materials))
            return set_error(WR_ERR_INVALID_ARGUMENT, "geometry without a valid material");
    }
    for (uint32_t m = 0; m < d->n_materials; m++)
        if (d->materials[m].type < 0 || d->materials[m].type > 3) return set_error(WR_ERR_INVALID_ARGUMENT, "unknown material type");
    for (uint32_t l = 0; l < d->n_lights; l++)
        if (d->lights[l].geom < 0 || (uint32_t)d->lights[l].geom >= d->n_geoms)
            return set_error(WR_ERR_INVALID_ARGUMENT, "light geometry out of range");
    return WR_OK;
}

int wr_scene_validate(const wr_scene_desc *desc) { return validate_desc(desc); }

int wr_bvh_selftest(const wr_scene_desc *d, uint64_t *n_nodes, uint32_t *max_stack, uint32_t *depth) {
    int rc = validate_desc(d);
    if (rc) return rc;
    BvhBuildResult bvh;
    if (!build_bvh4(d->verts, d->n_verts, d->tris, d->n_tris, d->tri_geom, &bvh))
        return set_error(WR_ERR_OUT_OF_MEMORY, "host allocation failed during BVH build");
    const std::string err = verify_bvh4(bvh, d->verts, d->tris, d->n_tris);
    if (n_nodes) *n_nodes = bvh.n_nodes;
    if (max_stack) *max_stack = bvh.max_stack;
    if (depth) *depth = bvh.depth;
    free_bvh(&bvh);
    if (!err.empty()) return set_error(WR_ERR_DEVICE, "BVH invariant violated: " + err);
    return WR_OK;
}

template <typename T>
static int upload(wr_device *dev, T **dst, const void *src, size_t bytes, uint64_t &total) {
    WR_HIP(dev->alloc(reinterpret_cast<void **>(dst), std::max<size_t>(bytes, 128)));
    if (bytes) WR_HIP(hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice));
    total += bytes;
    return WR_OK;
}

// Bounds of the vertices (lo xyz, hi xyz).
static void scene_bounds(wr_scene *s, const wr_scene_desc *d) {
    for (int k = 0; k < 3; k++) { s->box[k] = INFINITY; s->box[3 + k] = -INFINITY; }
    for (uint32_t v = 0; v < d->n_verts; v++)
        for (int k = 0; k < 3; k++) {
            s->box[k] = std::min(s->box[k], d->verts[3 * size_t(v) + k]);
            s->box[3 + k] = std::max(s->box[3 + k], d->verts[3 * size_t(v) + k]);
        }
}

// Host SAH build, uploaded.
static int bvh_host(wr_scene *s, const wr_scene_desc *d) {
    const auto t0 = std::chrono::steady_clock::now();
    BvhBuildResult bvh;
    if (!build_bvh4(d->verts, d->n_verts, d->tris, d->n_tris, d->tri_geom, &bvh))
        return set_error(WR_ERR_OUT_OF_MEMORY, "host allocation failed during BVH build");
    s->n_nodes = bvh.n_nodes;
    s->max_stack = bvh.max_stack;
    s->bvh_depth = bvh.depth;
    int rc = upload(s->dev, &s->d_nodes, bvh.nodes, sizeof(Node4) * bvh.n_nodes, s->device_bytes);
    if (!rc) rc = upload(s->dev, &s->d_tris, bvh.tris, sizeof(TriRecord) * bvh.n_tris, s->device_bytes);
    free_bvh(&bvh);
    s->build_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return rc;
}

// GPU checks and PLOC build from a temporary device copy of the mesh; also sets
// the scene's bounds.
static int bvh_gpu(wr_scene *s, const wr_scene_desc *d) {
    const auto t0 = std::chrono::steady_clock::now();
    const uint32_t n = d->n_tris;
    GpuBvhResult g;
    int rc = WR_OK;
    if (n == 0) {
        if ((rc = validate_desc(d))) return rc;
        scene_bounds(s, d);
        rc = build_bvh4_gpu(s->dev, BuildBuffers{}, 0, s->stream, s->ploc_radius, &g);
    } else {
        BuildArena arena(s->dev, s->stream);
        BuildBuffers b{};
        if ((rc = bvh_gpu_plan(n, d->n_verts, s->stream, &arena, &b))) return rc;
        WR_HIP(arena.commit());
        b.tris = reinterpret_cast<uint32_t *>(b.verts + 3 * size_t(d->n_verts));
        b.tri_geom = b.tris + 3 * size_t(n);
        WR_HIP(s->dev->ring.upload(s->dev->ordinal, s->stream, b.verts,
                                   {{d->verts, sizeof(float) * 3 * size_t(d->n_verts)},
                                    {d->tris, sizeof(uint32_t) * 3 * size_t(n)},
                                    {d->tri_geom, sizeof(uint32_t) * size_t(n)}}));
        bool valid = false;
        if ((rc = mesh_check_gpu(b, n, d->n_verts, d->n_geoms, s->stream, &valid, s->box))) return rc;
        if (!valid) {  // the host checks name the fault
            rc = validate_desc(d);
            return rc ? rc : set_error(WR_ERR_INVALID_ARGUMENT, "invalid mesh");
        }
        rc = build_bvh4_gpu(s->dev, b, n, s->stream, s->ploc_radius, &g);
    }
    s->d_nodes = g.nodes;
    s->d_tris = reinterpret_cast<float4 *>(g.tris);
    s->nodes_block = g.nodes_block;
    s->tris_block = g.tris_block;
    if (rc) return rc;
    s->device_bytes += sizeof(Node4) * uint64_t(g.n_nodes) + sizeof(TriRecord) * uint64_t(n);
    s->n_nodes = g.n_nodes;
    s->max_stack = g.max_stack;
    s->bvh_depth = g.depth;
    s->bvh_iterations = g.iterations;
    s->build_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return WR_OK;
}

static int scene_create_impl(wr_device *dev, const wr_scene_desc *d, int builder, int radius, wr_scene *s) {
    s->dev = dev;
    int rc = set_device(dev);
    if (rc) return rc;
    WR_HIP(hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking));
    WR_HIP(hipEventCreate(&s->ev[0]));
    WR_HIP(hipEventCreate(&s->ev[1]));
    s->W = d->camera.width;
    s->H = d->camera.height;
    // BVH
    s->builder = builder;
    s->ploc_radius = radius;
    s->n_tris = d->n_tris;
    if (builder == WR_BVH_HOST) scene_bounds(s, d);
    rc = builder == WR_BVH_HOST ? bvh_host(s, d) : bvh_gpu(s, d);
    if (rc) return rc;
    // each geometry's first triangle (kInvalid: none); the triangles are in geometry order
    s->geom_first.assign(d->n_geoms, kInvalid);
    if (d->n_geoms > d->n_tris / 32) {
        for (uint32_t t = d->n_tris; t-- > 0;) s->geom_first[d->tri_geom[t]] = t;
    } else {
        for (uint32_t g = 0; g < d->n_geoms; g++) {
            const uint32_t *first = std::lower_bound(d->tri_geom, d->tri_geom + d->n_tris, g);
            if (first != d->tri_geom + d->n_tris && *first == g) s->geom_first[g] = uint32_t(first - d->tri_geom);
        }
    }
    WR_HIP(dev->take(dev->geometry, sizeof(NodeQ) * std::max<uint64_t>(s->n_nodes, 1), &s->qnodes_block));
    s->d_qnodes = static_cast<NodeQ *>(s->qnodes_block.p);
    s->device_bytes += sizeof(NodeQ) * s->n_nodes;
    if (s->n_nodes) {
        k_quantize_nodes<<<uint32_t((s->n_nodes + 255) / 256), 256, 0, s->stream>>>(s->d_nodes, s->d_qnodes,
                                                                                    uint32_t(s->n_nodes));
        WR_HIP(hipGetLastError());
    }
    if (s->max_stack > (uint32_t)kStackDepth) return set_error(WR_ERR_UNSUPPORTED, "BVH deeper than the traversal stack");
    s->max_trav_blocks = dev->n_cu * kMaxTraversalBlocksPerCU;
    {
        const size_t spill_bytes = sizeof(uint2) * size_t(s->max_trav_blocks) * kBlock * kSpillDepth;
        WR_HIP(dev->take(dev->spills, spill_bytes, &s->spill));
        s->d_spill = static_cast<uint2 *>(s->spill.p);
        s->device_bytes += spill_bytes;
    }
    // geometry info
    std::vector<int2> gi(d->n_geoms);
    for (uint32_t g = 0; g < d->n_geoms; g++) gi[g] = make_int2(d->geom_material[g], d->geom_light[g]);
    std::vector<DMat> mats(d->n_materials);
    for (uint32_t m = 0; m < d->n_materials; m++) {
        const wr_material &src = d->materials[m];
        DMat &dm = mats[m];
        dm.type = src.type;
        dm.twosided = src.twosided;
        dm.sigma = src.sigma;
        dm.n = src.exponent;
        for (int k = 0; k < 3; k++) { dm.rho_d[k] = src.rho_d[k]; dm.rho_s[k] = src.rho_s[k]; }
        dm.rho_d[3] = dm.rho_s[3] = 0.f;
    }
    // lights: selection CdfTable over |L|_2, per-light triangle-area CdfTable (FP64 on the host)
    std::vector<DLight> lights(d->n_lights);
    std::vector<float4> ltris;
    std::vector<double> w(d->n_lights);
    double wsum = 0.0;
    for (uint32_t l = 0; l < d->n_lights; l++) {
        const float *L = d->lights[l].L;
        w[l] = std::sqrt(double(L[0]) * L[0] + double(L[1]) * L[1] + double(L[2]) * L[2]);
        wsum += w[l];
    }
    if (d->n_lights > 0 && !(wsum > 0.0)) return set_error(WR_ERR_INVALID_ARGUMENT, "all lights have zero radiance");
    s->light_w = w;
    double cdf = 0.0;
    for (uint32_t l = 0; l < d->n_lights; l++) {
        DLight &dl = lights[l];
        const uint32_t g = (uint32_t)d->lights[l].geom;
        const double pdf = w[l] / wsum;
        cdf += pdf;
        dl.pdf_select = float(pdf);
        dl.cdf_select = (l + 1 == d->n_lights) ? 1.0f : float(cdf);
        for (int k = 0; k < 3; k++) dl.L[k] = d->lights[l].L[k];
        uint32_t first = s->geom_first[g];
        if (first == kInvalid) return set_error(WR_ERR_INVALID_ARGUMENT, "light geometry has no triangles");
        uint32_t cnt = 0;
        while (first + cnt < d->n_tris && d->tri_geom[first + cnt] == g) cnt++;
        std::vector<double> area(cnt);
        double asum = 0.0;
        for (uint32_t i = 0; i < cnt; i++) {
            const uint32_t *t = d->tris + 3 * size_t(first + i);
            const float *a = d->verts + 3 * size_t(t[0]), *b = d->verts + 3 * size_t(t[1]), *c = d->verts + 3 * size_t(t[2]);
            double e1[3], e2[3];
            for (int k = 0; k < 3; k++) { e1[k] = double(b[k]) - a[k]; e2[k] = double(c[k]) - a[k]; }
            const double cx = e1[1] * e2[2] - e1[2] * e2[1], cy = e1[2] * e2[0] - e1[0] * e2[2], cz = e1[0] * e2[1] - e1[1] * e2[0];
            area[i] = std::sqrt(cx * cx + cy * cy + cz * cz) / 2.0;
            asum += area[i];
        }
        if (!(asum > 0.0)) return set_error(WR_ERR_INVALID_ARGUMENT, "light with zero area");
        dl.area = float(asum);
        dl.inv_area = float(1.0 / asum);
        dl.first_ltri = uint32_t(ltris.size() / 3);
        dl.n_ltri = cnt;
        double tc = 0.0;
        for (uint32_t i = 0; i < cnt; i++) {
            const uint32_t *t = d->tris + 3 * size_t(first + i);
            const double tp = area[i] / asum;
            tc += tp;
            const float tcdf = (i + 1 == cnt) ? 1.0f : float(tc);
            const float *a = d->verts + 3 * size_t(t[0]), *b = d->verts + 3 * size_t(t[1]), *c = d->verts + 3 * size_t(t[2]);
            ltris.push_back(make_float4(a[0], a[1], a[2], tcdf));
            ltris.push_back(make_float4(b[0], b[1], b[2], float(tp)));
            ltris.push_back(make_float4(c[0], c[1], c[2], 0.f));
        }
    }
    s->h_lights = lights;
    // the tables in one allocation and one copy, each with room for an entry
    {
        struct Table { void **p; const void *src; size_t bytes, at; };
        Table tabs[] = {{reinterpret_cast<void **>(&s->d_geom), gi.data(), sizeof(int2) * gi.size(), 0},
                        {reinterpret_cast<void **>(&s->d_geom_first), s->geom_first.data(), sizeof(uint32_t) * s->geom_first.size(), 0},
                        {reinterpret_cast<void **>(&s->d_mats), mats.data(), sizeof(DMat) * mats.size(), 0},
                        {reinterpret_cast<void **>(&s->d_lights), lights.data(), sizeof(DLight) * lights.size(), 0},
                        {reinterpret_cast<void **>(&s->d_ltris), ltris.data(), sizeof(float4) * ltris.size(), 0}};
        size_t total = 0;
        for (Table &t : tabs) {
            t.at = total;
            total += align256(std::max<size_t>(t.bytes, 1));
            s->device_bytes += t.bytes;
        }
        std::vector<char> host(total);
        WR_HIP(dev->alloc(&s->d_tables, total));
        for (Table &t : tabs) {
            if (t.bytes) std::memcpy(host.data() + t.at, t.src, t.bytes);
            *t.p = static_cast<char *>(s->d_tables) + t.at;
        }
        WR_HIP(hipMemcpyAsync(s->d_tables, host.data(), total, hipMemcpyHostToDevice, s->stream));
        WR_HIP(hipStreamSynchronize(s->stream));  // the tables and the quantised nodes are there for any stream
    }
    // camera (ThinlensCamera ctor, thinlens.h:40-55; Camera ctor, camera.h:9-17), FP64 then rounded
    const wr_camera &c = d->camera;
    double o[3] = {c.pos[0], c.pos[1], c.pos[2]}, la[3] = {c.lookat[0], c.lookat[1], c.lookat[2]},
           up[3] = {c.up[0], c.up[1], c.up[2]};
    auto norm = [](double v[3]) {
        double l = std::sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
        for (int k = 0; k < 3; k++) v[k] /= l;
    };
    auto cross = [](const double a[3], const double b[3], double r[3]) {
        r[0] = a[1] * b[2] - a[2] * b[1];
        r[1] = a[2] * b[0] - a[0] * b[2];
        r[2] = a[0] * b[1] - a[1] * b[0];
    };
    double z[3] = {la[0] - o[0], la[1] - o[1], la[2] - o[2]}, x[3], y[3];
    norm(z);
    cross(up, z, x);
    norm(x);
    cross(z, x, y);
    norm(y);
    DCamera &dc = s->ds.cam;
    dc.ox = c.pos[0]; dc.oy = c.pos[1]; dc.oz = c.pos[2];
    dc.xx = float(x[0]); dc.xy = float(x[1]); dc.xz = float(x[2]);
    dc.yx = float(y[0]); dc.yy = float(y[1]); dc.yz = float(y[2]);
    dc.zx = float(z[0]); dc.zy = float(z[1]); dc.zz = float(z[2]);
    const double fovy = double(c.fovy_deg) * 3.14159265358979323846 / 180.0;
    const double dist = double(c.height) * 0.5 / std::tan(fovy * 0.5);
    dc.d = float(dist);
    dc.W = c.width;
    dc.H = c.height;
    dc.invW = float(1.0 / c.width);
    dc.invH = float(1.0 / c.height);
    dc.per_pixel_norm = float(dist * dist / (double(c.width) * double(c.height)));
    dc.per_film_norm = float(dist * dist);
    dc.aperture = c.aperture_radius;
    dc.focal = c.focal_distance;
    s->ds.nodes = s->d_qnodes;
    s->ds.fnodes = s->d_nodes;
    s->ds.tris = s->d_tris;
    s->ds.geom_info = s->d_geom;
    s->ds.mats = s->d_mats;
    s->ds.lights = s->d_lights;
    s->ds.ltris = s->d_ltris;
    s->ds.n_lights = d->n_lights;
    return WR_OK;
}

int wr_scene_create(wr_device *dev, const wr_scene_desc *desc, wr_scene **out) {
    return wr_scene_create_ex(dev, desc, nullptr, out);
}

int wr_scene_create_ex(wr_device *dev, const wr_scene_desc *desc, const wr_build_params *params, wr_scene **out) {
    if (!dev || !out) return set_error(WR_ERR_INVALID_ARGUMENT, "null argument");
    *out = nullptr;
    const int builder = params ? params->builder : WR_BVH_GPU;
    const int radius = params ? params->ploc_radius : 0;
    if (builder != WR_BVH_GPU && builder != WR_BVH_HOST) return set_error(WR_ERR_INVALID_ARGUMENT, "unknown BVH builder");
    if (radius < 0 || radius > 64) return set_error(WR_ERR_INVALID_ARGUMENT, "ploc_radius must be in [0, 64]");
    // the GPU build checks the arrays on the device; where anything else is wrong,
    // the host's checks say what comes first
    int rc = validate_desc(desc, builder == WR_BVH_HOST);
    if (rc) return validate_desc(desc);
    wr_scene *s = new wr_scene;
    rc = scene_create_impl(dev, desc, builder, radius, s);
    if (rc) {
        std::string msg = wr::error_string();
        wr_scene_destroy(s);
        wr::error_string() = msg;
        return rc;
    }
    *out = s;
    return WR_OK;
}

int wr_scene_info(const wr_scene *s, uint64_t *n_nodes, uint64_t *n_tris, uint32_t *max_stack, uint64_t *bytes) {
    if (!s) return set_error(WR_ERR_INVALID_ARGUMENT, "scene is null");
    if (n_nodes) *n_nodes = s->n_nodes;
    if (n_tris) *n_tris = s->n_tris;
    if (max_stack) *max_stack = s->max_stack;
    if (bytes) *bytes = s->device_bytes;
    return WR_OK;
}

int wr_scene_bvh_check(wr_scene *s, const wr_scene_desc *d, wr_bvh_stats *st) {
    if (!s || !d || !st) return set_error(WR_ERR_INVALID_ARGUMENT, "null argument");
    if (d->n_tris != s->n_tris) return set_error(WR_ERR_INVALID_ARGUMENT, "desc is not the scene's description");
    int rc = set_device(s->dev);
    if (rc) return rc;
    BvhBuildResult r;
    r.n_nodes = uint32_t(s->n_nodes);
    r.n_tris = uint32_t(s->n_tris);
    r.max_stack = s->max_stack;
    r.depth = s->bvh_depth;
    std::vector<Node4> nodes(s->n_nodes);
    std::vector<TriRecord> tris(s->n_tris);
    WR_HIP(hipStreamSynchronize(s->stream));
    WR_HIP(hipMemcpy(nodes.data(), s->d_nodes, sizeof(Node4) * nodes.size(), hipMemcpyDeviceToHost));
    if (!tris.empty())
        WR_HIP(hipMemcpy(tris.data(), s->d_tris, sizeof(TriRecord) * tris.size(), hipMemcpyDeviceToHost));
    r.nodes = nodes.data();
    r.tris = tris.data();
    const std::string err = verify_bvh4(r, d->verts, d->tris, d->n_tris);
    if (!err.empty()) return set_error(WR_ERR_DEVICE, "BVH invariant violated: " + err);
    for (uint32_t i = 0; i < s->n_tris; i++)
        if (tris[i].geom != d->tri_geom[tris[i].orig])
            return set_error(WR_ERR_DEVICE, "BVH invariant violated: leaf triangle geometry id");
    // the traversal copy: same refs, and every child's planes (origin + q * spacing) contain its Node4 box
    {
        std::vector<NodeQ> qn(s->n_nodes);
        WR_HIP(hipMemcpy(qn.data(), s->d_qnodes, sizeof(NodeQ) * qn.size(), hipMemcpyDeviceToHost));
        for (size_t i = 0; i < qn.size(); i++) {
            const Node4 &a = nodes[i];
            const NodeQ &b = qn[i];
            const float *lo[3] = {a.lo_x, a.lo_y, a.lo_z}, *hi[3] = {a.hi_x, a.hi_y, a.hi_z};
            const float sc[3] = {b.scale_x, b.scale_y, b.scale_z};
            const uint32_t pl[6] = {b.x01, b.x23, b.y01, b.y23, b.z01, b.z23};
            const uint32_t ref[4] = {b.child0, b.child1, b.child2, b.child3};
            for (int c = 0; c < 4; c++) {
                if (ref[c] != a.child[c])
                    return set_error(WR_ERR_DEVICE, "BVH invariant violated: quantised node refs differ");
                if (a.child[c] == kEmptyChild) continue;
                for (int k = 0; k < 3; k++) {
                    if (std::isinf(sc[k])) continue;  // spacing * 2^24 overflows: the axis encloses everything
                    const uint32_t w = pl[2 * k + (c >> 1)] >> (8 * (c & 1));
                    const double sp = double(sc[k]) * 0x1p-24;
                    if (!((w & 0xFFu) * sp <= double(lo[k][c]) - double(b.org[k]) &&
                          ((w >> 16) & 0xFFu) * sp >= double(hi[k][c]) - double(b.org[k])))
                        return set_error(WR_ERR_DEVICE, "BVH invariant violated: quantised box of node " +
                                                            std::to_string(i) + " does not contain its child " +
                                                            std::to_string(c));
                }
            }
        }
    }
    // SAH cost relative to the root box
    auto area = [](const Node4 &n, int c) {
        const double dx = double(n.hi_x[c]) - n.lo_x[c], dy = double(n.hi_y[c]) - n.lo_y[c],
                     dz = double(n.hi_z[c]) - n.lo_z[c];
        return (dx < 0 || dy < 0 || dz < 0) ? 0.0 : dx * dy + dy * dz + dz * dx;
    };
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int c = 0; c < 4; c++)
        if (nodes[0].child[c] != kEmptyChild) {
            lo[0] = std::min(lo[0], double(nodes[0].lo_x[c])); hi[0] = std::max(hi[0], double(nodes[0].hi_x[c]));
            lo[1] = std::min(lo[1], double(nodes[0].lo_y[c])); hi[1] = std::max(hi[1], double(nodes[0].hi_y[c]));
            lo[2] = std::min(lo[2], double(nodes[0].lo_z[c])); hi[2] = std::max(hi[2], double(nodes[0].hi_z[c]));
        }
    const double dx = hi[0] - lo[0], dy = hi[1] - lo[1], dz = hi[2] - lo[2];
    const double aroot = (s->n_tris == 0) ? 0.0 : dx * dy + dy * dz + dz * dx;
    double cost = 1.0;
    if (aroot > 0.0)
        for (const Node4 &n : nodes)
            for (int c = 0; c < 4; c++) {
                if (n.child[c] == kEmptyChild) continue;
                cost += area(n, c) / aroot * ((n.child[c] & kLeafBit) ? double(n.count[c]) : 1.0);
            }
    // FNV-1a over nodes then triangles
    uint64_t h = 1469598103934665603ull;
    auto mix = [&h](const void *p, size_t bytes) {
        const uint8_t *b = static_cast<const uint8_t *>(p);
        for (size_t i = 0; i < bytes; i++) h = (h ^ b[i]) * 1099511628211ull;
    };
    mix(nodes.data(), sizeof(Node4) * nodes.size());
    mix(tris.data(), sizeof(TriRecord) * tris.size());
    st->builder = s->builder;
    st->depth = s->bvh_depth;
    st->max_stack = s->max_stack;
    st->iterations = s->bvh_iterations;
    st->n_nodes = s->n_nodes;
    st->build_ms = s->build_ms;
    st->sah_cost = cost;
    st->hash = h;
    return WR_OK;
}

int wr_scene_set_medium(wr_scene *s, const wr_medium *m) {
    if (!s) return set_error(WR_ERR_INVALID_ARGUMENT, "scene is null");
    DMedium dm{};
    if (m) {
        if (!(m->g > -1.f && m->g < 1.f)) return set_error(WR_ERR_INVALID_ARGUMENT, "HG g must be in (-1, 1)");
        for (int c = 0; c < 3; c++) {
            if (!(m->sigma_a[c] >= 0.f) || !(m->sigma_s[c] >= 0.f) || !std::isfinite(m->sigma_a[c] + m->sigma_s[c]))
                return set_error(WR_ERR_INVALID_ARGUMENT, "medium coefficients must be finite and >= 0");
            dm.sig_s[c] = m->sigma_s[c];
            dm.sig_t[c] = m->sigma_a[c] + m->sigma_s[c];
            dm.on |= dm.sig_t[c] > 0.f;
        }
        dm.g = m->g;
    }
    s->ds.med = dm;
    return WR_OK;
}

// The light-selection CdfTable over the area lights' |L|_2 and, last, the
// envmap's weight 1.23 (generalsubpathsampler.h:167-176; envmap.h:22-26).
static int rebuild_light_select(wr_scene *s, bool env) {
    double wsum = env ? 1.23 : 0.0;
    for (double w : s->light_w) wsum += w;
    double cdf = 0.0;
    for (size_t l = 0; l < s->h_lights.size(); l++) {
        const double pdf = s->light_w[l] / wsum;
        cdf += pdf;
        s->h_lights[l].pdf_select = float(pdf);
        s->h_lights[l].cdf_select = (!env && l + 1 == s->h_lights.size()) ? 1.0f : float(cdf);
    }
    s->ds.env_select = env ? float(1.23 / wsum) : 0.f;
    if (!s->h_lights.empty())
        WR_HIP(hipMemcpy(s->d_lights, s->h_lights.data(), sizeof(DLight) * s->h_lights.size(), hipMemcpyHostToDevice));
    return WR_OK;
}

int wr_scene_set_envmap(wr_scene *s, const float *rgb, uint32_t width, uint32_t height) {
    if (!s) return set_error(WR_ERR_INVALID_ARGUMENT, "scene is null");
    int rc = set_device(s->dev);
    if (rc) return rc;
    WR_HIP(hipStreamSynchronize(s->stream));
    if (!rgb || width == 0) {
        (void)hipFree(s->d_env);
        (void)hipFree(s->d_env_cdf);
        s->d_env = nullptr;
        s->d_env_cdf = nullptr;
        s->ds.env_tex = nullptr;
        s->ds.env_cdf = s->ds.env_pdf = nullptr;
        s->ds.env_w = s->ds.env_h = 0;
        return rebuild_light_select(s, false);
    }
    if (height == 0 || width != 2 * height) return set_error(WR_ERR_INVALID_ARGUMENT, "envmap has wrong size");
    if (uint64_t(width) * height > (uint64_t(1) << 26)) return set_error(WR_ERR_UNSUPPORTED, "envmap too large");
    const size_t n = size_t(width) * height;
    std::vector<float4> tex(n);
    std::vector<double> w(n);
    double sum = 0.0;
    for (uint32_t y = 0; y < height; y++) {
        const double sine = std::sin((double(y) + 0.5) / height * 3.14159265358979323846);
        for (uint32_t x = 0; x < width; x++) {
            const size_t i = size_t(y) * width + x;
            const float *t = rgb + 3 * i;
            for (int c = 0; c < 3; c++)
                if (!(t[c] >= 0.f) || !std::isfinite(t[c]))
                    return set_error(WR_ERR_INVALID_ARGUMENT, "envmap texels must be finite and >= 0");
            tex[i] = make_float4(t[0], t[1], t[2], 0.f);
            // EquiRectRep's texel weight: sin(theta) |rgb|_2 (equirectangular.h:40-58)
            w[i] = sine * std::sqrt(double(t[0]) * t[0] + double(t[1]) * t[1] + double(t[2]) * t[2]);
            sum += w[i];
        }
    }
    if (!(sum > 0.0)) return set_error(WR_ERR_INVALID_ARGUMENT, "envmap is black");
    std::vector<float> cp(2 * n);  // cdf, then pdf (CdfTable in FP64, rounded)
    double cdf = 0.0;
    for (size_t i = 0; i < n; i++) {
        const double pdf = w[i] / sum;
        cdf += pdf;
        cp[i] = i + 1 == n ? 1.0f : float(cdf);
        cp[n + i] = float(pdf);
    }
    float4 *d_tex = nullptr;
    float *d_cp = nullptr;
    uint64_t bytes = 0;
    rc = upload(s->dev, &d_tex, tex.data(), sizeof(float4) * n, bytes);
    if (!rc) rc = upload(s->dev, &d_cp, cp.data(), sizeof(float) * 2 * n, bytes);
    if (rc) {
        (void)hipFree(d_tex);
        return rc;
    }
    (void)hipFree(s->d_env);
    (void)hipFree(s->d_env_cdf);
    s->d_env = d_tex;
    s->d_env_cdf = d_cp;
    s->ds.env_tex = d_tex;
    s->ds.env_cdf = d_cp;
    s->ds.env_pdf = d_cp + n;
    s->ds.env_w = int(width);
    s->ds.env_h = int(height);
    return rebuild_light_select(s, true);
}

int wr_film_create(wr_scene *s, wr_film **out) {
    if (!s || !out) return set_error(WR_ERR_INVALID_ARGUMENT, "null argument");
    *out = nullptr;
    int rc = set_device(s->dev);
    if (rc) return rc;
    wr_film *f = new wr_film;
    f->scene = s;
    f->W = s->W;
    f->H = s->H;
    const size_t bytes = sizeof(double) * 3 * size_t(f->W) * f->H;
    hipError_t e = s->dev->alloc(reinterpret_cast<void **>(&f->d_base), bytes);
    if (e == hipSuccess) e = s->dev->alloc(reinterpret_cast<void **>(&f->d_splat), bytes);
    if (e != hipSuccess) {
        (void)hipFree(f->d_base);
        delete f;
        return set_error(e == hipErrorOutOfMemory ? WR_ERR_OUT_OF_MEMORY : WR_ERR_DEVICE, hipGetErrorString(e));
    }
    *out = f;
    return wr_film_clear(f);
}

void wr_film_destroy(wr_film *f) {
    if (!f) return;
    (void)hipSetDevice(f->scene->dev->ordinal);
    (void)hipStreamSynchronize(f->scene->stream);
    (void)hipFree(f->d_base);
    (void)hipFree(f->d_splat);
    delete f;
}

int wr_film_clear(wr_film *f) {
    if (!f) return set_error(WR_ERR_INVALID_ARGUMENT, "film is null");
    int rc = set_device(f->scene->dev);
    if (rc) return rc;
    const size_t n = 3 * size_t(f->W) * f->H;
    k_fill_f64<<<uint32_t(std::min<size_t>((n + 255) / 256, 1024)), 256, 0, f->scene->stream>>>(f->d_base, f->d_splat, n);
    WR_HIP(hipGetLastError());
    WR_HIP(hipStreamSynchronize(f->scene->stream));
    return WR_OK;
}

int wr_film_read(wr_film *f, double *base, double *splat) {
    if (!f) return set_error(WR_ERR_INVALID_ARGUMENT, "film is null");
    wr_device *dev = f->scene->dev;
    int rc = set_device(dev);
    if (rc) return rc;
    const size_t bytes = sizeof(double) * 3 * size_t(f->W) * f->H;
    hipStream_t st = f->scene->stream;
    WR_HIP(dev->ring.download(dev->ordinal, st, {{base, f->d_base, base ? bytes : 0}, {splat, f->d_splat, splat ? bytes : 0}}));
    WR_HIP(hipStreamSynchronize(st));
    return WR_OK;
}

int wr_film_image(wr_film *f, double base_div, double splat_div, double *rgb) {
    if (!f || !rgb) return set_error(WR_ERR_INVALID_ARGUMENT, "null argument");
    wr_device *dev = f->scene->dev;
    int rc = set_device(dev);
    if (rc) return rc;
    const size_t bytes = sizeof(double) * 3 * size_t(f->W) * f->H;
    hipStream_t st = f->scene->stream;
    WR_HIP(dev->ring.download(dev->ordinal, st, rgb, bytes, [&](size_t off, size_t n, char *slot) {
        const size_t first = off / sizeof(double);
        const uint32_t count = uint32_t(n / sizeof(double));
        k_film_image<<<(count + 255) / 256, 256, 0, st>>>(f->d_base + first, f->d_splat + first, base_div, splat_div,
                                                          reinterpret_cast<double *>(slot), count);
        return hipGetLastError();
    }));
    return WR_OK;
}

// Path pool: two queue-ordered states of 16*4 + 4 bytes per path (ray_o, ray_d,
// thr, rad, rec), the hit records (8 B), two shadow entries (2 * 48 B), and
// the per-sample radiance of a pass (16 B per sample).
// Byte layout of a path pool of `cap` paths and `samples` per-sample slots
// (every array 256-byte aligned): the state pair, hits, per-sample radiance,
// shadow queue (2 entries per path), counters (one 256-byte line each), stats.
constexpr size_t pool_bytes(size_t cap, size_t samples) {
    return 8 * align256(16 * cap) + 2 * align256(4 * cap) + align256(8 * cap) + align256(16 * samples) + 3 * align256(32 * cap) +
           align256(4 * kCounterStride * kNumCounterLines) + align256(64);
}
// Points pb's arrays into the pool at `base`; returns the bytes used (pool_bytes).
static size_t pool_layout(char *base, uint32_t cap, uint32_t samples, PathBuffers *pb) {
    const size_t c = cap;
    size_t off = 0;
    auto take = [&](size_t bytes) { char *q = base + off; off += align256(bytes); return q; };
    PathState *sts[2] = {&pb->cur, &pb->next};
    for (PathState *st : sts) {
        st->ray_o = reinterpret_cast<float4 *>(take(16 * c));
        st->ray_d = reinterpret_cast<float4 *>(take(16 * c));
        st->thr = reinterpret_cast<float4 *>(take(16 * c));
        st->rad = reinterpret_cast<float4 *>(take(16 * c));
        st->rec = reinterpret_cast<uint32_t *>(take(4 * c));
    }
    pb->hit = reinterpret_cast<uint2 *>(take(8 * c));
    pb->sample_rad = reinterpret_cast<float4 *>(take(16 * size_t(samples)));
    pb->sh_o = reinterpret_cast<float4 *>(take(32 * c));
    pb->sh_d = reinterpret_cast<float4 *>(take(32 * c));
    pb->sh_c = reinterpret_cast<float4 *>(take(32 * c));
    pb->counters = reinterpret_cast<uint32_t *>(take(4 * kCounterStride * kNumCounterLines));
    pb->cur.shadow_count = kShadowA;
    pb->next.shadow_count = kShadowB;
    pb->stats = reinterpret_cast<unsigned long long *>(take(64));
    return off;
}

static unsigned long long *progress_word(wr_scene *s) {
    return reinterpret_cast<unsigned long long *>(s->h_counters + kCounterStride * kNumCounterLines);
}

static int ensure_capacity(wr_scene *s, uint32_t cap, uint32_t samples) {
    if (s->capacity >= cap && s->sample_capacity >= samples) return WR_OK;
    // first: a scene with a capacity has the counters' copy and the progress word, which the device writes
    if (!s->h_counters) {
        void *p = nullptr;
        WR_HIP(hipHostMalloc(&p, sizeof(uint32_t) * kCounterStride * (kNumCounterLines + 1), hipHostMallocDefault));
        s->h_counters = static_cast<uint32_t *>(p);
        *progress_word(s) = 0;
    }
    cap = std::max(cap, s->capacity);
    samples = std::max(samples, s->sample_capacity);
    if (s->pool) {
        WR_HIP(hipStreamSynchronize(s->stream));
        WR_HIP(hipFree(s->pool));
        s->pool = nullptr;
        s->capacity = 0;
        s->sample_capacity = 0;
    }
    char *p = nullptr;
    WR_HIP(s->dev->alloc(reinterpret_cast<void **>(&p), pool_bytes(cap, samples)));
    s->pool = p;
    pool_layout(p, cap, samples, &s->pb);
    s->capacity = cap;
    s->sample_capacity = samples;
    return WR_OK;
}

static int grid_for(const wr_scene *s, uint32_t n, int per_cu) {
    const uint32_t blocks = (n + kBlock - 1) / kBlock;
    return int(std::max<uint32_t>(1, std::min<uint32_t>(blocks, uint32_t(s->dev->n_cu) * per_cu)));
}
// Traversal grids index the spill region by block, so they never exceed max_trav_blocks.
static int trav_grid(const wr_scene *s, uint32_t n, int per_cu) {
    return std::min(grid_for(s, n, std::min(per_cu, kMaxTraversalBlocksPerCU)), s->max_trav_blocks);
}

// Samples of one pass: bounds the per-sample radiance buffer to 2 GiB, enough
// for a 1920x1080 frame at 64 spp, so such a frame drains the pool once.
constexpr uint64_t kMaxSamplesPerPass = uint64_t(1) << 27;
// Paths in flight when the caller leaves max_paths_in_flight at 0.
constexpr uint64_t kDefaultPool = uint64_t(1) << 27;
// The default pool of a scene whose pool has to grow: `want` paths, but no
// more than a quarter of the device memory that is free (counting the scene's
// current pool, which the growth releases, and the blocks that the device handle
// holds idle, which an allocation gets where memory runs out) -- many scenes can then keep their
// pools in one process -- and never below the current pool or 2^20 paths.
static uint64_t default_pool_fit(const wr_scene *s, uint64_t want, uint64_t samples) {
    if (want <= s->capacity && samples <= s->sample_capacity) return want;
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) return want;
    uint64_t avail = free_b + s->dev->idle() + (s->pool ? pool_bytes(s->capacity, s->sample_capacity) : 0);
    const uint64_t per_path = pool_bytes(1 << 20, 0) >> 20;
    const uint64_t budget = avail / 4 > 16 * samples ? (avail / 4 - 16 * samples) / per_path : 0;
    const uint64_t floor = std::min<uint64_t>(want, std::max<uint64_t>(s->capacity, uint64_t(1) << 20));
    return std::max(floor, std::min(want, budget));
}

// Runs wavefront iterations until the pool drains and both shadow queues are
// traced.  launch(pb) issues one iteration (refill, one traversal launch for
// the closest-hit rays and the previous shadow queue, shade) for the state pb;
// without `progress` the host polls the device counters every kPoll iterations.  With a graph, the two
// iterations of a state round trip (cur -> next -> cur) are captured once and
// replayed, so a pass costs one graph launch per two iterations.  Every
// kernel reads its work counts from device memory, which is what makes the
// replays valid; nothing in an iteration is a memset.
//
// With `progress` (the pinned word that end_iteration writes) the host follows
// the pass without stopping it: it keeps kAhead iterations enqueued and reads
// the word, where a poll copies the counters and waits for the stream.
template <class Launch>
static int drain(wr_scene *s, PathBuffers &pb, uint64_t max_iters, bool use_graph, uint32_t *host_counters,
                 const volatile unsigned long long *progress, uint32_t tag, Launch &&launch) {
    constexpr int kPoll = 4;
    constexpr uint64_t kAhead = 4;
    auto poll = [&](bool &done) -> int {
        WR_HIP(hipMemcpyAsync(host_counters, pb.counters, sizeof(uint32_t) * kCounterStride * kNumCounterLines,
                              hipMemcpyDeviceToHost, s->stream));
        WR_HIP(hipStreamSynchronize(s->stream));
        // done: no path left and both shadow queues traced
        done = host_counters[kQ] == 0 && host_counters[kFresh] == 0 && host_counters[kShadowA] == 0 &&
               host_counters[kShadowB] == 0;
        return WR_OK;
    };
    if (!use_graph) {
        for (uint64_t it = 0;; it++) {
            if (it > max_iters) return set_error(WR_ERR_DEVICE, "path pool did not drain");
            launch(pb, it == 0);
            WR_HIP(hipGetLastError());
            std::swap(pb.cur, pb.next);
            if (progress) {
                uint64_t ended = 0;
                for (uint32_t spin = 0;; spin++) {
                    const unsigned long long w = *progress;
                    if (uint32_t(w >> 32) == tag) {
                        if (w & 1u) return WR_OK;
                        ended = uint32_t(w) >> 1;
                    }
                    if (it + 1 < ended + kAhead) break;
                    // an idle stream has written its last word: one that still lags means a failed launch
                    if (spin % 4096 == 4095) {
                        const hipError_t q = hipStreamQuery(s->stream);
                        if (q == hipSuccess) {
                            const unsigned long long last = *progress;
                            if (uint32_t(last >> 32) != tag || (uint32_t(last) >> 1) < it + 1)
                                return set_error(WR_ERR_DEVICE, "the pass stopped making progress");
                        } else if (q != hipErrorNotReady) {
                            WR_HIP(q);
                        }
                    }
                }
            } else if (it % kPoll == kPoll - 1) {
                bool done = false;
                int rc = poll(done);
                if (rc) return rc;
                if (done) return WR_OK;
            }
        }
    }
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    WR_HIP(hipStreamBeginCapture(s->stream, hipStreamCaptureModeThreadLocal));
    PathBuffers swapped = pb;
    std::swap(swapped.cur, swapped.next);
    launch(pb, true);
    launch(swapped, true);
    const hipError_t launch_err = hipGetLastError();
    WR_HIP(hipStreamEndCapture(s->stream, &graph));
    int rc = WR_OK;
    if (launch_err != hipSuccess) rc = set_error(WR_ERR_DEVICE, std::string("launch in graph capture: ") + hipGetErrorString(launch_err));
    if (!rc && hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) != hipSuccess)
        rc = set_error(WR_ERR_DEVICE, "hipGraphInstantiate failed");
    for (uint64_t it = 0; !rc; it += 2) {
        if (it > max_iters) {
            rc = set_error(WR_ERR_DEVICE, "path pool did not drain");
            break;
        }
        if (hipGraphLaunch(exec, s->stream) != hipSuccess) {
            rc = set_error(WR_ERR_DEVICE, "hipGraphLaunch failed");
            break;
        }
        if (it % kPoll == kPoll - 2) {
            bool done = false;
            rc = poll(done);
            if (done) break;
        }
    }
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    return rc;  // an even number of iterations: pb is the current state again
}

// Largest traversal work chunk: every wave claims at least one chunk from a
// 32-bit work counter, so chunk x waves must stay far below 2^32 (a wrapped
// counter would hand out entries twice).
constexpr uint32_t kMaxFetchChunk = 4096;

int wr_render_params_validate(const wr_render_params *p) {
    if (!p) return set_error(WR_ERR_INVALID_ARGUMENT, "params is null");
    if (p->spp < 0) return set_error(WR_ERR_INVALID_ARGUMENT, "spp must be >= 0");
    if (p->first_sample < 0) return set_error(WR_ERR_INVALID_ARGUMENT, "first_sample must be >= 0");
    if (p->max_paths_in_flight < 0) return set_error(WR_ERR_INVALID_ARGUMENT, "max_paths_in_flight must be >= 0");
    if (p->fetch_chunk > kMaxFetchChunk)
        return set_error(WR_ERR_INVALID_ARGUMENT, "fetch_chunk must be 0 (default) or 1.." + std::to_string(kMaxFetchChunk));
    if (p->refill_lanes > 64) return set_error(WR_ERR_INVALID_ARGUMENT, "refill_lanes must be 0 (default) or 1..64");
    return WR_OK;
}

// Threads per block of the shade and regenerate kernels for a pool of `paths`:
// kShadeBlock, which halves the appends' atomics against 256, down to one wave
// where that spreads a small pool over more of the CUs.
static int shade_block(const wr_device *d, uint64_t paths) {
    int block = kShadeBlock;
    while (block > 64 && paths < uint64_t(d->n_cu) * block * 2) block /= 2;
    return block;
}

// Estimators of the frame loop.
enum Estimator { kEstNee, kEstPrimitive, kEstLight };
// A path pool and traversal spill region that the caller already holds (the
// allocation-free entry point's scratch): render_impl then allocates nothing.
struct FixedPool {
    PathBuffers pb;
    uint32_t capacity, sample_capacity;  // paths in flight, samples per pass
    uint2 *spill;                        // kSpillDepth entries per lane of trav_blocks blocks
    int trav_blocks;
};
// The frame loop of wr_render_nee, wr_render_guided (g non-null),
// wr_render_primitive, wr_render_light and wr_render_nee_noalloc (fixed).
static int render_impl(wr_scene *s, wr_film *f, const wr_render_params *prm, wr_guide *g, const wr_guided_params *gp,
                       wr_render_stats *stats, wr_guide_stats *gstats, Estimator est = kEstNee,
                       const FixedPool *fixed = nullptr) {
    if (!s || !f || !prm) return set_error(WR_ERR_INVALID_ARGUMENT, "null argument");
    if (f->scene != s) return set_error(WR_ERR_INVALID_ARGUMENT, "film belongs to another scene");
    if (int rc0 = wr_render_params_validate(prm)) return rc0;
    if (g && !gp) return set_error(WR_ERR_INVALID_ARGUMENT, "null guided parameters");
    if (g && guide_scene(g) != s) return set_error(WR_ERR_INVALID_ARGUMENT, "guide belongs to another scene");
    if (g && !(gp->guide_fraction >= 0.f && gp->guide_fraction < 1.f))
        return set_error(WR_ERR_INVALID_ARGUMENT, "guide_fraction must be in [0, 1)");
    const bool env = s->ds.env_select > 0.f;
    if (est != kEstPrimitive && s->ds.n_lights == 0 && !env) return set_error(WR_ERR_INVALID_ARGUMENT, "scene has no lights");
    if (env && est == kEstLight) return set_error(WR_ERR_UNSUPPORTED, "the light tracer does not support envmap lights");
    if (env && g) return set_error(WR_ERR_UNSUPPORTED, "guided rendering does not support envmap lights");
    if (env && s->ds.med.on) return set_error(WR_ERR_UNSUPPORTED, "an envmap with a medium is not supported");
    wr_guide_stats gst{};
    const auto t0 = std::chrono::steady_clock::now();
    wr_render_stats st{};
    int rc = set_device(s->dev);
    if (rc) return rc;
    const int N = prm->num_path_vertices;
    const uint32_t wh = uint32_t(s->W) * uint32_t(s->H);
    if (N <= 1 || prm->spp == 0) {  // pathnextevent.h:163
        if (stats) *stats = st;
        if (gstats) *gstats = gst;
        return WR_OK;
    }
    if (fixed) {
        // the pool is the caller's fixed region: nothing may grow, and nothing
        // that allocates (events for profiling, graph instantiation) may run
        if (prm->profile) return set_error(WR_ERR_UNSUPPORTED, "profile = 1 needs HIP events; the allocation-free entry point creates none");
        if (prm->use_graph) return set_error(WR_ERR_UNSUPPORTED, "use_graph = 1 instantiates a graph, which allocates");
        if (wh > fixed->sample_capacity)
            return set_error(WR_ERR_UNSUPPORTED, "frame of " + std::to_string(wh) + " pixels exceeds the allocation-free "
                             "pass capacity of " + std::to_string(fixed->sample_capacity) + " samples");
        if (uint64_t(prm->max_paths_in_flight) > fixed->capacity)
            return set_error(WR_ERR_UNSUPPORTED, "max_paths_in_flight exceeds the allocation-free pool of " +
                             std::to_string(fixed->capacity) + " paths");
    }
    uint64_t spp_cap = std::min<uint64_t>((fixed ? fixed->sample_capacity : kMaxSamplesPerPass) / wh, uint64_t(prm->spp));
    if (g && gp->spp_per_pass > 0) spp_cap = std::min<uint64_t>(spp_cap, gp->spp_per_pass);
    const uint32_t spp_pass = uint32_t(std::max<uint64_t>(1, spp_cap));
    const uint32_t samples_pass = spp_pass * wh;
    // default pool: 2^27 paths, a whole 1080p 64-spp pass (about 35 GB of state
    // at full size, capped by the pass): large launches hide the traversal
    // latency and shrink the per-launch tail (2^25 / 2^26 / 2^27 paths:
    // 5,090 / 5,308 / 5,442 Mrays/s on the 1.31M-triangle frame)
    uint64_t pool = prm->max_paths_in_flight > 0 ? uint64_t(prm->max_paths_in_flight) : kDefaultPool;
    if (fixed) pool = std::min<uint64_t>(pool, fixed->capacity);
    pool = std::min<uint64_t>(pool, samples_pass);
    if (!fixed && prm->max_paths_in_flight == 0) pool = default_pool_fit(s, pool, samples_pass);
    if (pool > (uint64_t(1) << 30)) return set_error(WR_ERR_UNSUPPORTED, "too many paths in flight");
    const uint32_t P = uint32_t(pool);
    uint32_t fixed_counters[kCounterStride * kNumCounterLines];  // host copy of the counters (fixed pool)
    uint32_t *host_counters = fixed_counters;
    uint2 *spill = s->d_spill;
    if (fixed) {
        spill = fixed->spill;
    } else {
        rc = ensure_capacity(s, P, samples_pass);
        if (rc) return rc;
        host_counters = s->h_counters;
    }
    if (g) {
        rc = guide_reserve_draws(g, P);
        if (!rc) rc = guide_render_begin(g);
        if (rc) return rc;
    }
    PathBuffers pb = fixed ? fixed->pb : s->pb;
    pb.film_base = f->d_base;
    pb.film_splat = f->d_splat;
    k_fill_u32<<<1, 64, 0, s->stream>>>(reinterpret_cast<uint32_t *>(pb.stats), 0u, 12);
    WR_HIP(hipGetLastError());
    const bool prof = prm->profile != 0;
    const bool count = prm->count_traversal != 0;
    // per-kernel profiling records events between launches, which a graph cannot hold
    const bool use_graph = prm->use_graph != 0 && !prof;
    TravTune tune;
    if (prm->fetch_chunk) tune.chunk = prm->fetch_chunk;
    if (prm->refill_lanes) tune.refill = prm->refill_lanes;
    std::vector<hipEvent_t> evs;
    struct Mark { int kind; size_t e0; };
    std::vector<Mark> marks;
    auto ev_record = [&]() -> size_t {
        hipEvent_t e;
        (void)hipEventCreate(&e);
        (void)hipEventRecord(e, s->stream);
        evs.push_back(e);
        return evs.size() - 1;
    };
    auto begin = [&](int kind) { if (prof) marks.push_back({kind, ev_record()}); };
    auto end = [&]() { if (prof) ev_record(); };
    const int bs = shade_block(s->dev, P);
    const int g_regen = std::max(1, std::min<int>((P + bs - 1) / bs, s->dev->n_cu * s->dev->occ_generate * (kShadeBlock / bs)));
    // shading kernel: plain, or extended for guiding and/or a medium
    // the light tracer's sampler is not volumetric (lightsplatting.h:34): it sees vacuum
    DScene ds = s->ds;
    if (est == kEstLight) ds.med.on = 0;
    const bool medium = ds.med.on != 0;
    const void *shade_fn = est == kEstLight ? reinterpret_cast<const void *>(&k_shade_light)
                           : env            ? reinterpret_cast<const void *>(&k_shade<false, true>)
                                            : reinterpret_cast<const void *>(&k_shade<false>);
    if (g && medium) shade_fn = reinterpret_cast<const void *>(&k_shade_ext<true, true>);
    else if (g) shade_fn = reinterpret_cast<const void *>(&k_shade_ext<true, false>);
    else if (medium) shade_fn = reinterpret_cast<const void *>(&k_shade_ext<false, true>);
    const int g_shade = std::max(1, std::min<int>((P + bs - 1) / bs, s->dev->n_cu * occupancy(s->dev, shade_fn, kShadeBlock) *
                                                                         (kShadeBlock / bs)));
    int pass = 0;
    const bool fp8 = g && gp->fp8_inference != 0;
    const void *infer_fn = medium ? (fp8 ? reinterpret_cast<const void *>(&k_guide_infer<true, true>)
                                         : reinterpret_cast<const void *>(&k_guide_infer<true, false>))
                                  : (fp8 ? reinterpret_cast<const void *>(&k_guide_infer<false, true>)
                                         : reinterpret_cast<const void *>(&k_guide_infer<false, false>));
    const int g_infer = std::max(1, std::min<int>((P + kInferBlock - 1) / kInferBlock,
                                                  s->dev->n_cu * occupancy(s->dev, infer_fn, kInferBlock)));
    // passes that k_small_pass takes: the plain estimators, unless traversal
    // counters, per-kernel times or graph replays of the iterations are asked for.
    // A path's bounce is kept in 8 bits: with more vertices than that nothing but
    // the limit on iterations ends the paths of a closed scene, and only the
    // queues have one.
    const bool small_passes = est != kEstLight && !g && !medium && !count && !prof && !use_graph && N <= int(kBounceMask);
    const void *small_fn = env ? reinterpret_cast<const void *>(&k_small_pass<true>) : reinterpret_cast<const void *>(&k_small_pass<false>);
    const uint32_t small_blocks = uint32_t(s->dev->n_cu * occupancy(s->dev, small_fn, 2 * kBlock));
    const uint32_t small_slices = uint32_t(fixed ? fixed->trav_blocks : s->max_trav_blocks) / 2;
    guide::Net net{};
    // up to P closest-hit rays and 2P shadow rays (one per path and one per new sample)
    int g_trav = trav_grid(s, 2 * P, s->dev->occ_rays);
    if (fixed) g_trav = std::min(g_trav, fixed->trav_blocks);  // the fixed spill region covers trav_blocks blocks
    for (uint32_t done = 0; done < uint32_t(prm->spp); done += spp_pass) {
        const uint32_t k = std::min<uint32_t>(spp_pass, uint32_t(prm->spp) - done);
        RenderArgs a;
        a.total = k * wh;
        a.wh = wh;
        a.first_sample = uint32_t(prm->first_sample) + done;
        a.seed = prm->seed;
        a.capacity = P;
        a.N = N;
        a.use_mis = est == kEstNee && prm->use_mis ? 1 : 0;
        a.nee = est == kEstNee ? 1 : 0;
        a.guided = g ? 1 : 0;
        a.tag = ++s->pass_tag;
        a.progress = fixed || use_graph ? nullptr : progress_word(s);
        a.light = est == kEstLight ? 1 : 0;
        guide::Shade gs{};
        float record_prob = 0.f;
        const bool collect = g && gp->train_steps > 0;
        const int set = pass & 1;  // record set and inference copy of this pass
        if (g) {
            rc = guide_pass_net(g, set, gp->overlap_training != 0, &net);
            if (!rc && collect) rc = guide_begin_pass(g, set, a.total, &record_prob);
            if (rc) return rc;
            const bool sample_net = pass >= int(gp->warmup_passes);
            rc = guide_shade_view(g, set, sample_net ? gp->guide_fraction : 0.f, record_prob, collect,
                                  gp->max_guided_bounce ? gp->max_guided_bounce : 0xFFFFFFFFu, &gs);
            if (rc) return rc;
        }
        const uint32_t tiles = (a.total + kBlock - 1) / kBlock;
        const bool small = small_passes && a.total <= P &&
                           (tiles <= small_slices || (!fixed && a.total <= small_pass_samples(s->n_tris)));
        if (small) {
            // a tile per block as long as there are spill slices, else resident blocks with equal shares
            const uint32_t grid = tiles <= small_slices ? tiles : std::min(small_blocks, small_slices);
            const uint32_t per_block = tiles <= small_slices ? kBlock : (a.total + grid - 1) / grid;
            if (env) k_small_pass<true><<<grid, 2 * kBlock, 0, s->stream>>>(ds, pb, a, per_block, spill);
            else k_small_pass<false><<<grid, 2 * kBlock, 0, s->stream>>>(ds, pb, a, per_block, spill);
        } else {
            k_init<<<1, 64, 0, s->stream>>>(pb, a);
        }
        WR_HIP(hipGetLastError());
        // Each iteration refills the pool, extends every active path by one
        // vertex and resolves the shadow rays of the previous iteration's
        // vertices (so the last shadow queue takes one iteration more);
        // iterations past the end find empty queues.  Every path ends within
        // N-1 vertices, and each iteration that is not draining starts new
        // samples in all free entries.
        const uint64_t max_iters = (uint64_t(a.total) / P + 2) * uint64_t(N + 1) + 64;
        // a pool that holds the whole pass is filled by the first iteration's regeneration
        const bool refills = a.total > P;
        auto iteration = [&](const PathBuffers &q, bool first) {
            begin(3);
            if (!first && !refills) {}
            else if (env) k_regen<false, true><<<g_regen, bs, 0, s->stream>>>(ds, nullptr, 0, q, a);
            else k_regen<false><<<g_regen, bs, 0, s->stream>>>(ds, nullptr, 0, q, a);
            end();
            begin(0);
            if (count) k_trace_bounce<true, false><<<g_trav, kBlock, 0, s->stream>>>(ds, nullptr, q, spill, tune);
            else k_trace_bounce_fast<<<g_trav, kBlock, 0, s->stream>>>(ds, q, spill, tune);
            end();
            begin(2);
            if (g && gs.alpha > 0.f) {
                if (medium && fp8)
                    k_guide_infer<true, true><<<g_infer, kInferBlock, 0, s->stream>>>(ds, q.cur, q.hit, q.counters, N,
                                                                                      net, gs.alpha, gs.max_bounce, gs.draw);
                else if (medium)
                    k_guide_infer<true, false><<<g_infer, kInferBlock, 0, s->stream>>>(ds, q.cur, q.hit, q.counters, N,
                                                                                       net, gs.alpha, gs.max_bounce, gs.draw);
                else if (fp8)
                    k_guide_infer<false, true><<<g_infer, kInferBlock, 0, s->stream>>>(ds, q.cur, q.hit, q.counters, N,
                                                                                       net, gs.alpha, gs.max_bounce, gs.draw);
                else
                    k_guide_infer<false, false><<<g_infer, kInferBlock, 0, s->stream>>>(ds, q.cur, q.hit, q.counters, N,
                                                                                        net, gs.alpha, gs.max_bounce, gs.draw);
            }
            if (g && medium) k_shade_ext<true, true><<<g_shade, bs, 0, s->stream>>>(ds, q, a, gs);
            else if (g) k_shade_ext<true, false><<<g_shade, bs, 0, s->stream>>>(ds, q, a, gs);
            else if (medium) k_shade_ext<false, true><<<g_shade, bs, 0, s->stream>>>(ds, q, a, gs);
            else if (est == kEstLight) k_shade_light<<<g_shade, bs, 0, s->stream>>>(ds, q, a);
            else if (env) k_shade<false, true><<<g_shade, bs, 0, s->stream>>>(ds, nullptr, q, a);
            else k_shade<false><<<g_shade, bs, 0, s->stream>>>(ds, nullptr, q, a);
            end();
        };
        rc = small ? WR_OK : drain(s, pb, max_iters, use_graph, host_counters, a.progress, a.tag, iteration);
        if (rc) return rc;
        begin(4);
        k_accumulate<<<std::max<uint32_t>(1, std::min<uint32_t>((wh + 255) / 256, uint32_t(s->dev->n_cu) * 8)), 256, 0,
                       s->stream>>>(pb.sample_rad, pb.film_base, wh, k);
        end();
        WR_HIP(hipGetLastError());
        if (collect) {
            rc = guide_end_pass(g, set, pb.sample_rad, a.total, record_prob, gp->train_steps, &gst);
            if (rc) return rc;
        }
        pass++;
    }
    if (g) {
        rc = guide_render_end(g, &gst);
        if (rc) return rc;
    }
    unsigned long long hs[6] = {0};
    WR_HIP(hipMemcpyAsync(hs, pb.stats, sizeof hs, hipMemcpyDeviceToHost, s->stream));
    WR_HIP(hipStreamSynchronize(s->stream));
    st.paths = uint64_t(prm->spp) * wh;
    st.extend_rays = hs[0];
    st.shadow_rays = hs[1];
    st.extend_nodes = hs[2];
    st.extend_tris = hs[3];
    st.shadow_nodes = hs[4];
    st.shadow_tris = hs[5];
    if (prof) {
        for (const Mark &m : marks) {
            float ms = 0.f;
            (void)hipEventElapsedTime(&ms, evs[m.e0], evs[m.e0 + 1]);
            switch (m.kind) {
            case 0: st.extend_ms += ms; st.extend_launches++; break;
            case 1: st.shadow_ms += ms; st.shadow_launches++; break;
            case 2: st.shade_ms += ms; break;
            case 3: st.generate_ms += ms; break;
            default: st.accumulate_ms += ms; break;
            }
        }
    }
    for (hipEvent_t e : evs) (void)hipEventDestroy(e);
    st.wall_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    if (stats) *stats = st;
    if (gstats) *gstats = gst;
    return WR_OK;
}

int wr_render_nee(wr_scene *s, wr_film *f, const wr_render_params *prm, wr_render_stats *stats) {
    return render_impl(s, f, prm, nullptr, nullptr, stats, nullptr);
}

// ============================================================== allocation-free NEE + MIS
// wr_render_nee_noalloc renders through a fixed region of device memory that
// the library reserves once per GPU instead of the scene's lazily grown path
// pool: a pool of 2^17 paths with 2^20 per-sample slots (passes of at most
// 2^20 samples) and the traversal spill of 1024 blocks -- 74 MiB, held by each
// GPU the library runs on until the process ends.  The region is a file-scope
// device array; its device address on each GPU comes from hipGetSymbolAddress
// at wr_device_create (the array's name in host code is not a device address).
constexpr uint32_t kFixedPaths = 1u << 17;
constexpr uint32_t kFixedSamples = 1u << 20;
constexpr int kFixedTravBlocks = 1024;
constexpr size_t kFixedPoolBytes = pool_bytes(kFixedPaths, kFixedSamples);
constexpr size_t kFixedSpillBytes = sizeof(uint2) * size_t(kFixedTravBlocks) * kBlock * kSpillDepth;
constexpr size_t kScratchBytes = kFixedPoolBytes + kFixedSpillBytes;
static_assert(kFixedPoolBytes % 256 == 0, "the spill region starts 256-byte aligned");
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// Device address of `scratch` on the device current in wr_device_create.
static int scratch_setup(wr_device *d) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
        return set_error(WR_ERR_DEVICE, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    d->scratch = ptr;
    return WR_OK;
}

int wr_render_nee_noalloc(wr_scene *s, wr_film *f, const wr_render_params *prm, wr_render_stats *stats) {
    if (!s || !f || !prm) return set_error(WR_ERR_INVALID_ARGUMENT, "null argument");
    if (!s->dev->scratch) return set_error(WR_ERR_DEVICE, "the device has no scratch region");
    char *base = static_cast<char *>(s->dev->scratch);
    FixedPool fp{};
    pool_layout(base, kFixedPaths, kFixedSamples, &fp.pb);
    fp.capacity = kFixedPaths;
    fp.sample_capacity = kFixedSamples;
    fp.spill = reinterpret_cast<uint2 *>(base + kFixedPoolBytes);
    fp.trav_blocks = kFixedTravBlocks;
    return render_impl(s, f, prm, nullptr, nullptr, stats, nullptr, kEstNee, &fp);
}

int wr_render_guided(wr_scene *s, wr_film *f, wr_guide *g, const wr_render_params *prm, const wr_guided_params *gp,
                     wr_render_stats *stats, wr_guide_stats *gstats) {
    if (!g) return set_error(WR_ERR_INVALID_ARGUMENT, "guide is null");
    return render_impl(s, f, prm, g, gp, stats, gstats);
}

int wr_render_primitive(wr_scene *s, wr_film *f, const wr_render_params *prm, wr_render_stats *stats) {
    return render_impl(s, f, prm, nullptr, nullptr, stats, nullptr, kEstPrimitive);
}

int wr_render_light(wr_scene *s, wr_film *f, const wr_render_params *prm, wr_render_stats *stats) {
    return render_impl(s, f, prm, nullptr, nullptr, stats, nullptr, kEstLight);
}

int wr_render_visualize(wr_scene *s, wr_film *f, const wr_render_params *prm, wr_render_stats *stats) {
    if (!s || !f || !prm) return set_error(WR_ERR_INVALID_ARGUMENT, "null argument");
    if (f->scene != s) return set_error(WR_ERR_INVALID_ARGUMENT, "film belongs to another scene");
    if (int rc0 = wr_render_params_validate(prm)) return rc0;
    const auto t0 = std::chrono::steady_clock::now();
    int rc = set_device(s->dev);
    if (rc) return rc;
    wr_render_stats st{};
    const uint32_t wh = uint32_t(s->W) * uint32_t(s->H);
    if (prm->spp > 0) {
        // as many blocks as there are spill slices, 8,192, of which 5,120 are resident: the 1.31M-triangle scene
        // at 1920 x 1080 takes 323 us (7,168, the residency of k_trace: 372), at 1280 x 720 187 (5,120: 234)
        const int grid = trav_grid(s, wh, kMaxTraversalBlocksPerCU);
        if (prm->profile) WR_HIP(hipEventRecord(s->ev[0], s->stream));
        k_visualize<<<grid, kBlock, 0, s->stream>>>(s->ds, wh, uint32_t(prm->spp), uint32_t(prm->first_sample),
                                                    prm->seed, f->d_base, s->d_spill);
        WR_HIP(hipGetLastError());
        if (prm->profile) WR_HIP(hipEventRecord(s->ev[1], s->stream));
        WR_HIP(hipStreamSynchronize(s->stream));
        if (prm->profile) {
            float ms = 0.f;
            WR_HIP(hipEventElapsedTime(&ms, s->ev[0], s->ev[1]));
            st.extend_ms = ms;
            st.extend_launches = 1;
        }
    }
    st.paths = uint64_t(prm->spp) * wh;
    st.extend_rays = st.paths;
    st.wall_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    if (stats) *stats = st;
    return WR_OK;
}

int wr_render_bdpt(wr_scene *s, wr_film *f, const wr_render_params *prm, wr_render_stats *stats) {
    if (!s || !f || !prm) return set_error(WR_ERR_INVALID_ARGUMENT, "null argument");
    if (f->scene != s) return set_error(WR_ERR_INVALID_ARGUMENT, "film belongs to another scene");
    if (int rc0 = wr_render_params_validate(prm)) return rc0;
    const auto t0 = std::chrono::steady_clock::now();
    wr_render_stats st{};
    const int N = prm->num_path_vertices;
    if (N <= 1 || prm->spp == 0) {  // BidirPathRenderer::render returns at once for N <= 1 (bidirpath.h:318)
        st.wall_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
        if (stats) *stats = st;
        return WR_OK;
    }
    if (N > kBdptMaxVertices) return set_error(WR_ERR_UNSUPPORTED, "bidirectional path tracing supports at most 64 path vertices");
    if (s->ds.n_lights == 0) return set_error(WR_ERR_INVALID_ARGUMENT, "scene has no lights");
    if (s->ds.env_select > 0.f) return set_error(WR_ERR_UNSUPPORTED, "the bidirectional path tracer does not support envmap lights");
    int rc = set_device(s->dev);
    if (rc) return rc;
    const uint32_t wh = uint32_t(s->W) * uint32_t(s->H);
    const int grid = trav_grid(s, wh, occupancy(s->dev, reinterpret_cast<const void *>(&k_bdpt), kBlock));
    // records of N - 1 light vertices per lane, behind 256 bytes of counters
    const size_t need = 256 + sizeof(float4) * 4 * size_t(N - 1) * size_t(grid) * kBlock;
    if (need > s->bdpt_bytes) {
        WR_HIP(hipStreamSynchronize(s->stream));
        (void)hipFree(s->d_bdpt);
        s->device_bytes -= s->bdpt_bytes;
        s->d_bdpt = nullptr;
        s->bdpt_bytes = 0;
        WR_HIP(s->dev->alloc(reinterpret_cast<void **>(&s->d_bdpt), need));
        s->bdpt_bytes = need;
        s->device_bytes += need;
    }
    auto *counts = reinterpret_cast<unsigned long long *>(s->d_bdpt);
    WR_HIP(hipMemsetAsync(counts, 0, 16, s->stream));
    // the medium is not passed on: the reference's subpath sampler here is not volumetric
    DScene ds = s->ds;
    ds.med.on = 0;
    if (prm->profile) WR_HIP(hipEventRecord(s->ev[0], s->stream));
    k_bdpt<<<grid, kBlock, 0, s->stream>>>(ds, wh, uint32_t(prm->spp), uint32_t(prm->first_sample), prm->seed, N,
                                           f->d_base, f->d_splat, s->d_bdpt + 16, counts, s->d_spill);
    WR_HIP(hipGetLastError());
    if (prm->profile) WR_HIP(hipEventRecord(s->ev[1], s->stream));
    unsigned long long h[2] = {0, 0};
    WR_HIP(hipMemcpyAsync(h, counts, sizeof h, hipMemcpyDeviceToHost, s->stream));
    WR_HIP(hipStreamSynchronize(s->stream));
    if (prm->profile) {
        float ms = 0.f;
        WR_HIP(hipEventElapsedTime(&ms, s->ev[0], s->ev[1]));
        st.extend_ms = ms;
        st.extend_launches = 1;
    }
    st.paths = uint64_t(prm->spp) * wh;
    st.extend_rays = h[0];
    st.shadow_rays = h[1];
    st.wall_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    if (stats) *stats = st;
    return WR_OK;
}

// ============================================================== batches (host)
int wr_render_batch(const wr_batch_job *jobs, uint32_t n_jobs, const wr_render_params *prm, wr_render_stats *stats) {
    if (!jobs || !prm) return set_error(WR_ERR_INVALID_ARGUMENT, "null argument");
    if (int rc0 = wr_render_params_validate(prm)) return rc0;
    if (n_jobs == 0) return set_error(WR_ERR_INVALID_ARGUMENT, "empty batch");
    if (n_jobs > uint32_t(kMaxBatchJobs)) return set_error(WR_ERR_UNSUPPORTED, "too many jobs in a batch");
    wr_scene *s0 = jobs[0].scene;
    for (uint32_t j = 0; j < n_jobs; j++) {
        const wr_batch_job &J = jobs[j];
        if (!J.scene || !J.film) return set_error(WR_ERR_INVALID_ARGUMENT, "batch job without scene or film");
        if (J.film->scene != J.scene) return set_error(WR_ERR_INVALID_ARGUMENT, "batch job film belongs to another scene");
        if (J.scene->dev != s0->dev) return set_error(WR_ERR_INVALID_ARGUMENT, "batch scenes on different devices");
        if (J.spp < 0 || J.first_sample < 0) return set_error(WR_ERR_INVALID_ARGUMENT, "negative spp or first_sample");
        if (J.num_path_vertices > int(kBounceMask)) return set_error(WR_ERR_UNSUPPORTED, "num_path_vertices above 255");
        if (uint64_t(J.scene->W) * J.scene->H > kMaxSamplesPerPass)
            return set_error(WR_ERR_UNSUPPORTED, "resolution too large for a batch pass");
        if (J.scene->ds.med.on) return set_error(WR_ERR_UNSUPPORTED, "batch scenes with a medium are not supported");
        if (J.scene->ds.n_lights == 0 && !(J.scene->ds.env_select > 0.f))
            return set_error(WR_ERR_INVALID_ARGUMENT, "scene has no lights");
    }
    const auto t0 = std::chrono::steady_clock::now();
    wr_render_stats st{};
    int rc = set_device(s0->dev);
    if (rc) return rc;
    std::vector<uint32_t> done(n_jobs, 0);
    uint64_t paths = 0, max_pass = 0;
    int maxN = 2;
    for (uint32_t j = 0; j < n_jobs; j++) {
        const uint64_t wh = uint64_t(jobs[j].scene->W) * jobs[j].scene->H;
        if (jobs[j].num_path_vertices > 1) {
            paths += wh * uint64_t(jobs[j].spp);
            maxN = std::max(maxN, jobs[j].num_path_vertices);
        }
        max_pass += wh * uint64_t(jobs[j].spp);
    }
    if (paths == 0) {
        if (stats) *stats = st;
        return WR_OK;
    }
    max_pass = std::min<uint64_t>(max_pass, kMaxSamplesPerPass);
    uint64_t pool = prm->max_paths_in_flight > 0 ? uint64_t(prm->max_paths_in_flight) : kDefaultPool;
    pool = std::min<uint64_t>(pool, max_pass);
    if (prm->max_paths_in_flight == 0) pool = default_pool_fit(s0, pool, max_pass);
    if (pool > (uint64_t(1) << 30)) return set_error(WR_ERR_UNSUPPORTED, "too many paths in flight");
    const uint32_t P = uint32_t(pool);
    rc = ensure_capacity(s0, P, uint32_t(max_pass));
    if (rc) return rc;
    PathBuffers pb = s0->pb;
    pb.film_base = nullptr;  // per job, from the table
    pb.film_splat = nullptr;
    BatchJob *d_tab = nullptr;
    WR_HIP(s0->dev->alloc(reinterpret_cast<void **>(&d_tab), sizeof(BatchJob) * n_jobs));
    struct Free { BatchJob *p; ~Free() { if (p) (void)hipFree(p); } } free_tab{d_tab};
    k_fill_u32<<<1, 64, 0, s0->stream>>>(reinterpret_cast<uint32_t *>(pb.stats), 0u, 12);
    WR_HIP(hipGetLastError());
    const bool prof = prm->profile != 0;
    const bool count = prm->count_traversal != 0;
    const bool use_graph = prm->use_graph != 0 && !prof;
    TravTune tune;
    if (prm->fetch_chunk) tune.chunk = prm->fetch_chunk;
    if (prm->refill_lanes) tune.refill = prm->refill_lanes;
    std::vector<hipEvent_t> evs;
    struct Mark { int kind; size_t e0; };
    std::vector<Mark> marks;
    auto ev_record = [&]() -> size_t {
        hipEvent_t e;
        (void)hipEventCreate(&e);
        (void)hipEventRecord(e, s0->stream);
        evs.push_back(e);
        return evs.size() - 1;
    };
    auto begin = [&](int kind) { if (prof) marks.push_back({kind, ev_record()}); };
    auto end = [&]() { if (prof) ev_record(); };
    wr_device *dev = s0->dev;
    const int bs = shade_block(dev, P);
    auto grid = [&](const void *fn) {
        return std::max(1, std::min<int>((P + bs - 1) / bs, dev->n_cu * occupancy(dev, fn, kShadeBlock) * (kShadeBlock / bs)));
    };
    bool env = false;
    for (uint32_t j = 0; j < n_jobs; j++) env = env || jobs[j].scene->ds.env_select > 0.f;
    const int g_regen = grid(env ? reinterpret_cast<const void *>(&k_regen<true, true>)
                                 : reinterpret_cast<const void *>(&k_regen<true>));
    const int g_shade = grid(env ? reinterpret_cast<const void *>(&k_shade<true, true>)
                                 : reinterpret_cast<const void *>(&k_shade<true>));
    const int g_trav =
        trav_grid(s0, 2 * P, occupancy(dev, reinterpret_cast<const void *>(&k_trace_bounce<false, true>), kBlock));
    std::vector<BatchJob> tab;
    for (;;) {
        // plan the pass: whole spp planes of each unfinished job, job-major, within the pass budget
        tab.clear();
        std::vector<uint32_t> tab_job;
        uint64_t budget = kMaxSamplesPerPass, offset = 0;
        for (uint32_t j = 0; j < n_jobs; j++) {
            const wr_batch_job &J = jobs[j];
            if (J.num_path_vertices <= 1 || done[j] >= uint32_t(J.spp)) continue;
            const uint32_t wh = uint32_t(J.scene->W) * uint32_t(J.scene->H);
            const uint32_t k = uint32_t(std::min<uint64_t>(uint64_t(J.spp) - done[j], budget / wh));
            if (k == 0) continue;
            BatchJob b{};
            b.s = J.scene->ds;
            b.offset = uint32_t(offset);
            b.count = k * wh;
            b.wh = wh;
            b.k = k;
            b.first_sample = uint32_t(J.first_sample) + done[j];
            b.seed = J.seed;
            b.N = J.num_path_vertices;
            b.use_mis = J.use_mis ? 1 : 0;
            b.film_base = J.film->d_base;
            b.film_splat = J.film->d_splat;
            tab.push_back(b);
            tab_job.push_back(j);
            offset += b.count;
            budget -= b.count;
        }
        if (tab.empty()) break;
        WR_HIP(hipMemcpyAsync(d_tab, tab.data(), sizeof(BatchJob) * tab.size(), hipMemcpyHostToDevice, s0->stream));
        RenderArgs a{};
        a.total = uint32_t(offset);
        a.capacity = P;
        a.N = maxN;
        a.nee = 1;
        a.tag = ++s0->pass_tag;
        a.progress = use_graph ? nullptr : progress_word(s0);
        const uint32_t nt = uint32_t(tab.size());
        k_init<<<1, 64, 0, s0->stream>>>(pb, a);
        WR_HIP(hipGetLastError());
        const uint64_t max_iters = (uint64_t(a.total) / P + 2) * uint64_t(maxN + 1) + 64;
        const bool refills = a.total > P;
        auto iteration = [&](const PathBuffers &q, bool first) {
            begin(3);
            if (!first && !refills) {}
            else if (env) k_regen<true, true><<<g_regen, bs, 0, s0->stream>>>(s0->ds, d_tab, nt, q, a);
            else k_regen<true><<<g_regen, bs, 0, s0->stream>>>(s0->ds, d_tab, nt, q, a);
            end();
            begin(0);
            if (count) k_trace_bounce<true, true><<<g_trav, kBlock, 0, s0->stream>>>(s0->ds, d_tab, q, s0->d_spill, tune);
            else k_trace_bounce<false, true><<<g_trav, kBlock, 0, s0->stream>>>(s0->ds, d_tab, q, s0->d_spill, tune);
            end();
            begin(2);
            if (env) k_shade<true, true><<<g_shade, bs, 0, s0->stream>>>(s0->ds, d_tab, q, a);
            else k_shade<true><<<g_shade, bs, 0, s0->stream>>>(s0->ds, d_tab, q, a);
            end();
        };
        rc = drain(s0, pb, max_iters, use_graph, s0->h_counters, a.progress, a.tag, iteration);
        if (rc) return rc;
        begin(4);
        for (uint32_t t = 0; t < nt; t++) {
            const BatchJob &b = tab[t];
            k_accumulate<<<std::max<uint32_t>(1, std::min<uint32_t>((b.wh + 255) / 256, uint32_t(dev->n_cu) * 8)), 256, 0,
                           s0->stream>>>(pb.sample_rad + b.offset, b.film_base, b.wh, b.k);
            done[tab_job[t]] += b.k;
        }
        end();
        WR_HIP(hipGetLastError());
    }
    unsigned long long hs[6] = {0};
    WR_HIP(hipMemcpyAsync(hs, pb.stats, sizeof hs, hipMemcpyDeviceToHost, s0->stream));
    WR_HIP(hipStreamSynchronize(s0->stream));
    st.paths = paths;
    st.extend_rays = hs[0];
    st.shadow_rays = hs[1];
    st.extend_nodes = hs[2];
    st.extend_tris = hs[3];
    st.shadow_nodes = hs[4];
    st.shadow_tris = hs[5];
    for (const Mark &m : marks) {
        float ms = 0.f;
        (void)hipEventElapsedTime(&ms, evs[m.e0], evs[m.e0 + 1]);
        switch (m.kind) {
        case 0: st.extend_ms += ms; st.extend_launches++; break;
        case 1: st.shadow_ms += ms; st.shadow_launches++; break;
        case 2: st.shade_ms += ms; break;
        case 3: st.generate_ms += ms; break;
        default: st.accumulate_ms += ms; break;
        }
    }
    for (hipEvent_t e : evs) (void)hipEventDestroy(e);
    st.wall_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    if (stats) *stats = st;
    return WR_OK;
}

int wr_autotune(const wr_batch_job *jobs, uint32_t n_jobs, const wr_render_params *base, wr_render_params *best,
                double *mrays) {
    if (!jobs || !base || !best) return set_error(WR_ERR_INVALID_ARGUMENT, "null argument");
    if (int rc0 = wr_render_params_validate(base)) return rc0;
    if (n_jobs == 0) return set_error(WR_ERR_INVALID_ARGUMENT, "empty batch");
    // trial jobs: 1 spp each into scratch films
    std::vector<wr_batch_job> trial(jobs, jobs + n_jobs);
    std::vector<wr_film *> films;
    int rc = WR_OK;
    for (auto &t : trial) {
        if (!t.scene) { rc = set_error(WR_ERR_INVALID_ARGUMENT, "batch job without scene"); break; }
        wr_film *f = nullptr;
        rc = wr_film_create(t.scene, &f);
        if (rc) break;
        films.push_back(f);
        t.film = f;
        t.spp = std::min(t.spp, 1);
    }
    struct Candidate { uint32_t pool, chunk, refill; int graph; };
    std::vector<Candidate> cands;
    for (uint32_t pool : {1u << 23, 1u << 24, 1u << 25, 1u << 26, 1u << 27})
        for (auto ck : {std::make_pair(96u, 16u), std::make_pair(256u, 16u), std::make_pair(128u, 32u), std::make_pair(256u, 32u)})
            for (int graph : {0, 1}) cands.push_back({pool, ck.first, ck.second, graph});
    double best_rate = -1.0;
    wr_render_params bp = *base;
    if (!rc) {
        wr_render_params warm = *base;
        warm.profile = 0;
        warm.count_traversal = 0;
        wr_render_stats ws;
        rc = wr_render_batch(trial.data(), n_jobs, &warm, &ws);  // allocations, first launches
    }
    for (size_t c = 0; !rc && c < cands.size(); c++) {
        wr_render_params p = *base;
        p.profile = 0;
        p.count_traversal = 0;
        p.max_paths_in_flight = int32_t(cands[c].pool);
        p.fetch_chunk = cands[c].chunk;
        p.refill_lanes = cands[c].refill;
        p.use_graph = cands[c].graph;
        wr_render_stats st;
        rc = wr_render_batch(trial.data(), n_jobs, &p, &st);
        if (rc) break;
        const double rate = double(st.extend_rays + st.shadow_rays) / (st.wall_ms * 1e-3) / 1e6;
        if (rate > best_rate) {
            best_rate = rate;
            bp = p;
        }
    }
    const std::string err = rc ? wr::error_string() : std::string();
    for (wr_film *f : films) wr_film_destroy(f);
    if (rc) {
        wr::error_string() = err;
        return rc;
    }
    bp.profile = base->profile;
    bp.count_traversal = base->count_traversal;
    *best = bp;
    if (mrays) *mrays = best_rate;
    return WR_OK;
}

static int trace_impl(wr_scene *s, const float *d_rays, uint32_t n, void *d_hits, uint8_t *d_occ, bool any, float *ms,
                      bool ids = false) {
    int rc = set_device(s->dev);
    if (rc) return rc;
    if (n == 0) { if (ms) *ms = 0.f; return WR_OK; }
    const void *fn = any ? reinterpret_cast<const void *>(&k_trace<true>)
                    : ids ? reinterpret_cast<const void *>(&k_trace<false, true>)
                          : reinterpret_cast<const void *>(&k_trace<false>);
    const int grid = trav_grid(s, n, occupancy(s->dev, fn, kBlock));
    if (ms) WR_HIP(hipEventRecord(s->ev[0], s->stream));
    const float4 *rays = reinterpret_cast<const float4 *>(d_rays);
    uint2 *hits = reinterpret_cast<uint2 *>(d_hits);
    if (any) k_trace<true><<<grid, kBlock, 0, s->stream>>>(s->ds, rays, n, nullptr, d_occ, nullptr, s->d_spill);
    else if (ids) k_trace<false, true><<<grid, kBlock, 0, s->stream>>>(s->ds, rays, n, hits, nullptr, s->d_geom_first, s->d_spill);
    else k_trace<false><<<grid, kBlock, 0, s->stream>>>(s->ds, rays, n, hits, nullptr, nullptr, s->d_spill);
    WR_HIP(hipGetLastError());
    if (ms) {
        WR_HIP(hipEventRecord(s->ev[1], s->stream));
        WR_HIP(hipEventSynchronize(s->ev[1]));
        WR_HIP(hipEventElapsedTime(ms, s->ev[0], s->ev[1]));
    }
    return WR_OK;
}

int wr_trace_closest_device(wr_scene *s, const float *d_rays, uint32_t n, void *d_hits, float *ms) {
    if (!s || (n && (!d_rays || !d_hits))) return set_error(WR_ERR_INVALID_ARGUMENT, "null argument");
    return trace_impl(s, d_rays, n, d_hits, nullptr, false, ms);
}

int wr_trace_any_device(wr_scene *s, const float *d_rays, uint32_t n, uint8_t *d_occ, float *ms) {
    if (!s || (n && (!d_rays || !d_occ))) return set_error(WR_ERR_INVALID_ARGUMENT, "null argument");
    return trace_impl(s, d_rays, n, nullptr, d_occ, true, ms);
}

// Rays from host arrays; results, n words in each of three host arrays for hits or
// n bytes in one for flags, to host arrays.  Up to 32,768 rays (a chunk of the
// pinned ring) the kernel reads the rays, and up to 1,310,720 hits or 15.7M flags
// it writes the results, in pinned memory: one launch, one wait, and for the
// smaller calls no device memory (1,000 hits: 28 us; with hipMemcpy each way and
// the ids looked up on the host 61, through four staged transfers 102).  More rays
// go up by the runtime's own copy, which the ring's threads do not beat (98,304
// rays 138 us and 199, 1,048,576 rays 1.24 ms and 1.16 from memory, 0.94 and
// 1.13 from the caches).  Where another thread has the ring, everything goes by
// plain copies instead of waiting for it (4 threads with 30,000 hits each, per query:
// 70 us, in turn on the ring 99, with plain copies alone 83).
static int trace_host(wr_scene *s, const float *rays, uint32_t n, bool any, void *r0, void *r1 = nullptr, void *r2 = nullptr) {
    int rc = set_device(s->dev);
    if (rc) return rc;
    TransferRing &ring = s->dev->ring;
    const size_t ray_bytes = sizeof(float) * 8 * size_t(n);
    const size_t row = (any ? 1 : sizeof(uint32_t)) * size_t(n), more = any ? 0 : row;
    const bool fits = row + 2 * more <= ring.kLeaseOut;  // the results; they are smaller than the rays
    bool up = ray_bytes > ring.kLeaseIn;                 // the rays go to device memory
    TransferRing::Lease lease;
    if (!up) WR_HIP(ring.try_lease(&lease));
    up = up || !lease.in;
    char *d = nullptr;  // rays, then results
    hipError_t e = hipSuccess;
    if (up) {
        WR_HIP(s->dev->alloc(reinterpret_cast<void **>(&d), ray_bytes + row + 2 * more));
        e = hipMemcpyAsync(d, rays, ray_bytes, hipMemcpyHostToDevice, s->stream);
        if (e == hipSuccess && fits) e = ring.try_lease(&lease);
    }
    if (e == hipSuccess) {
        if (!up) std::memcpy(lease.in, rays, ray_bytes);
        const float *in = reinterpret_cast<const float *>(up ? d : lease.in);
        char *out = lease.in ? lease.out : d + ray_bytes;
        rc = any ? trace_impl(s, in, n, nullptr, reinterpret_cast<uint8_t *>(out), true, nullptr)
                 : trace_impl(s, in, n, out, nullptr, false, nullptr, true);
        const std::initializer_list<TransferRing::Out> parts = {{r0, out, row}, {r1, out + row, more}, {r2, out + 2 * row, more}};
        if (rc == WR_OK && lease.in) {
            if ((e = hipStreamSynchronize(s->stream)) == hipSuccess) ring.copy(parts);
        } else if (rc == WR_OK) {
            e = fits ? ring.plain(s->stream, parts) : ring.download(s->dev->ordinal, s->stream, parts);
        }
    }
    if (rc || e != hipSuccess) (void)hipStreamSynchronize(s->stream);
    if (d) (void)hipFree(d);
    if (rc) return rc;
    if (e != hipSuccess) return set_error(WR_ERR_DEVICE, hipGetErrorString(e));
    return WR_OK;
}

int wr_trace_closest(wr_scene *s, const float *rays, uint32_t n, uint32_t *geom, uint32_t *prim, float *t) {
    if (!s || (n && (!rays || !geom || !prim || !t))) return set_error(WR_ERR_INVALID_ARGUMENT, "null argument");
    if (n == 0) return WR_OK;
    return trace_host(s, rays, n, false, geom, prim, t);
}

int wr_trace_any(wr_scene *s, const float *rays, uint32_t n, uint8_t *occluded) {
    if (!s || (n && (!rays || !occluded))) return set_error(WR_ERR_INVALID_ARGUMENT, "null argument");
    if (n == 0) return WR_OK;
    return trace_host(s, rays, n, true, occluded);
}
