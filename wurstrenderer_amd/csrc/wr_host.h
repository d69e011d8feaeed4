// wr_host.h -- host-side state shared by the library's translation units:
// error reporting, the path-pool layout and the device, scene and film handles.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "../../include/wurst_amd.h"
#include "wr_device.h"
#include "wr_layout.h"
#include "wr_memory.h"
#include "wr_transfer.h"

namespace wr {
// Thread-local message behind wr_last_error().
inline std::string &error_string() {
    static thread_local std::string s;
    return s;
}
}  // namespace wr

using namespace wr;

// ============================================================== errors
static inline int set_error(int code, const std::string &msg) {
    wr::error_string() = msg;
    return code;
}
#define WR_HIP(expr)                                                                                     \
    do {                                                                                                 \
        hipError_t e_ = (expr);                                                                          \
        if (e_ != hipSuccess)                                                                            \
            return set_error(e_ == hipErrorOutOfMemory ? WR_ERR_OUT_OF_MEMORY : WR_ERR_DEVICE,           \
                             std::string(#expr) + ": " + hipGetErrorString(e_));                         \
    } while (0)

// ============================================================== kernel arguments
constexpr int kBlock = 64;  // one wavefront per block; LDS stack indexed by lane

// Shadow-ray targets: where a visible connection's contribution goes.
constexpr uint32_t kTargetMask = 0x3FFFFFFFu;
constexpr uint32_t kToNextPath = 0u << 30;   // radiance of a continuing path (its index in the state that
                                             // the shade kernel wrote, current when the ray is traced)
constexpr uint32_t kToSample = 1u << 30;     // per-sample radiance of a finished path
constexpr uint32_t kToSplat = 2u << 30;      // light->camera splat (pixel of the FP64 splat film)

// Path state in queue order (SoA, double buffered): entry i of the current
// state is the i-th active path.  Shade writes continuing paths compacted into
// the next state; regen appends new samples behind them.  Every kernel walks
// the state in order, so all path-state traffic is coalesced, and the shade
// kernel, which reads and writes it all, is close to the rate of a plain copy:
// an entry is four full 16-byte rows, the integers in the rows' fourth words.
struct PathState {
    float4 *ray_o, *ray_d;  // ray to extend; w: RNG key, sample index in the pass (bits)
    float4 *thr;            // rgb: throughput of the next vertex; w: pdfW of the ray direction
    float4 *rad;            // rgb: radiance gathered so far (FP32); w: bounce of the next vertex,
                            // and the job in the bits above kBounceBits (bits)
    uint32_t *rec;          // 1 + training record of the previous vertex (0: none); guided renders only
    uint32_t shadow_count;  // counter (kShadowA or kShadowB) of the shadow queue that the shade
                            // kernel appends to while this state is current; the two states
                            // hold the two counters and swap them with everything else
};

struct PathBuffers {
    PathState cur, next;
    uint2 *hit;                  // per current entry: leaf-order triangle (or kInvalid), t bits
    float4 *sample_rad;          // per sample of the pass: final radiance (FP32)
    float4 *sh_o, *sh_d, *sh_c;  // shadow rays: o.xyz+tmax, d.xyz+target, contribution
    uint32_t *counters;          // see Counter
    unsigned long long *stats;   // [0] extend rays [1] shadow rays [2] ext nodes [3] ext tris [4] shd nodes [5] shd tris
    double *film_base, *film_splat;
};

// Each counter sits on its own 256-byte line: atomics on one line serialise.
constexpr int kCounterStride = 64;
constexpr int kXcds = 8;  // MI355X: 8 accelerator complex dies, each with its own L2
enum Counter : int {
    kQ = 0 * kCounterStride,         // continuing paths at the head of the current state
    kFresh = 1 * kCounterStride,     // new samples started behind them this iteration
    kQn = 2 * kCounterStride,        // paths continuing into the next state
    kTicket = 3 * kCounterStride,    // blocks of the shade kernel that have finished (the last one ends the
                                     // iteration); word 1: iterations ended in this pass
    // Shadow queue: the shade kernel of iteration i appends its shadow rays,
    // then the regeneration of iteration i + 1 its t = 1 connections, and the
    // traversal launch of iteration i + 1 traces them beside that iteration's
    // closest-hit rays.  Consecutive iterations alternate between the two
    // counters (PathState::shadow_count), so a queue's count survives the end
    // of its iteration while the next shade kernel appends from zero.
    kShadowA = 4 * kCounterStride,
    kShadowB = 5 * kCounterStride,
    kClaimed = 6 * kCounterStride,   // samples started so far in the pass
    kBase = 7 * kCounterStride,      // first sample index started this iteration
    kFetchExtX = 8 * kCounterStride,   // extend: work counter of XCD x's share at kFetchExtX + x * kCounterStride
    kFetchShdX = 16 * kCounterStride,  // shadow: likewise
    kNumCounterLines = 24
};

struct RenderArgs {
    uint32_t total;           // samples of this pass = spp * W * H
    uint32_t wh;
    uint32_t first_sample;    // sample index of the pass's first spp
    uint32_t seed;
    uint32_t capacity;        // path pool size
    int N;                    // num_path_vertices
    int use_mis;
    int nee;                  // 1: PathNeeRenderer (NEE, t = 1 splats); 0: PrimitivePathRenderer (BSDF sampling only)
    int guided;               // 1: entries carry a training record (PathState::rec)
    uint32_t tag;             // pass tag of the progress word
    unsigned long long *progress;  // pinned host word (null: the host polls the counters): tag << 32 | iterations
                                   // ended << 1 | drained, written at the end of each iteration
    int light;                // 1: LightSplattingRenderer (light subpaths connected to the camera)
};

// ============================================================== host objects
struct wr_device : wr::DeviceMemory {
    int ordinal = 0;
    int n_cu = 256;
    // resident blocks per CU of each kernel (HIP occupancy API), used to size persistent grids
    int occ_rays = 8, occ_generate = 8;
    std::mutex occ_mutex;  // guards occ_cache
    std::map<const void *, int> occ_cache;  // other kernels, filled on first use
    TransferRing ring;        // pinned buffers of large host transfers
    void *scratch = nullptr;  // device address of wr_render_nee_noalloc's fixed region on this GPU
};

struct wr_scene {
    wr_device *dev = nullptr;
    hipStream_t stream = nullptr;
    DScene ds{};
    // device allocations
    Node4 *d_nodes = nullptr;   // the build's BVH4 (checks and statistics)
    NodeQ *d_qnodes = nullptr;  // its quantised copy, which the kernels traverse
    float4 *d_tris = nullptr;
    void *d_tables = nullptr;   // one allocation behind the five tables below
    float4 *d_ltris = nullptr;
    uint2 *d_spill = nullptr;   // traversal stack spill: kSpillDepth entries per lane of the largest grid
    BlockPool::Block spill;     // the block behind it, from the device's pool
    BlockPool::Block nodes_block, tris_block, qnodes_block;  // behind the geometry, if it came from the pool
    float4 *d_bdpt = nullptr;   // bidirectional light-vertex records (+ 2 ray counters), grown on demand
    size_t bdpt_bytes = 0;
    int max_trav_blocks = 0;
    int2 *d_geom = nullptr;
    uint32_t *d_geom_first = nullptr;  // each geometry's first triangle
    DMat *d_mats = nullptr;
    DLight *d_lights = nullptr;
    float4 *d_env = nullptr;            // envmap texels; cdf and pdf follow in d_env_cdf
    float *d_env_cdf = nullptr;
    std::vector<DLight> h_lights;       // host copy of the light table
    std::vector<double> light_w;        // area-light selection weights |L|_2
    uint64_t n_nodes = 0, n_tris = 0, device_bytes = 0;
    uint32_t max_stack = 0;
    int builder = WR_BVH_GPU;           // which builder made the BVH
    int ploc_radius = 0;                // its clustering window (GPU builder; 0 = default)
    uint32_t bvh_depth = 0, bvh_iterations = 0;
    double build_ms = 0.0;
    // first triangle of each geometry
    std::vector<uint32_t> geom_first;
    int W = 0, H = 0;
    float box[6] = {0, 0, 0, 0, 0, 0};  // bounds of the vertices (lo xyz, hi xyz)
    // path buffers (lazily sized)
    PathBuffers pb{};
    uint32_t capacity = 0, sample_capacity = 0;
    void *pool = nullptr;
    uint32_t *h_counters = nullptr;  // pinned host copy of the pool counters; the progress word behind it
    uint32_t pass_tag = 0;           // passes started
    hipEvent_t ev[2] = {nullptr, nullptr};
};

struct wr_film {
    wr_scene *scene = nullptr;
    double *d_base = nullptr, *d_splat = nullptr;
    int W = 0, H = 0;
};

static inline int set_device(wr_device *dev) {
    WR_HIP(hipSetDevice(dev->ordinal));
    return WR_OK;
}

// ============================================================== GPU BVH build (wr_bvh_gpu.hip)
namespace wr {
struct GpuBvhResult {
    Node4 *nodes = nullptr;     // device, n_nodes, breadth-first (root = 0, children after parents)
    TriRecord *tris = nullptr;  // device, leaf order
    BlockPool::Block nodes_block, tris_block;  // the blocks of the device's geometry pool behind them, if any
    uint32_t n_nodes = 0, max_stack = 0, depth = 0, iterations = 0;
    double ms = 0.0;            // wall time of the build
};
// Temporary device memory of one build: every array is asked for with want(),
// commit() takes one block for all of them from the device's pool and sets the
// pointers, and the block goes back when the object dies, after the stream has
// finished.  (26 allocations and frees took 5 ms of a 15 ms scene creation.)
struct BuildArena {
    wr_device *dev;
    hipStream_t stream;
    BlockPool::Block block;
    size_t total = 0;
    std::vector<std::pair<void **, size_t>> wants;
    BuildArena(wr_device *d, hipStream_t st) : dev(d), stream(st) {}
    BuildArena(const BuildArena &) = delete;
    BuildArena &operator=(const BuildArena &) = delete;
    template <typename T>
    void want(T **p, size_t count) {
        wants.emplace_back(reinterpret_cast<void **>(p), total);
        total += (std::max<size_t>(count * sizeof(T), 1) + 255) / 256 * 256;
    }
    hipError_t commit() {
        const hipError_t e = dev->take(dev->build_memory, total, &block);
        if (e == hipSuccess)
            for (auto &w : wants) *w.first = static_cast<char *>(block.p) + w.second;
        return e;
    }
    ~BuildArena() {
        (void)hipStreamSynchronize(stream);
        dev->build_memory.give(block);
    }
};
// The clustering's state: m clusters in buffer `which`, the next node id, the
// iteration (seed of the tie-breaking hash), and whether no progress was made
// (m is 0 then).  It stays on the device: the host enqueues kPlocBatch
// iterations with grids for the clusters it last knew of and then looks (a look
// at each of the 29 iterations above the tail at 1.31M triangles, with a library
// scan in each: first frame 7.1 ms; so: 6.85).
struct PlocState {
    uint32_t m, base, iteration, which, stuck;
};
// The build's arrays, all in a BuildArena.
struct BuildBuffers {
    float *verts;                  // the mesh: one array, so that it goes up in one transfer
    uint32_t *tris, *tri_geom;     // inside it, set by the caller of bvh_gpu_plan after commit()
    float *partial, *cbox;         // bounds: per block, then min xyz and max xyz
    uint32_t *flags32;             // [0]: the mesh is invalid
    uint64_t *keys, *keys2;
    uint32_t *vals, *order, *cl, *cl2, *nearest, *sums, *einner, *eincl, *counts;
    PlocState *ploc;
    float4 *nlo, *nhi, *wc;
    uint32_t *wd;
    uint2 *kids;
    uint4 *q, *q2, *ekid, *eoff;
    Node4 *nodes_tmp;
    uint8_t *tmp;                  // the library's temporary storage
    size_t sort_bytes, scan32_bytes;
};
// Asks for the arrays of a build over n > 0 triangles and n_verts vertices.
int bvh_gpu_plan(uint32_t n, uint32_t n_verts, hipStream_t stream, BuildArena *arena, BuildBuffers *b);
// Checks the mesh in the build's arrays as the host checks of a scene do (finite
// vertices, indices in range, triangles of a geometry contiguous and ordered)
// and finds the bounds of its vertices (lo xyz, hi xyz).
int mesh_check_gpu(const BuildBuffers &b, uint32_t n, uint32_t n_verts, uint32_t n_geoms, hipStream_t stream, bool *valid,
                   float box[6]);
// Builds from a checked mesh with a clustering window of `radius` clusters on
// each side (0: default, at most 64).  On error the caller frees whatever
// out->nodes / out->tris hold.
int build_bvh4_gpu(wr_device *dev, const BuildBuffers &b, uint32_t n, hipStream_t stream, int radius, GpuBvhResult *out);
}  // namespace wr

// ============================================================== guiding (wr_guide.hip)
#include "wr_guide.h"
// A render call: guide_render_begin; per pass (record set k = pass % 2):
// guide_pass_net (the network inference reads: the one trained on the previous
// pass; the render stream waits for that training on the GPU),
// guide_begin_pass, guide_shade_view, the pass, guide_end_pass (training
// weights from the pass's final per-sample radiance, then `steps` Adam steps
// enqueued on the guide's own stream); guide_render_end waits for the last
// training.
int guide_render_begin(wr_guide *g);
int guide_pass_net(wr_guide *g, int set, bool overlap, wr::guide::Net *net);
int guide_shade_view(wr_guide *g, int set, float alpha, float record_prob, bool collect, uint32_t max_bounce,
                     wr::guide::Shade *out);
// Clears the record set and picks the fraction of paths to record so that
// about 90% of the capacity fills.
int guide_begin_pass(wr_guide *g, int set, uint64_t samples, float *record_prob);
int guide_end_pass(wr_guide *g, int set, const float4 *sample_rad, uint64_t samples, float record_prob, uint32_t steps,
                   wr_guide_stats *gs);
int guide_render_end(wr_guide *g, wr_guide_stats *gs);
// Sizes the per-entry draws of the inference kernel for a path pool of `capacity` entries.
int guide_reserve_draws(wr_guide *g, uint32_t capacity);
wr_scene *guide_scene(const wr_guide *g);
