// Batched pairwise geometry entry points: narrowphase on arbitrary shape pairs
// and GJK / EPA on shape cores.  These expose the collision routines the world
// step uses (dev_geom.hpp) on caller-chosen configurations.
#include <algorithm>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <utility>

#include "axiom/axm.h"
#include "dev_geom.hpp"
#include "host_copy.hpp"
#include "staging.hpp"

using namespace axm;

// ---------------------------------------------------------------- allocation-free staging
// Staging of axm_collide_pairs_noalloc: the inputs, outputs and per-pair status of at
// most NOALLOC_MAX_PAIRS pairs, one region of 32-bit words per field (each region holds
// that field for every pair slot: NOALLOC_MAX_PAIRS x width words).  One copy per
// device, held until the process ends; the calls on a device take turns on it.
constexpr uint32_t NOALLOC_MAX_PAIRS = 16384;
// region offsets, in words per pair slot: ta 1, pa 3, xa 3, qa 4, tb 1, pb 3, xb 3, qb 4 (inputs),
// npts 1, pos 12, normal 12, depth 4, feature 4, status 1 (outputs), queue of deep pairs 1; the
// queue's length follows
constexpr uint32_t NA_TA = 0, NA_PA = 1, NA_XA = 4, NA_QA = 7, NA_TB = 11, NA_PB = 12, NA_XB = 15, NA_QB = 18,
                   NA_NP = 22, NA_POS = 23, NA_NRM = 35, NA_DEP = 47, NA_FID = 51, NA_ST = 55, NA_QUEUE = 56, NA_WORDS = 57;
static __device__ __align__(256) uint32_t scratch[(size_t)NOALLOC_MAX_PAIRS * NA_WORDS + 64];

namespace {

struct PairIn {
    const uint32_t* ta;
    const float* pa;
    const float* xa;
    const float* qa;
    const uint32_t* tb;
    const float* pb;
    const float* xb;
    const float* qb;
};

__device__ __forceinline__ Shp shape_at(const uint32_t* t, const float* p, const float* x, const float* q, uint32_t i) {
    Shp s;
    s.type = t[i];
    s.prm = f3{p[3 * i], p[3 * i + 1], p[3 * i + 2]};
    s.c = f3{x[3 * i], x[3 * i + 1], x[3 * i + 2]};
    s.R = quat_to_mat(q4{q[4 * i], q[4 * i + 1], q[4 * i + 2], q[4 * i + 3]});
    return s;
}

struct PairOut {
    uint32_t* npts;
    float *pos, *nrm, *depth;
    uint32_t* fid;
    int32_t* status;
};
// Pairs whose cores intersect, for the expansion kernel: their numbers and how many.
struct DeepQueue {
    uint32_t *list, *count;
};
__device__ __forceinline__ void queue_deep(const DeepQueue& Q, bool deep, uint32_t i) {
    const unsigned long long m = __ballot(deep);
    if (!m) return;
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t base = 0;
    if (lane == 0u) base = atomicAdd(Q.count, (uint32_t)__popcll(m));
    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    if (deep) Q.list[base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = i;
}

// Inlined: called, it has the manifold and its own arguments in scratch memory (1000 pairs of boxes
// 28 us, inlined 21; spheres 8 and 4).
__device__ __forceinline__ void store_pair(const PairOut& out, uint32_t i, const Man& m, int st) {
    out.npts[i] = m.np;
    out.status[i] = st;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        const bool on = k < m.np;
        const size_t s = (size_t)i * 4 + k;
        out.pos[3 * s] = on ? m.pt[k].p.x : 0.f;
        out.pos[3 * s + 1] = on ? m.pt[k].p.y : 0.f;
        out.pos[3 * s + 2] = on ? m.pt[k].p.z : 0.f;
        out.nrm[3 * s] = on ? m.pt[k].n.x : 0.f;
        out.nrm[3 * s + 1] = on ? m.pt[k].n.y : 0.f;
        out.nrm[3 * s + 2] = on ? m.pt[k].n.z : 0.f;
        out.depth[s] = on ? m.pt[k].depth : 0.f;
        out.fid[s] = on ? m.pt[k].fid : 0u;
    }
}

// Narrowphase of the pairs, a wave per tile of pairs and group of tests (blockIdx.y): box-capsule,
// box-box, the light pairs, planes.  A wave lists the tile's pairs of its group and takes them 64 at
// a time, so its lanes run one test together and the groups run side by side; a thread per pair in
// the caller's order ran every test of its wave in turn (and the expansions of deep pairs in
// scratch memory).  The chain of one test bounds a small batch, so tiles are 64 pairs while every
// wave has a SIMD of its own (16384 pairs: 1024 waves) and grow with the batch to fill the lanes.
// 16384 mixed pairs: 27 us, and 29 us for their deep pairs; together they took 317.
constexpr uint32_t PAIR_TILE_MIN = 64u, PAIR_TILE_MAX = 1024u, PAIR_TILES = 256u;
constexpr uint32_t PAIR_GROUPS = 4u;
__device__ __forceinline__ uint32_t pair_group(uint32_t ta, uint32_t tb) {
    if (tb == SHAPE_PLANE) return 3u;
    const uint32_t lo = min(ta, tb), hi = max(ta, tb);
    return lo == SHAPE_BOX ? (hi == SHAPE_CAPSULE ? 0u : 1u) : 2u;
}
__global__ void __launch_bounds__(64) k_collide_pairs(PairIn in, uint32_t n, uint32_t tile, float margin, PairOut out,
                                                      DeepQueue Q) {
    __shared__ uint16_t list[PAIR_TILE_MAX];
    const uint32_t lane = threadIdx.x, first = blockIdx.x * tile, len = min(tile, n - first), group = blockIdx.y;
    uint32_t count = 0;
    for (uint32_t o = 0; o < len; o += 64u) {
        const uint32_t i = first + o + lane;
        const bool mine = o + lane < len && pair_group(in.ta[i], in.tb[i]) == group;
        const unsigned long long m = __ballot(mine);
        if (mine) list[count + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)(o + lane);
        count += (uint32_t)__popcll(m);
    }
    __syncthreads();
    for (uint32_t o = 0; o < count; o += 64u) {
        const bool on = o + lane < count;
        const uint32_t i = first + (on ? list[o + lane] : 0u);
        bool deep = false;
        if (on) {
            const Shp A = shape_at(in.ta, in.pa, in.xa, in.qa, i);
            Man m;
            m.np = 0;
            int st = GEOM_OK;
            if (group == 3u) {
                // plane given as params = normal, pos.x = offset d
                collide_plane(m, A, f3{in.pb[3 * i], in.pb[3 * i + 1], in.pb[3 * i + 2]}, in.xb[3 * i], margin);
            } else {
                const Shp B = shape_at(in.tb, in.pb, in.xb, in.qb, i);
                const bool swap = A.type > B.type;
                const Shp S0 = select_shape(swap, B, A), S1 = select_shape(swap, A, B);
                st = group < 2u ? collide_canon<COLLIDE_HEAVY>(m, S0, S1, margin, deep)
                                : collide_canon<COLLIDE_LIGHT>(m, S0, S1, margin, deep);
                if (swap) flip_manifold(m);
            }
            if (!deep) store_pair(out, i, m, st);
        }
        queue_deep(Q, deep, i);
    }
}
__global__ void k_queue_clear(uint32_t* count) { *count = 0u; }
// The deep box-capsule pairs, one wave each.
__global__ void __launch_bounds__(64) k_collide_deep(PairIn in, PairOut out, DeepQueue Q) {
    __shared__ EpaWork W;
    const uint32_t nq = *Q.count;
    for (uint32_t q = blockIdx.x; q < nq; q += gridDim.x) {
        const uint32_t i = Q.list[q];
        const Shp A = shape_at(in.ta, in.pa, in.xa, in.qa, i), B = shape_at(in.tb, in.pb, in.xb, in.qb, i);
        const bool swap = A.type > B.type;
        Man m;
        m.np = 0;
        const int st = box_capsule_epa(m, select_shape(swap, B, A), select_shape(swap, A, B), W);
        if (swap) flip_manifold(m);
        if (threadIdx.x == 0u) store_pair(out, i, m, st);
    }
}

// GJK of the pairs, a thread each; those whose cores intersect are queued for expansion.
__global__ void __launch_bounds__(64) k_gjk_pairs(PairIn in, uint32_t n, float* out, int32_t* status, int gjk_iters,
                                                  DeepQueue Q) {
    const uint32_t i = blockIdx.x * 64u + threadIdx.x;
    bool deep = false;
    if (i < n) {
        const GjkOut g = gjk(shape_at(in.ta, in.pa, in.xa, in.qa, i), shape_at(in.tb, in.pb, in.xb, in.qb, i), gjk_iters);
        deep = g.status == 1;
        if (!deep) {
            float* o = out + (size_t)i * 10;
            o[0] = g.dist;
            o[1] = g.pA.x; o[2] = g.pA.y; o[3] = g.pA.z;
            o[4] = g.pB.x; o[5] = g.pB.y; o[6] = g.pB.z;
            o[7] = o[8] = o[9] = 0.f;
            status[i] = g.status == 0 ? 0 : GEOM_GJK_FAIL;
        }
    }
    queue_deep(Q, deep, i);
}
// EPA of the queued pairs, one wave each (16384 pairs, 3500 of them deep: 23 us the pairs' GJK,
// 67 us the expansions; with the expansion on the pair's own thread 420).
__global__ void __launch_bounds__(64) k_epa_pairs(PairIn in, float* out, int32_t* status, int gjk_iters, int epa_iters,
                                                  DeepQueue Q) {
    __shared__ EpaWork W;
    const uint32_t nq = *Q.count;
    for (uint32_t q = blockIdx.x; q < nq; q += gridDim.x) {
        const uint32_t i = Q.list[q];
        const Shp A = shape_at(in.ta, in.pa, in.xa, in.qa, i), B = shape_at(in.tb, in.pb, in.xb, in.qb, i);
        const EpaOut e = epa(A, B, gjk(A, B, gjk_iters), W, epa_iters);
        if (threadIdx.x == 0u) {
            float* o = out + (size_t)i * 10;
            o[0] = e.depth;
            o[1] = e.pA.x; o[2] = e.pA.y; o[3] = e.pA.z;
            o[4] = e.pB.x; o[5] = e.pB.y; o[6] = e.pB.z;
            o[7] = e.n.x; o[8] = e.n.y; o[9] = e.n.z;
            status[i] = e.status == 0 ? 1 : GEOM_EPA_FAIL;
        }
    }
}

// Waves of an expansion kernel: two on a SIMD are all that its registers leave room for; they
// stride over the queue.
uint32_t deep_waves(uint32_t n) { return std::min<uint32_t>(n, 2048u); }
// deep: some pair may be queued.
void launch_collide(const PairIn& in, uint32_t n, float margin, const PairOut& out, const DeepQueue& Q, bool deep,
                    hipStream_t s) {
    uint32_t tile = PAIR_TILE_MIN;
    while (tile < PAIR_TILE_MAX && (uint64_t)tile * PAIR_TILES < n) tile *= 2u;
    hipLaunchKernelGGL(k_collide_pairs, dim3((n - 1u) / tile + 1u, PAIR_GROUPS), dim3(64), 0, s, in, n, tile, margin, out, Q);
    if (deep) hipLaunchKernelGGL(k_collide_deep, dim3(deep_waves(n)), dim3(64), 0, s, in, out, Q);
}

// What a batched call holds while it runs: staging for its arrays and a stream.  A process keeps
// one idle workspace per device for the next call (calls that overlap make their own): at most
// STAGE_PINNED of pinned and KEPT_BYTES of device memory, more is freed at the call's end.  The
// table lives until the process ends and takes its memory along: a destructor at exit could
// find the runtime gone.
constexpr size_t KEPT_BYTES = 32u << 20;
struct PairSpace {
    int device = 0;
    hipStream_t stream = nullptr;
    Staging stage;
    ~PairSpace() {
        if (stream) (void)hipStreamDestroy(stream);
    }
};
constexpr int PAIR_DEVICES = 64;
std::mutex g_space_mu;
PairSpace* g_space[PAIR_DEVICES] = {};

// The workspace of one call: the device's idle one or a new one, with room for `bytes`.
class PairCall {
public:
    axm_status open(int32_t device, size_t bytes) {
        if (hipSetDevice(device) != hipSuccess) return AXM_GPU_OPERATION_FAILED;
        if (device >= 0 && device < PAIR_DEVICES) {
            std::lock_guard<std::mutex> lk(g_space_mu);
            w_.reset(std::exchange(g_space[device], nullptr));
        }
        if (!w_) {
            w_.reset(new (std::nothrow) PairSpace);
            if (!w_) return AXM_OUT_OF_MEMORY;
            w_->device = device;
        }
        if (!w_->stream && hipStreamCreateWithFlags(&w_->stream, hipStreamNonBlocking) != hipSuccess)
            return AXM_GPU_OPERATION_FAILED;
        return w_->stage.ensure(bytes);
    }
    // Keeps the workspace for the next call; one that met an error is not kept.
    void keep() {
        const int device = w_ ? w_->device : -1;
        if (device < 0 || device >= PAIR_DEVICES) return;
        w_->stage.trim(KEPT_BYTES);
        std::lock_guard<std::mutex> lk(g_space_mu);
        if (!g_space[device]) g_space[device] = w_.release();
    }
    PairSpace* operator->() const { return w_.get(); }

private:
    std::unique_ptr<PairSpace> w_;
};

// The arrays of a batched call in its device block: inputs, the queue's length, then the outputs
// and the queue (each region on a 16-byte boundary).
struct PairLayout {
    StagePart part[10];
    int parts = 0;
    size_t total = 0;
    size_t add(const void* host, size_t words) {
        const size_t at = total;
        if (host) part[parts++] = StagePart{const_cast<void*>(host), at, 4 * words};
        total += (4 * words + 15) / 16 * 16;
        return at;
    }
};
const uint32_t NO_PAIRS = 0u;

// per device: the address of its copy of `scratch`, set on first use
constexpr int NOALLOC_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
uint32_t* g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};
// per device: held by a call from its first upload to its last read.  Two calls at once would share
// the queue's length and append past the queue.
std::mutex g_scratch_use[NOALLOC_MAX_DEVICES];

// The device address of `scratch` on `device`, looked up once per device with that device
// current (each device holds its own copy at its own address; the host-side name of the
// array is not a device address and is never passed to the device).
uint32_t* scratch_on(int32_t device) {
    if (device < 0 || device >= NOALLOC_MAX_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return nullptr;
        g_scratch_ptr[device] = static_cast<uint32_t*>(p);
    }
    return g_scratch_ptr[device];
}

// Whether the types are allowed; sets *deep when a pair may go through the queue of deep pairs (a box
// with a capsule).
bool valid_types(uint32_t n, const uint32_t* ta, const uint32_t* tb, bool allow_plane_b, bool* deep = nullptr) {
    const uint32_t top_b = allow_plane_b ? (uint32_t)AXM_SHAPE_PLANE : (uint32_t)AXM_SHAPE_CAPSULE;
    uint32_t bad = 0, any = 0;  // no branch in the loop: the compiler takes several pairs at a time
    for (uint32_t i = 0; i < n; ++i) {
        const uint32_t a = ta[i], b = tb[i];
        bad |= (uint32_t)(a > (uint32_t)AXM_SHAPE_CAPSULE) | (uint32_t)(b > top_b);
        any |= (uint32_t)(a + b == SHAPE_BOX + SHAPE_CAPSULE) & (uint32_t)(b - SHAPE_BOX <= SHAPE_CAPSULE - SHAPE_BOX);
    }
    if (deep) *deep = any != 0u;
    return bad == 0u;
}

}  // namespace

extern "C" {

axm_status axm_collide_pairs(int32_t device, uint32_t n, const uint32_t* type_a, const float* prm_a,
                             const float* pos_a, const float* quat_a, const uint32_t* type_b, const float* prm_b,
                             const float* pos_b, const float* quat_b, float margin, uint32_t* npts, float* pos,
                             float* normal, float* depth, uint32_t* feature) {
    if (!n) return AXM_SUCCESS;
    if (!type_a || !prm_a || !pos_a || !quat_a || !type_b || !prm_b || !pos_b || !quat_b || !npts || !pos || !normal ||
        !depth || !feature)
        return AXM_NULL_POINTER;
    bool deep;
    if (!valid_types(n, type_a, type_b, true, &deep)) return AXM_INVALID_SHAPE;
    PairLayout up, down;
    const size_t N = n;
    const size_t ta = up.add(type_a, N), pa = up.add(prm_a, 3 * N), xa = up.add(pos_a, 3 * N), qa = up.add(quat_a, 4 * N),
                 tb = up.add(type_b, N), pb = up.add(prm_b, 3 * N), xb = up.add(pos_b, 3 * N), qb = up.add(quat_b, 4 * N),
                 qn = up.add(&NO_PAIRS, 1);
    // the first failing pair's status is the call's: the status words come down last
    std::unique_ptr<int32_t[]> st(new (std::nothrow) int32_t[N]);
    if (!st) return AXM_OUT_OF_MEMORY;
    const size_t d_np = down.add(npts, N), d_pos = down.add(pos, 12 * N), d_n = down.add(normal, 12 * N),
                 d_d = down.add(depth, 4 * N), d_f = down.add(feature, 4 * N), d_s = down.add(st.get(), N);
    PairCall c;
    const axm_status opened = c.open(device, up.total + down.total + 4 * N);
    if (opened != AXM_SUCCESS) return opened;
    hipStream_t s = c->stream;
    if (c->stage.up(up.part, up.parts, up.total, s) != hipSuccess) return AXM_GPU_OPERATION_FAILED;
    uint8_t* d = c->stage.dev();
    uint8_t* o = d + up.total;
    auto f32 = [](uint8_t* p) { return reinterpret_cast<float*>(p); };
    auto u32 = [](uint8_t* p) { return reinterpret_cast<uint32_t*>(p); };
    const PairIn in{u32(d + ta), f32(d + pa), f32(d + xa), f32(d + qa), u32(d + tb), f32(d + pb), f32(d + xb), f32(d + qb)};
    const PairOut out{u32(o + d_np), f32(o + d_pos), f32(o + d_n), f32(o + d_d), u32(o + d_f),
                      reinterpret_cast<int32_t*>(o + d_s)};
    launch_collide(in, n, margin, out, DeepQueue{u32(o + down.total), u32(d + qn)}, deep, s);
    if (hipGetLastError() != hipSuccess ||
        c->stage.down(down.part, down.parts, up.total, down.total, s) != hipSuccess)
        return AXM_GPU_OPERATION_FAILED;
    c.keep();
    for (uint32_t i = 0; i < n; ++i)
        if (st[i] != GEOM_OK) return st[i];
    return AXM_SUCCESS;
}

axm_status axm_collide_pairs_noalloc(int32_t device, uint32_t n, const uint32_t* type_a, const float* prm_a,
                                     const float* pos_a, const float* quat_a, const uint32_t* type_b,
                                     const float* prm_b, const float* pos_b, const float* quat_b, float margin,
                                     uint32_t* npts, float* pos, float* normal, float* depth, uint32_t* feature) {
    if (!n) return AXM_SUCCESS;
    if (!type_a || !prm_a || !pos_a || !quat_a || !type_b || !prm_b || !pos_b || !quat_b || !npts || !pos || !normal ||
        !depth || !feature)
        return AXM_NULL_POINTER;
    if (n > NOALLOC_MAX_PAIRS) return AXM_OUT_OF_RANGE;
    bool deep;
    if (!valid_types(n, type_a, type_b, true, &deep)) return AXM_INVALID_SHAPE;
    if (hipSetDevice(device) != hipSuccess) return AXM_GPU_OPERATION_FAILED;
    uint32_t* base = scratch_on(device);
    if (!base) return AXM_GPU_OPERATION_FAILED;
    std::lock_guard<std::mutex> turn(g_scratch_use[device]);
    // region r starts at base + r * NOALLOC_MAX_PAIRS
    auto reg = [&](uint32_t r) { return base + (size_t)r * NOALLOC_MAX_PAIRS; };
    struct Up {
        uint32_t r;
        const void* h;
        size_t bytes;
    };
    const Up ups[] = {{NA_TA, type_a, 4ull * n}, {NA_PA, prm_a, 12ull * n}, {NA_XA, pos_a, 12ull * n},
                      {NA_QA, quat_a, 16ull * n}, {NA_TB, type_b, 4ull * n}, {NA_PB, prm_b, 12ull * n},
                      {NA_XB, pos_b, 12ull * n}, {NA_QB, quat_b, 16ull * n}};
    // cleared by a launch, which the uploads do not wait for: a ninth upload took 13 us of a small call's
    // 205, this and the queue's launch 5, and neither is made when no pair can be deep
    if (deep) hipLaunchKernelGGL(k_queue_clear, dim3(1), dim3(1), 0, 0, reg(NA_WORDS));
    for (const Up& u : ups)
        if (copy_sync(reg(u.r), u.h, u.bytes, hipMemcpyHostToDevice) != hipSuccess) return AXM_GPU_OPERATION_FAILED;
    PairIn in;
    in.ta = reg(NA_TA);
    in.pa = reinterpret_cast<const float*>(reg(NA_PA));
    in.xa = reinterpret_cast<const float*>(reg(NA_XA));
    in.qa = reinterpret_cast<const float*>(reg(NA_QA));
    in.tb = reg(NA_TB);
    in.pb = reinterpret_cast<const float*>(reg(NA_PB));
    in.xb = reinterpret_cast<const float*>(reg(NA_XB));
    in.qb = reinterpret_cast<const float*>(reg(NA_QB));
    // the kernel writes every output word of the n pairs (zeros past a pair's point count),
    // so nothing left by an earlier call is read back
    const PairOut out{reg(NA_NP), reinterpret_cast<float*>(reg(NA_POS)), reinterpret_cast<float*>(reg(NA_NRM)),
                      reinterpret_cast<float*>(reg(NA_DEP)), reg(NA_FID), reinterpret_cast<int32_t*>(reg(NA_ST))};
    launch_collide(in, n, margin, out, DeepQueue{reg(NA_QUEUE), reg(NA_WORDS)}, deep, 0);
    if (hipStreamSynchronize(0) != hipSuccess) return AXM_GPU_OPERATION_FAILED;
    if (copy_sync(npts, reg(NA_NP), 4ull * n, hipMemcpyDeviceToHost) != hipSuccess ||
        copy_sync(pos, reg(NA_POS), 48ull * n, hipMemcpyDeviceToHost) != hipSuccess ||
        copy_sync(normal, reg(NA_NRM), 48ull * n, hipMemcpyDeviceToHost) != hipSuccess ||
        copy_sync(depth, reg(NA_DEP), 16ull * n, hipMemcpyDeviceToHost) != hipSuccess ||
        copy_sync(feature, reg(NA_FID), 16ull * n, hipMemcpyDeviceToHost) != hipSuccess)
        return AXM_GPU_OPERATION_FAILED;
    // the first failing pair's status, as axm_collide_pairs reports it; read 4096 at a time
    // into a fixed host buffer
    int32_t st[4096];
    for (uint32_t i0 = 0; i0 < n; i0 += 4096) {
        const uint32_t c = std::min<uint32_t>(4096u, n - i0);
        if (copy_sync(st, reg(NA_ST) + i0, 4ull * c, hipMemcpyDeviceToHost) != hipSuccess)
            return AXM_GPU_OPERATION_FAILED;
        for (uint32_t i = 0; i < c; ++i)
            if (st[i] != GEOM_OK) return st[i];
    }
    return AXM_SUCCESS;
}

axm_status axm_gjk_epa_pairs(int32_t device, uint32_t n, const uint32_t* type_a, const float* prm_a,
                             const float* pos_a, const float* quat_a, const uint32_t* type_b, const float* prm_b,
                             const float* pos_b, const float* quat_b, float* out, int32_t* status) {
    return axm_gjk_epa_pairs_capped(device, n, type_a, prm_a, pos_a, quat_a, type_b, prm_b, pos_b, quat_b, 0u, 0u, out,
                                    status);
}

axm_status axm_gjk_epa_pairs_capped(int32_t device, uint32_t n, const uint32_t* type_a, const float* prm_a,
                                    const float* pos_a, const float* quat_a, const uint32_t* type_b,
                                    const float* prm_b, const float* pos_b, const float* quat_b,
                                    uint32_t gjk_max_iters, uint32_t epa_max_iters, float* out, int32_t* status) {
    if (gjk_max_iters > 4096u || epa_max_iters > 4096u) return AXM_INVALID_PARAMETER;
    const int gi = gjk_max_iters ? (int)gjk_max_iters : 32, ei = epa_max_iters ? (int)epa_max_iters : 48;
    if (!n) return AXM_SUCCESS;
    if (!type_a || !prm_a || !pos_a || !quat_a || !type_b || !prm_b || !pos_b || !quat_b || !out || !status)
        return AXM_NULL_POINTER;
    if (!valid_types(n, type_a, type_b, false)) return AXM_INVALID_SHAPE;
    PairLayout up, down;
    const size_t N = n;
    const size_t ta = up.add(type_a, N), pa = up.add(prm_a, 3 * N), xa = up.add(pos_a, 3 * N), qa = up.add(quat_a, 4 * N),
                 tb = up.add(type_b, N), pb = up.add(prm_b, 3 * N), xb = up.add(pos_b, 3 * N), qb = up.add(quat_b, 4 * N),
                 qn = up.add(&NO_PAIRS, 1);
    const size_t d_o = down.add(out, 10 * N), d_s = down.add(status, N);
    PairCall c;
    const axm_status opened = c.open(device, up.total + down.total + 4 * N);
    if (opened != AXM_SUCCESS) return opened;
    hipStream_t s = c->stream;
    if (c->stage.up(up.part, up.parts, up.total, s) != hipSuccess) return AXM_GPU_OPERATION_FAILED;
    uint8_t* d = c->stage.dev();
    uint8_t* o = d + up.total;
    auto f32 = [](uint8_t* p) { return reinterpret_cast<float*>(p); };
    auto u32 = [](uint8_t* p) { return reinterpret_cast<uint32_t*>(p); };
    const PairIn in{u32(d + ta), f32(d + pa), f32(d + xa), f32(d + qa), u32(d + tb), f32(d + pb), f32(d + xb), f32(d + qb)};
    const DeepQueue Q{u32(o + down.total), u32(d + qn)};
    int32_t* st = reinterpret_cast<int32_t*>(o + d_s);
    hipLaunchKernelGGL(k_gjk_pairs, dim3((n - 1u) / 64u + 1u), dim3(64), 0, s, in, n, f32(o + d_o), st, gi, Q);
    hipLaunchKernelGGL(k_epa_pairs, dim3(deep_waves(n)), dim3(64), 0, s, in, f32(o + d_o), st, gi, ei, Q);
    if (hipGetLastError() != hipSuccess ||
        c->stage.down(down.part, down.parts, up.total, down.total, s) != hipSuccess)
        return AXM_GPU_OPERATION_FAILED;
    c.keep();
    return AXM_SUCCESS;
}

}  // extern "C"
