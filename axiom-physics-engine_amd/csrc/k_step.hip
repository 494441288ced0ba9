// gfx950 kernels of one simulation step (single world or a batch of worlds).
//
// Stage order per step (the reference sketches the same four stages,
// examples/profiling_example.cpp:132-165, with semi-implicit Euler from
// examples/body_inspector_example.cpp:48-60):
//   k_begin            gravity/damping -> solver velocities, world inverse inertia, AABB, cell key
//   radix sort         (key, body) stable
//   k_cell_table       hash of cell -> (first sorted index, count)
//   k_pair_count/emit  27-neighbour grid scan, inclusive AABB test, j > i; exclusive scan between
//   k_narrow(+_epa)    primitive narrowphase -> <= 4 points per pair (staged per pair)
//   k_compact          pairs with points -> manifolds (pair order, exclusive scan of the flags)
//   k_col_*            Jones-Plassmann colouring with first-fit colours
//   k_prep             per-point rows + warm start (previous-step impulses keyed by (a, b, feature))
//   k_pgs_solve        all sweeps of all islands (k_pgs_own: very large ones; k_pgs: one colour of
//                      one sweep)
//   k_residual         velocity-space fixed-point residual
//   k_integrate        x += v dt, q += dt/2 (w,0) q, normalise
// Every body-parallel kernel is one thread per body; every manifold-parallel
// kernel one thread per manifold.  Colour batches are contiguous in the
// solve-order arrays, so a wave of 64 manifolds of one colour reads 64
// consecutive 16-byte rows.
#include "dev_geom.hpp"
#include "dev_islands.hpp"
#include "k_mlp.hpp"
#include "k_step.hpp"

namespace axm {

__device__ __forceinline__ uint32_t fbits(float f) { return __float_as_uint(f); }
__device__ __forceinline__ float4 f4(f3 v, float w) { return make_float4(v.x, v.y, v.z, w); }

// Adds the sum of v over the wave to field f of the workgroup's spread row with one
// atomic (every lane of the wave must call it: the reduction reads all 64 lanes).
template <class T> __device__ __forceinline__ void spread_add(Counters* cnt, T SpreadRow::*f, T v) {
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63u) == 0u && v != T(0)) atomicAdd(&(cnt->sp[blockIdx.x % SPREAD].*f), v);
}
template <class T> __device__ __forceinline__ T spread_sum(const Counters* cnt, T SpreadRow::*f) {
    T s = 0;
#pragma unroll 8
    for (uint32_t k = 0; k < SPREAD; ++k) s += cnt->sp[k].*f;
    return s;
}

constexpr uint32_t PAIR_KINDS = 16;  // narrowphase test kinds (pair_kind)
// The per-step counters back to zero (the threads of one workgroup).
__device__ __forceinline__ void counters_reset(Counters* cnt, uint32_t* __restrict__ kinds, const Meeting& meet) {
    uint32_t* w = reinterpret_cast<uint32_t*>(cnt);
    constexpr uint32_t BAR_WORDS = sizeof(GridBar) / sizeof(uint32_t);
    if (threadIdx.x < BAR_WORDS) reinterpret_cast<uint32_t*>(meet.colour)[threadIdx.x] = 0u;
    else if (threadIdx.x - BAR_WORDS < SORT_MEET_WORDS) meet.sort[threadIdx.x - BAR_WORDS] = 0u;
    if (threadIdx.x < COUNTERS_RESET_WORDS) w[threadIdx.x] = 0u;
    for (uint32_t k = threadIdx.x; k < SPREAD; k += blockDim.x) {
        cnt->sp[k].islands = 0u;
        cnt->sp[k].sleeping = 0u;
        cnt->sp[k].contacts = 0u;
        cnt->sp[k].warm_hits = 0u;
        cnt->sp[k].cells = 0u;
        cnt->sp[k].pgs_bytes = 0ull;
    }
    if (kinds && threadIdx.x < 2u * PAIR_KINDS) kinds[threadIdx.x] = 0u;
}
// ---------------------------------------------------------------- k_begin
__global__ void __launch_bounds__(256) k_begin(Bodies B, StepParams sp, uint32_t n, uint64_t* __restrict__ key,
                                               uint32_t* __restrict__ key32, uint32_t* __restrict__ val, uint64_t* __restrict__ bmax0,
                                               uint64_t* __restrict__ bmax1, uint64_t* __restrict__ bmask,
                                               uint32_t* __restrict__ bdeg, Counters* __restrict__ cnt,
                                               uint32_t* __restrict__ kinds, Meeting meet, CellTable ct) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    // the step's counters start from zero (the kernels that count run after this launch;
    // steps_done, read below, is kept across steps)
    if (blockIdx.x == 0) counters_reset(cnt, kinds, meet);
    // with the Morton bitmap: the words the last step set go back to zero (several bodies
    // may name one word: all write zero); the cell table sets this step's after the sort
    if (ct.mbits && i < ct.mlist_n) {
        const uint32_t w = ct.mlist[i];
        if (w != UNSET) ct.mbits[w] = 0u;
    }
    if (i >= n) return;
    // the colouring's per-body words start from zero every step
    bmax0[i] = 0ull;
    bmax1[i] = 0ull;
    bmask[i] = 0ull;
    bdeg[i] = 0u;
    // islands start as singletons; a sleeping body whose island an awake body touched in
    // the previous step wakes up (the request carries the number of this step)
    B.upar[i] = i;
    B.imin[i] = 0x7F800000u;  // +inf
    B.icnt[i] = 0u;
    bool asleep = false;
    {
        const uint2 sl = B.slp[i];
        if (sl.y & ASLEEP_BIT) {
            const uint32_t lab = sl.y & LABEL_MASK;
            if (lab < n && B.wake[lab] == cnt->steps_done) B.slp[i] = make_uint2(0u, lab);
            else asleep = true;
        }
    }
    const float4 x4 = B.x[i], q4v = B.q[i], v4 = B.vel[i], w4 = B.angv[i], sh = B.shape[i];
    const uint32_t type = fbits(sh.w);
    // a sleeping body acts as a static one for the whole step
    const bool dyn = v4.w > 0.0f && !asleep;
    f3 v = xyz(v4), w = xyz(w4);
    if (dyn) {
        const f3 g = {sp.gx, sp.gy, sp.gz};
        const float4 mt = B.mat[i];
        v = (v + g * sp.dt) * mt.z;
        w = w * mt.w;
    }
    B.sv[i] = f4(v, dyn ? v4.w : 0.0f);
    B.sw[i] = f4(w, 0.0f);
    const m3 R = quat_to_mat(q4v);
    const float mg = sp.margin;
    f3 e;
    if (type == SHAPE_SPHERE) {
        e = {sh.x + mg, sh.x + mg, sh.x + mg};
    } else if (type == SHAPE_BOX) {
        e.x = fabsf(R.r0.x) * sh.x + fabsf(R.r0.y) * sh.y + fabsf(R.r0.z) * sh.z + mg;
        e.y = fabsf(R.r1.x) * sh.x + fabsf(R.r1.y) * sh.y + fabsf(R.r1.z) * sh.z + mg;
        e.z = fabsf(R.r2.x) * sh.x + fabsf(R.r2.y) * sh.y + fabsf(R.r2.z) * sh.z + mg;
    } else {
        e.x = fabsf(R.r0.y) * sh.y + sh.x + mg;
        e.y = fabsf(R.r1.y) * sh.y + sh.x + mg;
        e.z = fabsf(R.r2.y) * sh.y + sh.x + mg;
    }
    const f3 c = xyz(x4);
    // the AABB as one 32-byte record, with whether the body is dynamic this step, so that
    // the gather in cell order reads one place per body
    B.aabb[2u * i] = f4(c - e, 0.0f);
    B.aabb[2u * i + 1u] = f4(c + e, dyn ? 1.0f : 0.0f);
    auto cc = [&](float p, float o) -> uint32_t {
        float f = (p - o) * sp.inv_cell;
        f = f > 0.0f ? f : 0.0f;
        f = f < 1023.0f ? f : 1023.0f;
        return (uint32_t)floorf(f);
    };
    const uint32_t cx = cc(c.x, sp.ox), cy = cc(c.y, sp.oy), cz = cc(c.z, sp.oz);
    if (key32) key32[i] = morton3(cx, cy, cz);  // one world: the Morton code alone
    else key[i] = ((uint64_t)B.world[i] << 30) | morton3(cx, cy, cz);
    val[i] = i;
}

// ---------------------------------------------------------------- cell table
__global__ void k_fill_u64(uint64_t* __restrict__ p, uint64_t v, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}
__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t v, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Linear-probing tables.  Every probe loop visits at most mask + 1 slots, so a
// full table ends the loop (insert returns false, lookup misses) instead of
// spinning; tables are sized >= 2x their maximum entry count.
__device__ __forceinline__ uint64_t ent_key(uint4 e) { return (uint64_t)e.x | ((uint64_t)e.y << 32); }
__device__ __forceinline__ bool ht_insert(CellTable t, uint64_t k, uint2 v, uint32_t s) {
    for (uint32_t probe = 0; probe <= t.mask; ++probe) {
        const unsigned long long prev =
            atomicCAS((unsigned long long*)&t.ent[s], (unsigned long long)EMPTY_KEY, (unsigned long long)k);
        if (prev == EMPTY_KEY || prev == k) {
            reinterpret_cast<uint2*>(&t.ent[s])[1] = v;
            return true;
        }
        s = (s + 1) & t.mask;
    }
    return false;
}
// Continues a lookup of key k at slot s (linear probing).
__device__ __forceinline__ bool ht_find_from(const CellTable& t, uint64_t k, uint32_t s, uint2& v) {
    for (uint32_t probe = 0; probe <= t.mask; ++probe) {
        const uint4 e = t.ent[s];
        const uint64_t kk = ent_key(e);
        if (kk == k) {
            v = make_uint2(e.z, e.w);
            return true;
        }
        if (kk == EMPTY_KEY) return false;
        s = (s + 1) & t.mask;
    }
    return false;
}
// Occupancy bit of a cell hash (the high half of the hash; the slot takes the low bits).
__device__ __forceinline__ uint32_t cell_bit(uint64_t h, uint32_t bmask) { return (uint32_t)(h >> 32) & bmask; }

// The hash table and its occupancy bits (the Morton bitmap is cleared by k_begin).
__global__ void __launch_bounds__(256) k_cell_clear(CellTable t) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i <= t.mask) t.ent[i] = make_uint4((uint32_t)EMPTY_KEY, (uint32_t)(EMPTY_KEY >> 32), 0u, 0u);
    if (i <= (t.bmask >> 5)) t.bits[i] = 0u;
}

// The cell table is built in two passes, so that most cells need no atomic.  Pass 1
// (k_cell_table): the first body of each cell stores the cell's key into its home
// slot (an untorn 8-byte store; of heads whose homes collide, one key stays), sets
// its occupancy bit and counts it.  Pass 2 (k_cell_place): a head whose key is in
// its home slot writes its range there; the others insert by compare-and-swap from
// the next slot on.  Slots claimed in pass 1 never change, so every key still lies
// after its home with no empty slot between (the linear-probing invariant).
// Each thread also gathers the AABB of sorted body s into smin / smax (body index in
// smin.w), so that the candidates of a cell are contiguous and carry what the test needs.
__global__ void __launch_bounds__(256) k_cell_table(Bodies B, SortedKeys skey,
                                                    const uint32_t* __restrict__ sval, uint32_t n, CellTable t,
                                                    Counters* __restrict__ cnt) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t lane = __lane_id();
    if (s < n) {
        const uint32_t i = sval[s];
        const float4 mn = B.aabb[2u * i], mx = B.aabb[2u * i + 1u];
        B.smin[s] = make_float4(mn.x, mn.y, mn.z, __uint_as_float(i));
        B.smax[s] = mx;
    }
    // the first body of each cell inserts it; one count per wave
    const uint64_t k = s < n ? skey[s] : EMPTY_KEY;
    const bool head = s < n && (s == 0 || skey[s - 1] != k);
    spread_add(cnt, &SpreadRow::cells, head ? 1u : 0u);
    const uint64_t heads = __ballot(head);
    const uint32_t code = (uint32_t)(k & 0x3FFFFFFFull);
    if (t.mbits) {
        if (s < n) {
            t.mlist[s] = head ? code >> 5 : UNSET;
            t.crank[s] = head ? 1u : 0u;
        }
        // the wave's cells are consecutive in Morton order and share bitmap words: one
        // atomic per distinct word, with the bits of every head in the wave that names it
        uint64_t todo = heads;
        while (todo) {
            const uint32_t lead = (uint32_t)__ffsll((unsigned long long)todo) - 1u;
            const uint32_t word = __shfl(code >> 5, (int)lead, 64);
            const bool mine = head && (code >> 5) == word;
            uint32_t b = mine ? 1u << (code & 31u) : 0u;
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) b |= __shfl_xor(b, o, 64);
            if (lane == lead) atomicOr(&t.mbits[word], b);
            todo &= ~__ballot(mine);
        }
        return;  // cells are found by rank (k_cell_rank), no hash table
    }
    if (!head) return;
    __hip_atomic_store(reinterpret_cast<uint64_t*>(&t.ent[(uint32_t)mix64(k) & t.mask]), k, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    if (!t.mbits) {
        const uint32_t bit = cell_bit(mix64(k), t.bmask);
        atomicOr(&t.bits[bit >> 5], 1u << (bit & 31u));
    }
}
// With the Morton bitmap (crank holds the exclusive scan of the cell heads): each cell's
// first sorted position by rank, and each bitmap word's rank base (its first cell's rank).
// Also decides the broadphase mode of the step (bp_sparse: fewer than four bodies per
// occupied cell), as k_cell_place does in the hash mode.
__device__ __forceinline__ void decide_mode(Counters* cnt, uint32_t n) {
    cnt->bp_sparse = (uint64_t)spread_sum(cnt, &SpreadRow::cells) * 4u > n ? 1u : 0u;
}
__global__ void __launch_bounds__(256) k_cell_rank(SortedKeys skey, uint32_t n, CellTable t,
                                                   Counters* __restrict__ cnt) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s == 0u) decide_mode(cnt, n);
    if (s >= n) return;
    const uint64_t k = skey[s];
    const uint64_t kp = s ? skey[s - 1u] : EMPTY_KEY;
    const uint32_t r = t.crank[s];
    const bool head = s == 0u || kp != k;
    if (head) {
        t.cstart[r] = s;
        const uint32_t word = (uint32_t)(k & 0x3FFFFFFFull) >> 5;
        if (s == 0u || ((uint32_t)(kp & 0x3FFFFFFFull) >> 5) != word) t.wrank[word] = r;
    }
    if (s == n - 1u) t.cstart[r + (head ? 1u : 0u)] = n;
}
__global__ void __launch_bounds__(256) k_cell_place(SortedKeys skey, uint32_t n, CellTable t,
                                                    Counters* __restrict__ cnt) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t lane = __lane_id();
    if (s == 0u) decide_mode(cnt, n);
    const uint64_t k = s < n ? skey[s] : EMPTY_KEY;
    const bool head = s < n && (s == 0 || skey[s - 1] != k);
    const uint64_t heads = __ballot(head);
    if (!head) return;
    // the cell's count: up to the next head in the wave, else read on past the wave
    const uint64_t above = lane == 63u ? 0ull : heads & (~0ull << (lane + 1u));
    uint32_t c;
    if (above) {
        c = (uint32_t)__ffsll((unsigned long long)above) - 1u - lane;
    } else {
        c = 64u - lane;
        while (s + c < n && skey[s + c] == k) ++c;
        if (s + c > n) c = n - s;
    }
    const uint32_t h = (uint32_t)mix64(k) & t.mask;
    if (*reinterpret_cast<const uint64_t*>(&t.ent[h]) == k) {
        reinterpret_cast<uint2*>(&t.ent[h])[1] = make_uint2(s, c);
    } else if (!ht_insert(t, k, make_uint2(s, c), (h + 1u) & t.mask)) {
        atomicOr(&cnt->sticky, STICKY_INTERNAL);
    }
}

// ---------------------------------------------------------------- XCD-aware block order
// Workgroups are dispatched round-robin over the 8 XCDs (workgroup b runs on XCD b % 8),
// and each XCD has its own L2.  Kernels whose neighbouring items share gathered data
// and cost about the same (the pair kernels: neighbour cells of bodies in Morton order)
// take their block index from here instead: each XCD gets one contiguous run of blocks,
// so the shared lines stay in one L2.  Not for lists sorted by cost (pairs by kind,
// manifolds by island), where contiguous runs would load some XCDs far more than
// others.  A bijection of 0..gridDim.x-1, so a kernel that writes by item index is
// unchanged.
__device__ __forceinline__ uint32_t xcd_block() {
    const uint32_t G = gridDim.x, b = blockIdx.x;
    const uint32_t per = G >> 3, rem = G & 7u, x = b & 7u;
    return x * per + min(x, rem) + (b >> 3);
}

// ---------------------------------------------------------------- pairs
// Visits candidate partners of the body at sorted position t in the canonical
// order: planes, then the 27 neighbour cells (dz, dy, dx in -1..1), then
// ascending sorted position.  f(partner) is called for every emitted pair.
// AABBs in sorted order (k_cell_table): smin = (min, body index bits), smax = (max,
// 1 if dynamic).  The broadphase mode of the step (k_cell_rank / k_cell_place) is
// sparse when there are fewer than four bodies per occupied cell (the pair kernels
// come in a sparse and a dense build, each with only the registers its mode needs,
// and the one not chosen returns at once).

// Collision filter of two bodies (flags, category, mask, group): a shared nonzero group
// decides (positive: always, negative: never), else each category must meet the other's mask.
__device__ __forceinline__ bool should_collide(uint4 a, uint4 b) {
    const int ga = (int)a.w, gb = (int)b.w;
    if (ga == gb && ga != 0) return ga > 0;
    return (a.z & b.y) != 0u && (a.y & b.z) != 0u;
}

// Broadphase modes: cells found by rank in the occupancy bitmap (one large world), or
// through the hash table with few bodies per occupied cell (occupancy bits first) or
// many.  Each mode is its own kernel build, with only the registers its path needs.
constexpr int BP_RANK = 0, BP_SPARSE = 1, BP_DENSE = 2;

// The candidates of sorted body t in z slice dz (-1, 0, 1) of its neighbour cells,
// in canonical order; the planes come with slice -1.
template <int MODE, class F>
__device__ __forceinline__ void visit_pairs(const Bodies& B, const StepParams& sp, const SortedKeys& skey,
                                            const uint32_t* __restrict__ sval, const CellTable& ct, uint32_t t,
                                            int dz, F&& f) {
    const uint64_t key = MODE == BP_RANK ? (uint64_t)skey.k32[t] : skey.k64[t];
    const float4 mn = B.smin[t], mx = B.smax[t];
    const uint32_t i = __float_as_uint(mn.w);
    const bool dyn_i = mx.w > 0.0f;
    if (dyn_i && dz < 0) {
        const f3 c = xyz(B.x[i]);
        const f3 e = xyz(mx) - c;
        for (uint32_t k = 0; k < sp.num_planes; ++k) {
            const float4 pl = sp.planes[k];
            const float s = (pl.x * c.x + pl.y * c.y + pl.z * c.z) -
                            (fabsf(pl.x) * e.x + fabsf(pl.y) * e.y + fabsf(pl.z) * e.z);
            if (s <= pl.w) f(PLANE_BIT | k);
        }
    }
    const uint32_t mort = (uint32_t)(key & 0x3FFFFFFFull);
    const uint64_t wbits = key & ~0x3FFFFFFFull;
    const int cx = (int)compact1by2(mort), cy = (int)compact1by2(mort >> 1), cz = (int)compact1by2(mort >> 2);
    const int Z = cz + dz;
    if (Z < 0 || Z > 1023) return;
    // the cell's bodies in sorted order, four loaded at a time (a dense cell holds
    // dozens, and each load of the loop would otherwise wait on its own)
    auto test = [&](const float4 mnj, const float4 mxj) {
        const uint32_t j = __float_as_uint(mnj.w);
        if (j <= i) return;
        if (!dyn_i && !(mxj.w > 0.0f)) return;
        if (mn.x <= mxj.x && mx.x >= mnj.x && mn.y <= mxj.y && mx.y >= mnj.y && mn.z <= mxj.z && mx.z >= mnj.z) {
            if (sp.use_filter && !should_collide(B.bfl[i], B.bfl[j])) return;
            f(j);
        }
    };
    auto visit_range = [&](uint2 r) {
        const uint32_t se = r.x + r.y;
        uint32_t s = r.x;
        for (; s + 4u <= se; s += 4u) {
            float4 mn4[4], mx4[4];
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) {
                mn4[u] = B.smin[s + u];
                mx4[u] = B.smax[s + u];
            }
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) test(mn4[u], mx4[u]);
        }
        for (; s < se; ++s) test(B.smin[s], B.smax[s]);
    };
    // the nine cells of this z slice in canonical (dy, dx) order; Morton codes from the
    // dilated coordinates (three per axis instead of nine full interleavings)
    uint32_t px[3], py[3];
    bool okx[3], oky[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int X = cx + a - 1, Y = cy + a - 1;
        okx[a] = X >= 0 && X <= 1023;
        oky[a] = Y >= 0 && Y <= 1023;
        px[a] = part1by2((uint32_t)(okx[a] ? X : 0));
        py[a] = part1by2((uint32_t)(oky[a] ? Y : 0)) << 1;
    }
    const uint32_t pz = part1by2((uint32_t)Z) << 2;
    if constexpr (MODE == BP_RANK) {
        // one large world: the nine occupancy words are read once (they stay in the cache);
        // an occupied cell's range comes by rank from two arrays in Morton order
        // per cell: occupied, and the occupied cells of its word below it (5 bits each, six
        // to a register, so the nine words need not stay in registers)
        uint32_t occ = 0, below0 = 0, below1 = 0;
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            const uint32_t code = px[q % 3] | py[q / 3] | pz;
            const uint32_t wv = okx[q % 3] && oky[q / 3] ? ct.mbits[code >> 5] : 0u;
            occ |= ((wv >> (code & 31u)) & 1u) << q;
            const uint32_t b = (uint32_t)__popc(wv & ((1u << (code & 31u)) - 1u));
            if (q < 6) below0 |= b << (5 * q);
            else below1 |= b << (5 * (q - 6));
        }
        while (occ) {
            const int q = __ffs(occ) - 1;
            occ &= occ - 1u;
            const uint32_t code = px[q % 3] | py[q / 3] | pz;
            const uint32_t below = (q < 6 ? below0 >> (5 * q) : below1 >> (5 * (q - 6))) & 31u;
            const uint32_t k = ct.wrank[code >> 5] + below;
            const uint32_t s0 = ct.cstart[k];
            visit_range(make_uint2(s0, ct.cstart[k + 1u] - s0));
        }
        return;
    }
    if constexpr (MODE == BP_SPARSE) {
        // few bodies per occupied cell: the occupancy bits (which stay in the cache) are
        // read first, then only the occupied cells are hashed and probed, in order
        uint32_t occ = 0;
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            const uint32_t code = px[q % 3] | py[q / 3] | pz;
            const uint32_t bit = cell_bit(mix64(wbits | code), ct.bmask);
            const bool on = okx[q % 3] && oky[q / 3] && ((ct.bits[bit >> 5] >> (bit & 31u)) & 1u) != 0u;
            occ |= on ? 1u << q : 0u;
        }
        while (occ) {
            const int q = __ffs(occ) - 1;
            occ &= occ - 1u;
            const uint64_t nk = wbits | (px[q % 3] | py[q / 3] | pz);
            const uint32_t hs = (uint32_t)mix64(nk) & ct.mask;
            const uint4 e = ct.ent[hs];
            const uint64_t kk = ent_key(e);
            if (kk == EMPTY_KEY) continue;
            uint2 r = make_uint2(e.z, e.w);
            if (kk != nk && !ht_find_from(ct, nk, (hs + 1u) & ct.mask, r)) continue;
            visit_range(r);
        }
        return;
    }
    // dense: the first probes of all nine cells in flight together
    uint64_t nk[9];
    uint4 e[9];
    uint32_t hs[9];
    bool ok[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) {
        ok[q] = okx[q % 3] && oky[q / 3];
        nk[q] = wbits | (px[q % 3] | py[q / 3] | pz);
        hs[q] = (uint32_t)mix64(nk[q]) & ct.mask;
    }
#pragma unroll
    for (int q = 0; q < 9; ++q)
        e[q] = ok[q] ? ct.ent[hs[q]] : make_uint4((uint32_t)EMPTY_KEY, (uint32_t)(EMPTY_KEY >> 32), 0u, 0u);
#pragma unroll
    for (int q = 0; q < 9; ++q) {
        const uint64_t kk = ent_key(e[q]);
        if (!ok[q] || kk == EMPTY_KEY) continue;
        uint2 r = make_uint2(e[q].z, e[q].w);
        if (kk != nk[q] && !ht_find_from(ct, nk[q], (hs[q] + 1u) & ct.mask, r)) continue;
        visit_range(r);
    }
}

// Exclusive scan over a 256-thread workgroup (four waves); the workgroup's total in `total`.
__device__ __forceinline__ uint32_t wg_excl_scan(uint32_t v, uint32_t& total) {
    __shared__ uint32_t s_w[4];
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    uint32_t inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(inc, o, 64);
        if (lane >= (uint32_t)o) inc += t;
    }
    if (lane == 63u) s_w[wv] = inc;
    __syncthreads();
    uint32_t base = 0, tot = 0;
#pragma unroll
    for (uint32_t w = 0; w < 4u; ++w) {
        const uint32_t x = s_w[w];
        if (w < wv) base += x;
        tot += x;
    }
    __syncthreads();
    total = tot;
    return base + inc - v;
}

// Counts the pairs of each (body, z slice) part u = 3 t + dz + 1 and keeps the
// first PAIR_STASH partners, so that the emit pass only re-visits the grid for the
// few parts with more.  Three threads per body: the probes of a body's slices are
// in flight together.
// The workgroup's total goes to bsum[block] (block in the XCD-aware order): the emit pass
// forms each part's offset from the scanned totals and a scan within its workgroup.
template <int MODE>
__device__ __forceinline__ void pair_count_body(const Bodies& B, const StepParams& sp, const SortedKeys& skey,
                                                const uint32_t* __restrict__ sval, const CellTable& ct, uint32_t n,
                                                uint32_t* __restrict__ cnt, uint32_t* __restrict__ bsum,
                                                uint32_t* __restrict__ stash, const Counters* __restrict__ ctr) {
    if (MODE != BP_RANK && (ctr->bp_sparse != 0u) != (MODE == BP_SPARSE)) return;
    const uint32_t lb = xcd_block();
    const uint32_t u = lb * blockDim.x + threadIdx.x;
    uint32_t c = 0;
    if (u < BP_PARTS * n) {
        const uint32_t t = u / BP_PARTS;
        const int dz = (int)(u - BP_PARTS * t) - 1;
        uint32_t* st = stash + (size_t)u * PAIR_STASH;
        visit_pairs<MODE>(B, sp, skey, sval, ct, t, dz, [&](uint32_t j) {
            if (c < PAIR_STASH) st[c] = j;
            ++c;
        });
        cnt[u] = c;
    }
    uint32_t tot;
    (void)wg_excl_scan(c, tot);
    if (threadIdx.x == 0u) bsum[lb] = tot;
}
// The rank and sparse builds fit 64 registers without scratch, so eight waves per SIMD
// hide more of the probe latency; the dense build keeps its registers.
template <int MODE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8)))
k_pair_count(Bodies B, StepParams sp, SortedKeys skey, const uint32_t* __restrict__ sval,
             CellTable ct, uint32_t n, uint32_t* __restrict__ cnt, uint32_t* __restrict__ bsum,
             uint32_t* __restrict__ stash, const Counters* __restrict__ ctr) {
    pair_count_body<MODE>(B, sp, skey, sval, ct, n, cnt, bsum, stash, ctr);
}
__global__ void __launch_bounds__(256)
k_pair_count_dense(Bodies B, StepParams sp, SortedKeys skey, const uint32_t* __restrict__ sval,
                   CellTable ct, uint32_t n, uint32_t* __restrict__ cnt, uint32_t* __restrict__ bsum,
                   uint32_t* __restrict__ stash, const Counters* __restrict__ ctr) {
    pair_count_body<BP_DENSE>(B, sp, skey, sval, ct, n, cnt, bsum, stash, ctr);
}

// Part u's pairs start at boff[block] (the scanned workgroup totals; boff[blocks] is the
// pair count) plus the counts of the parts before it in its workgroup.
template <int MODE>
__global__ void __launch_bounds__(256) k_pair_emit(Bodies B, StepParams sp, SortedKeys skey,
                                                   const uint32_t* __restrict__ sval, CellTable ct, uint32_t n,
                                                   const uint32_t* __restrict__ pcnt, const uint32_t* __restrict__ boff,
                                                   uint32_t cap, uint32_t* __restrict__ pa, uint32_t* __restrict__ pb,
                                                   Counters* __restrict__ cnt, const uint32_t* __restrict__ stash) {
    if (MODE != BP_RANK && (cnt->bp_sparse != 0u) != (MODE == BP_SPARSE)) return;
    const uint32_t lb = xcd_block();
    const uint32_t u = lb * blockDim.x + threadIdx.x;
    const uint32_t parts = BP_PARTS * n;
    if (u == 0) {
        const uint32_t P = boff[(parts + 255u) / 256u];
        cnt->p_eff = P < cap ? P : cap;
        if (P > cap) atomicOr(&cnt->sticky, STICKY_PAIRS);
    }
    const uint32_t c = u < parts ? pcnt[u] : 0u;
    uint32_t tot;
    const uint32_t ex = wg_excl_scan(c, tot);
    if (u >= parts) return;
    const uint32_t t = u / BP_PARTS;
    const int dz = (int)(u - BP_PARTS * t) - 1;
    uint32_t o = boff[lb] + ex;
    const uint32_t i = sval[t];
    if (c <= PAIR_STASH) {
        const uint32_t* st = stash + (size_t)u * PAIR_STASH;
        for (uint32_t k = 0; k < c && o + k < cap; ++k) {
            pa[o + k] = i;
            pb[o + k] = st[k];
        }
        return;
    }
    visit_pairs<MODE>(B, sp, skey, sval, ct, t, dz, [&](uint32_t j) {
        if (o < cap) {
            pa[o] = i;
            pb[o] = j;
        }
        ++o;
    });
}

// ---------------------------------------------------------------- narrowphase
__device__ __forceinline__ Shp load_shape(const Bodies& B, uint32_t i) {
    Shp s;
    const float4 sh = B.shape[i];
    s.c = xyz(B.x[i]);
    s.R = quat_to_mat(B.q[i]);
    s.type = fbits(sh.w);
    s.prm = xyz(sh);
    return s;
}

__device__ __forceinline__ void store_pair(uint32_t p, const Man& m, uint32_t* __restrict__ p_np,
                                           float4* __restrict__ p_pt, float4* __restrict__ p_nf) {
    p_np[p] = m.np;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        if (k >= m.np) break;
        p_pt[(size_t)p * 4 + k] = f4(m.pt[k].p, m.pt[k].depth);
        p_nf[(size_t)p * 4 + k] = f4(m.pt[k].n, __uint_as_float(m.pt[k].fid));
    }
}

// Processing order of the narrowphase: pairs grouped by the kind of test (the two
// shape types, or the shape type against a plane), so that a wave runs one test
// rather than every test its lanes need.  Results stay indexed by pair (PAIR_KINDS
// kinds, defined with the step counters).
__device__ __forceinline__ uint32_t pair_kind(const Bodies& B, uint32_t a, uint32_t b) {
    const uint32_t ta = fbits(B.shape[a].w) & 3u;
    if (b & PLANE_BIT) return 12u + ta;
    const uint32_t tb = fbits(B.shape[b].w) & 3u;
    const uint32_t lo = ta < tb ? ta : tb, hi = ta < tb ? tb : ta;
    return lo * 4u + hi;
}
// Per pair its kind; per kind the count (kinds[0..15]; kinds[16..31] are the fill
// cursors of k_pair_order, both cleared at the step start).
__global__ void __launch_bounds__(256) k_pair_kind(Bodies B, const uint32_t* __restrict__ pa,
                                                   const uint32_t* __restrict__ pb, uint32_t* __restrict__ p_kind,
                                                   uint32_t* __restrict__ kinds, const Counters* __restrict__ cnt) {
    __shared__ uint32_t h[PAIR_KINDS];
    if (threadIdx.x < PAIR_KINDS) h[threadIdx.x] = 0u;
    __syncthreads();
    const uint32_t P = cnt->p_eff;
    for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < P; p += gridDim.x * blockDim.x) {
        const uint32_t k = pair_kind(B, pa[p], pb[p]);
        p_kind[p] = k;
        atomicAdd(&h[k], 1u);
    }
    __syncthreads();
    if (threadIdx.x < PAIR_KINDS && h[threadIdx.x]) atomicAdd(&kinds[threadIdx.x], h[threadIdx.x]);
}
__global__ void __launch_bounds__(256) k_pair_order(const uint32_t* __restrict__ p_kind, uint32_t* __restrict__ kinds,
                                                    uint32_t* __restrict__ order, const Counters* __restrict__ cnt) {
    __shared__ uint32_t base[PAIR_KINDS], off[PAIR_KINDS], h[PAIR_KINDS];
    const uint32_t P = cnt->p_eff;
    if (threadIdx.x < PAIR_KINDS) {
        uint32_t o = 0;
        for (uint32_t k = 0; k < threadIdx.x; ++k) o += kinds[k];
        base[threadIdx.x] = o;
    }
    // a bounded grid strides over the pairs (block-uniform trip count: the barriers below)
    for (uint32_t b0 = blockIdx.x * blockDim.x; b0 < P; b0 += gridDim.x * blockDim.x) {
        const uint32_t p = b0 + threadIdx.x;
        if (threadIdx.x < PAIR_KINDS) h[threadIdx.x] = 0u;
        __syncthreads();
        const uint32_t k = p < P ? p_kind[p] : 0u;
        const uint32_t r = p < P ? atomicAdd(&h[k], 1u) : 0u;
        __syncthreads();
        if (threadIdx.x < PAIR_KINDS)
            off[threadIdx.x] = base[threadIdx.x] +
                               (h[threadIdx.x] ? atomicAdd(&kinds[PAIR_KINDS + threadIdx.x], h[threadIdx.x]) : 0u);
        __syncthreads();
        if (p < P) {
            const uint32_t q = off[k] + r;
            if (q < P) order[q] = p;
        }
        __syncthreads();
    }
}

// The heavy tests (box-box, box-capsule) run in a kernel of their own, so that the
// other tests keep a small register allocation and no scratch memory.  In the
// kind-sorted order the heavy pairs are one contiguous range [h0, h1).
constexpr uint32_t KIND_BOX_BOX = 1u * 4u + 1u, KIND_BOX_CAPSULE = 1u * 4u + 2u;
static_assert(KIND_BOX_CAPSULE == KIND_BOX_BOX + 1u, "heavy kinds are adjacent");
template <bool HEAVY>
__global__ void __launch_bounds__(256) k_narrow(Bodies B, StepParams sp, const uint32_t* __restrict__ pa,
                                                const uint32_t* __restrict__ pb, uint32_t* __restrict__ p_np,
                                                float4* __restrict__ p_pt, float4* __restrict__ p_nf,
                                                uint32_t* __restrict__ epa_list, Counters* __restrict__ cnt,
                                                const uint32_t* __restrict__ order, const uint32_t* __restrict__ kinds) {
    const uint32_t P = cnt->p_eff;
    uint32_t h0 = 0;
    for (uint32_t k = 0; k < KIND_BOX_BOX; ++k) h0 += kinds[k];
    uint32_t h1 = h0 + kinds[KIND_BOX_BOX] + kinds[KIND_BOX_CAPSULE];
    h1 = min(h1, P);
    h0 = min(h0, h1);
    const uint32_t nh = h1 - h0, N = HEAVY ? nh : P - nh;
    for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < N; v += gridDim.x * blockDim.x) {
    const uint32_t t = HEAVY ? h0 + v : (v < h0 ? v : v + nh);
    const uint32_t p = order[t];
    const uint32_t a = pa[p], b = pb[p];
    Man m;
    m.np = 0;
    const Shp A = load_shape(B, a);
    if (!HEAVY && (b & PLANE_BIT)) {
        const float4 pl = sp.planes[b & ~PLANE_BIT];
        collide_plane(m, A, f3{pl.x, pl.y, pl.z}, pl.w, sp.margin);
    } else {
        const Shp Bs = load_shape(B, b);
        bool need_epa = false;
        // the shapes are put in order by selects: a branch on the order would run the tests twice
        // in a wave with both (a pile of 6000 bodies: 42 us, so 28)
        const bool swap = A.type > Bs.type;
        constexpr int TESTS = HEAVY ? COLLIDE_HEAVY : COLLIDE_LIGHT;
        const int st = collide_canon<TESTS>(m, select_shape(swap, Bs, A), select_shape(swap, A, Bs), sp.margin, need_epa);
        if (need_epa) {
            const uint32_t slot = atomicAdd(&cnt->epa_count, 1u);
            epa_list[slot] = p;
        } else if (swap) {
            flip_manifold(m);
        }
        if (st == GEOM_GJK_FAIL) atomicAdd(&cnt->gjk_fail, 1u);
    }
    store_pair(p, m, p_np, p_pt, p_nf);
    }
}

// Deep box-capsule pairs (cores intersect): EPA, one queued pair per wave at a time (a fixed
// grid strides over the queue).
__global__ void __launch_bounds__(64) k_narrow_epa(Bodies B, StepParams sp, const uint32_t* __restrict__ pa,
                                                   const uint32_t* __restrict__ pb,
                                                   const uint32_t* __restrict__ epa_list, uint32_t cap,
                                                   uint32_t* __restrict__ p_np, float4* __restrict__ p_pt,
                                                   float4* __restrict__ p_nf, Counters* __restrict__ cnt) {
    const uint32_t nq = min(cnt->epa_count, cap);
    __shared__ EpaWork W;
    for (uint32_t q = blockIdx.x; q < nq; q += gridDim.x) {
        const uint32_t p = epa_list[q];
        const uint32_t a = pa[p], b = pb[p];
        Shp A = load_shape(B, a), Bs = load_shape(B, b);
        const bool swap = A.type > Bs.type;
        Man m;
        m.np = 0;
        const int st = box_capsule_epa(m, select_shape(swap, Bs, A), select_shape(swap, A, Bs), W);
        if (swap) flip_manifold(m);
        if (threadIdx.x != 0u) continue;
        if (st == GEOM_EPA_FAIL) atomicAdd(&cnt->epa_fail, 1u);
        store_pair(p, m, p_np, p_pt, p_nf);
    }
}

__global__ void __launch_bounds__(256) k_compact(const uint32_t* __restrict__ pa, const uint32_t* __restrict__ pb,
                                                 const uint32_t* __restrict__ p_np,
                                                 const float4* __restrict__ p_pt, const float4* __restrict__ p_nf,
                                                 const uint32_t* __restrict__ moff, uint32_t cap,
                                                 uint2* __restrict__ m_ab, uint32_t* __restrict__ m_np,
                                                 float4* __restrict__ c_pt, float4* __restrict__ c_nf,
                                                 Counters* __restrict__ cnt) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const uint32_t M = cnt->manifolds;
        cnt->m_eff = M < cap ? M : cap;
        if (M > cap) atomicOr(&cnt->sticky, STICKY_MANIFOLDS);
    }
    const uint32_t P = cnt->p_eff;
    uint32_t contacts = 0;
    for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < P; p += gridDim.x * blockDim.x) {
        const uint32_t np = p_np[p];
        contacts += np;
        if (np == 0) continue;
        const uint32_t m = moff[p];
        if (m >= cap) continue;
        m_ab[m] = make_uint2(pa[p], pb[p]);
        m_np[m] = np;
        for (uint32_t k = 0; k < np; ++k) {
            c_pt[(size_t)m * 4 + k] = p_pt[(size_t)p * 4 + k];
            c_nf[(size_t)m * 4 + k] = p_nf[(size_t)p * 4 + k];
        }
    }
    spread_add(cnt, &SpreadRow::contacts, contacts);
}

// ---------------------------------------------------------------- colouring
__device__ __forceinline__ bool dyn_body(const Bodies& B, uint32_t b) {
    return !(b & PLANE_BIT) && B.sv[b].w > 0.0f;
}
__device__ __forceinline__ uint32_t local_id(const Bodies& B, uint32_t b) {
    return (b & PLANE_BIT) ? b : b - B.world_first[B.world[b]];
}

// Grid-wide barrier for a kernel whose workgroups are all resident (grid sized
// from the occupancy query).  Every wave first waits until its own stores are
// complete in the XCD's L2 (a workgroup barrier does not wait for them); then one
// thread per workgroup writes the L2 back and arrives (agent-scope release), waits
// for the last arrival and invalidates the stale L1/L2 lines for the whole
// workgroup (agent-scope acquire).  One writeback per workgroup instead of one per
// wave: the writeback of an XCD's L2 is the expensive part of a fence.  A bounded
// wait sets STICKY_TIMEOUT instead of hanging.
// Grid barrier over `nblocks` resident workgroups.  The last workgroup to arrive
// copies *snap (a counter the workgroups update before arriving) into the barrier
// before releasing it, and every workgroup returns that copy: all of them see the
// value as it stood when the whole grid had arrived, even if a fast workgroup
// already updates the counter again in the next round.
__device__ __forceinline__ uint32_t grid_sync(GridBar* bar, uint32_t nblocks, Counters* cnt, const uint32_t* snap) {
    __shared__ uint32_t s_snap;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t g = __hip_atomic_load(&bar->gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t arrived = __hip_atomic_fetch_add(&bar->count, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (arrived == nblocks - 1) {
            const uint32_t v = __hip_atomic_load(snap, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&bar->pad[0], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&bar->count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_fetch_add(&bar->gen, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            s_snap = v;
        } else {
            const uint64_t t0 = wall_clock64();  // 100 MHz constant clock
            bool late = false;
            while (__hip_atomic_load(&bar->gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == g) {
                __builtin_amdgcn_s_sleep(2);
                if (wall_clock64() - t0 > 200000000ull) {  // 2 s
                    atomicOr(&cnt->sticky, STICKY_TIMEOUT);
                    late = true;
                    break;
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            s_snap = late ? 0u : __hip_atomic_load(&bar->pad[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    __syncthreads();
    return s_snap;
}

// Jones-Plassmann colouring in one persistent launch.  Round r: every
// uncoloured manifold offers tag(r, m) = (r+1) << 48 | hash24(a,b) << 24 | m at
// its dynamic bodies (atomic max into the round's buffer); a manifold holding
// the max at all its dynamic bodies takes the first colour free in both bodies'
// 64-bit masks (64 + r once they are full).  Winners of one round share no
// dynamic body, so their mask updates cannot collide.  Losers offer their next
// tag into the other buffer in the same pass, so each round costs one barrier;
// tags grow with the round, so the buffers never need clearing.
struct PrevCache {
    const uint64_t* key;  // (a << 32 | b) -> previous slot
    const uint32_t* slot;
    uint32_t mask;
    const float4* lam;    // [k * cap + s]
    const uint32_t* fid;  // [k * cap + s]
    const uint32_t* np;   // points per previous slot
    const uint32_t* colour;  // colour per previous slot
    uint32_t cap;
    uint32_t valid;
};

__device__ __forceinline__ bool prev_find(const PrevCache& c, uint64_t k, uint32_t& s) {
    uint32_t h = (uint32_t)mix64(k) & c.mask;
    for (uint32_t probe = 0; probe <= c.mask; ++probe) {
        const uint64_t kk = c.key[h];
        if (kk == k) {
            s = c.slot[h];
            return true;
        }
        if (kk == EMPTY_KEY) return false;
        h = (h + 1) & c.mask;
    }
    return false;
}

// Per-island atomics of a wave: the lanes whose island is that of the first lane taking
// part combine their values into one atomic made by that lane; the others make their own.
// In one giant island a wave makes one atomic instead of 64 on the same word.
template <class Op>
__device__ __forceinline__ void wave_by_island(bool on, uint32_t r, uint32_t v, uint32_t idle, Op op) {
    const uint64_t act = __ballot(on);
    if (act == 0ull) return;
    const uint32_t lead = (uint32_t)__ffsll((unsigned long long)act) - 1u;
    const uint32_t lr = (uint32_t)__shfl((int)r, (int)lead, 64);
    const bool same = on && r == lr;
    uint32_t c = same ? v : idle;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) c = op.combine(c, (uint32_t)__shfl_xor((int)c, o, 64));
    if (__lane_id() == lead) op.apply(lr, c);
    if (on && !same) op.apply(r, v);
}
// Manifolds per island (after the union kernel), run by the colouring's first launch
// (k_colour_keep), every thread of its grid.
__device__ __forceinline__ void isl_count_part(const Bodies& B, const uint2* __restrict__ m_ab, uint32_t cap,
                                               const Counters* __restrict__ cnt) {
    if (cnt->sticky != 0u) return;
    const uint32_t M = min(cap, cnt->m_eff);
    struct Add {
        uint32_t* icnt;
        __device__ uint32_t combine(uint32_t a, uint32_t b) const { return a + b; }
        __device__ void apply(uint32_t r, uint32_t c) const { atomicAdd(icnt + r, c); }
    };
    // every lane of a wave runs the same number of rounds (the wave-wide combine)
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t m0 = blockIdx.x * blockDim.x + (threadIdx.x & ~63u); m0 < M; m0 += stride) {
        const uint32_t m = m0 + __lane_id();
        const uint32_t r = m < M ? man_root(B, m_ab[m]) : UNSET;
        wave_by_island(r != UNSET, r, 1u, 0u, Add{B.icnt});
    }
}
// Pass 1 (one thread per manifold, no barrier): degrees, priorities, the kept
// colours of persisting contacts (with their mask bits) and, for every other
// manifold, its round-0 tag at its dynamic bodies and an entry in the list of
// manifolds to colour (cnt->remaining counts them).  The per-body arrays were
// cleared by k_begin.  Temporal coherence: between full recolourings (every
// recolour_period steps) a manifold whose body pair was in contact in the
// previous step keeps that step's colour (the kept ones stay a valid colouring:
// a subset of one); Jones-Plassmann then colours only the others around them.
__global__ void __launch_bounds__(256) k_colour_keep(Bodies B, const uint2* __restrict__ m_ab,
                                                     uint32_t* __restrict__ col, uint64_t* __restrict__ prio,
                                                     uint64_t* __restrict__ bmax0, uint64_t* __restrict__ bmask,
                                                     uint32_t* __restrict__ bdeg, uint32_t* __restrict__ list,
                                                     Counters* cnt, PrevCache pc, uint32_t recolour_period,
                                                     uint32_t count_cap) {
    // with the island split, the manifolds per island first (count_cap: the manifold capacity)
    if (count_cap) isl_count_part(B, m_ab, count_cap, cnt);
    const uint32_t M = cnt->m_eff;
    const bool incremental = pc.valid != 0u && (cnt->steps_done % recolour_period) != 0u;
    // per workgroup, the largest kept colour and the list entries are gathered in LDS
    // and go out with one atomic each (atomics on one address queue one after another)
    __shared__ uint32_t s_cmax, s_n, s_base;
    // a bounded grid strides over the manifolds (block-uniform trip count: the barriers below)
    for (uint32_t b0 = blockIdx.x * blockDim.x; b0 < M; b0 += gridDim.x * blockDim.x) {
        const uint32_t m = b0 + threadIdx.x;
        if (threadIdx.x == 0) {
            s_cmax = 0u;
            s_n = 0u;
        }
        __syncthreads();
        bool fresh = false;
        if (m < M) {
            const uint2 ab = m_ab[m];
            const bool bd = dyn_body(B, ab.y);
            atomicAdd(&bdeg[ab.x], 1u);
            if (bd) atomicAdd(&bdeg[ab.y], 1u);
            const uint64_t pr =
                ((uint64_t)pair_hash24(local_id(B, ab.x), local_id(B, ab.y)) << 24) | (uint64_t)(m & 0xFFFFFFu);
            prio[m] = pr;
            uint32_t c = UNSET, ps;
            if (incremental && prev_find(pc, ((uint64_t)ab.x << 32) | ab.y, ps)) {
                const uint32_t pcol = pc.colour[ps];
                if (pcol < 64u) c = pcol;
            }
            col[m] = c;
            if (c != UNSET) {
                atomicOr((unsigned long long*)&bmask[ab.x], 1ull << c);
                if (bd) atomicOr((unsigned long long*)&bmask[ab.y], 1ull << c);
                atomicMax(&s_cmax, c + 1u);
            } else {
                const uint64_t t = (1ull << 48) | pr;
                atomicMax((unsigned long long*)&bmax0[ab.x], (unsigned long long)t);
                if (bd) atomicMax((unsigned long long*)&bmax0[ab.y], (unsigned long long)t);
                fresh = true;
            }
        }
        // list entries of the manifolds to colour: a slot range per wave within the workgroup's
        const unsigned long long fb = __ballot(fresh);
        const uint32_t lane = __lane_id();
        uint32_t wbase = 0;
        if (fb && lane == 0u) wbase = atomicAdd(&s_n, (uint32_t)__popcll(fb));
        wbase = __shfl(wbase, 0, 64);
        __syncthreads();
        if (threadIdx.x == 0) {
            if (s_cmax) atomicMax(&cnt->max_colour, s_cmax);
            s_base = s_n ? atomicAdd(&cnt->remaining, s_n) : 0u;
        }
        __syncthreads();
        if (fresh) list[s_base + wbase + (uint32_t)__popcll(fb & ((1ull << lane) - 1ull))] = m;
        __syncthreads();  // s_base and s_n are reset by the next iteration
    }
}

// One Jones-Plassmann visit of list entry m in round r: a manifold holding the
// round's tag at all its dynamic bodies takes the first colour free in both
// bodies' 64-bit masks (64 + r once they are full); a loser offers its next tag
// into the other buffer.  Winners of one round share no dynamic body, so their
// mask updates cannot collide; tags grow with the round, so the buffers never
// need clearing.  AT: shared words through agent-scope atomics (the one-workgroup
// form, which has no cache invalidation between rounds).
template <bool AT>
__device__ __forceinline__ void jp_visit(const Bodies& B, const uint2* __restrict__ m_ab, uint32_t* __restrict__ col,
                                         const uint64_t* __restrict__ prio, const uint64_t* cur, uint64_t* nxt,
                                         uint64_t* bmask, uint32_t m, uint32_t r, uint32_t& won, uint32_t& cmax) {
    if (col[m] != UNSET) return;
    auto ld = [](const uint64_t* p) -> uint64_t {
        if constexpr (AT) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else return *p;
    };
    auto st = [](uint64_t* p, uint64_t v) {
        if constexpr (AT) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else *p = v;
    };
    const uint2 ab = m_ab[m];
    const bool bd = dyn_body(B, ab.y);
    const uint64_t t = ((uint64_t)(r + 1) << 48) | prio[m];
    if (ld(&cur[ab.x]) == t && (!bd || ld(&cur[ab.y]) == t)) {
        const uint64_t ma = ld(&bmask[ab.x]), mb = bd ? ld(&bmask[ab.y]) : 0ull;
        const uint64_t used = ma | mb;
        uint32_t c;
        if (~used == 0ull) {
            c = 64u + r;
        } else {
            c = (uint32_t)__ffsll((unsigned long long)~used) - 1u;
            st(&bmask[ab.x], ma | (1ull << c));
            if (bd) st(&bmask[ab.y], mb | (1ull << c));
        }
        col[m] = c;
        ++won;
        cmax = c + 1u > cmax ? c + 1u : cmax;
    } else {
        const uint64_t t2 = ((uint64_t)(r + 2) << 48) | prio[m];
        atomicMax((unsigned long long*)&nxt[ab.x], (unsigned long long)t2);
        if (bd) atomicMax((unsigned long long*)&nxt[ab.y], (unsigned long long)t2);
    }
}

// The rounds for a short list: one workgroup, a workgroup barrier per round
// (every wave first waits for its own stores: they are agent-scope and must have
// landed before another wave loads them).  Runs when 0 < list length <= small.
__global__ void __launch_bounds__(1024) k_colour_small(Bodies B, const uint2* __restrict__ m_ab,
                                                       uint32_t* __restrict__ col, const uint64_t* __restrict__ prio,
                                                       uint64_t* bmax0, uint64_t* bmax1, uint64_t* bmask,
                                                       const uint32_t* __restrict__ list, Counters* cnt,
                                                       uint32_t max_rounds, uint32_t small) {
    // per-round totals in three slots: round r adds into slot r % 3 and reads it after
    // barrier r; thread 0 then clears slot (r + 2) % 3, which nobody touches before
    // round r + 2 (it starts after barrier r + 1, which thread 0 reaches after the clear)
    __shared__ uint32_t s_won[3], s_cmax[3];
    const uint32_t L = cnt->remaining;
    if (L == 0u || L > small) return;  // uniform
    if (threadIdx.x < 3u) {
        s_won[threadIdx.x] = 0u;
        s_cmax[threadIdx.x] = 0u;
    }
    __syncthreads();
    uint32_t left = L;
    for (uint32_t r = 0;; ++r) {
        const uint32_t q = r % 3u;
        const uint64_t* cur = (r & 1u) ? bmax1 : bmax0;
        uint64_t* nxt = (r & 1u) ? bmax0 : bmax1;
        uint32_t won = 0, cmax = 0;
        for (uint32_t i = threadIdx.x; i < L; i += blockDim.x)
            jp_visit<true>(B, m_ab, col, prio, cur, nxt, bmask, list[i], r, won, cmax);
        if (won) {
            atomicAdd(&s_won[q], won);
            atomicMax(&s_cmax[q], cmax);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const uint32_t w = s_won[q];
        if (threadIdx.x == 0) {
            if (w) {
                atomicMax(&cnt->max_colour, s_cmax[q]);
                atomicMax(&cnt->last_round, r + 1u);
            }
            s_won[(r + 2u) % 3u] = 0u;
            s_cmax[(r + 2u) % 3u] = 0u;
        }
        left -= w;
        if (left == 0u) break;
        if (r + 1 >= max_rounds) {
            if (threadIdx.x == 0) atomicOr(&cnt->sticky, STICKY_COLOURS);
            break;
        }
    }
    if (threadIdx.x == 0) cnt->remaining = 0u;
}

// The rounds for a long list (a full recolouring): persistent, one workgroup per
// CU, a grid barrier per round.  Runs when the list is longer than `small`.
__global__ void __launch_bounds__(256) k_colour(Bodies B, const uint2* __restrict__ m_ab, uint32_t* __restrict__ col,
                                                const uint64_t* __restrict__ prio, uint64_t* __restrict__ bmax0,
                                                uint64_t* __restrict__ bmax1, uint64_t* __restrict__ bmask,
                                                const uint32_t* __restrict__ list, GridBar* bar, Counters* cnt,
                                                uint32_t max_rounds, uint32_t small) {
    const uint32_t L = cnt->remaining;
    if (L <= small) return;  // uniform across the grid: no barrier is entered
    const uint32_t nb = gridDim.x;
    const uint32_t gs = nb * blockDim.x;
    const uint32_t g0 = blockIdx.x * blockDim.x + threadIdx.x;
    for (uint32_t r = 0;; ++r) {
        const uint64_t* cur = (r & 1u) ? bmax1 : bmax0;
        uint64_t* nxt = (r & 1u) ? bmax0 : bmax1;
        uint32_t won = 0, cmax = 0;
        for (uint32_t i = g0; i < L; i += gs) jp_visit<false>(B, m_ab, col, prio, cur, nxt, bmask, list[i], r, won, cmax);
        if (won) {
            atomicSub(&cnt->remaining, won);
            atomicMax(&cnt->max_colour, cmax);
            atomicMax(&cnt->last_round, r + 1u);
        }
        // the count left after round r, as it stood when every workgroup had finished round r
        const uint32_t left = grid_sync(bar, nb, cnt, &cnt->remaining);
        const uint32_t bad = __hip_atomic_load(&cnt->sticky, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (left == 0 || (bad & STICKY_TIMEOUT)) break;
        if (r + 1 >= max_rounds) {
            if (g0 == 0) atomicOr(&cnt->sticky, STICKY_COLOURS);
            break;
        }
    }
}

// Size classes of the islands of more than ISLAND_LANE_MAX manifolds (islands_part solves
// the largest first): 0 above 256 manifolds, 1 above 64, 2 above 32, 3 above 16, 4 the rest.
// Their work list entries (first slot, manifolds) lie in one region per class, each as long as
// the manifold capacity allows islands of its class.
__device__ __forceinline__ uint32_t isl_class(uint32_t n) {
    return n > 256u ? 0u : (n > 64u ? 1u : (n > 32u ? 2u : (n > 16u ? 3u : 4u)));
}
__device__ __forceinline__ uint32_t isl_region(uint32_t c, uint32_t cap) {
    uint32_t o = 0;
    if (c > 0u) o += cap / 257u;
    if (c > 1u) o += cap / 65u;
    if (c > 2u) o += cap / 33u;
    if (c > 3u) o += cap / 17u;
    return o;
}
// One pass over the sorted keys skey (thread gid of gsz, both whole waves; every lane of a
// wave takes part in each round): with off, the colour offsets off[c] = first position whose
// key has colour >= c (c = 0..K, a small island's key counting as colour K, since those
// keys sort above every colour) and m_glob = off[K]; with list, the work list of the small
// islands of more than ISLAND_LANE_MAX manifolds (the smaller ones are found by their slots).
// An island starts where its key differs from the one before it above the colour bits.
__device__ __forceinline__ void sorted_keys_part(const Bodies& B, const uint32_t* __restrict__ skey,
                                                 uint32_t* __restrict__ off, uint2* __restrict__ list, uint32_t cap,
                                                 Counters* cnt, uint32_t gid, uint32_t gsz) {
    const uint32_t M = min(cap, cnt->m_eff), K = cnt->max_colour, lane = gid & 63u;
    auto colour_of = [K](uint32_t k) { return (k & LOCAL_KEY) != 0u ? K : k; };
    for (uint32_t base = gid - lane; base <= M; base += gsz) {
        const uint32_t s = base + lane;
        bool start = false;
        uint32_t size = 0;
        if (s <= M) {
            const uint32_t k = s < M ? skey[s] : 0u, kp = s > 0u ? skey[s - 1u] : 0u;
            if (off) {
                // the colours from just above the previous key's to this key's (to K at the end)
                const uint32_t c0 = s > 0u ? colour_of(kp) + 1u : 0u, c1 = s < M ? colour_of(k) : K;
                for (uint32_t c = c0; c <= c1; ++c) {
                    off[c] = s;
                    if (c == K) cnt->m_glob = s;
                }
            }
            if (list && s < M) {
                start = (k & LOCAL_KEY) != 0u && (s == 0u || ((kp ^ k) >> 8) != 0u);
                if (start) size = B.icnt[(k & ~LOCAL_KEY) >> 8];
            }
        }
        if (list) {
            const bool big = start && size > ISLAND_LANE_MAX;
            if (__ballot(big) != 0ull) {
                // one atomic per class of the wave's islands
                const uint32_t cls = isl_class(size);
                for (uint32_t c = 0; c < ISLAND_CLASSES; ++c) {
                    const uint64_t in = __ballot(big && cls == c);
                    if (in == 0ull) continue;
                    uint32_t at = 0;
                    if (c == 0u && big && cls == 0u) {
                        atomicAdd(&cnt->isl_wide, (size + 31u) / 32u);
                        atomicMax(&cnt->isl_most, size);
                    }
                    if (lane == 0u) at = atomicAdd(&cnt->isl_n[c], (uint32_t)__popcll(in));
                    at = (uint32_t)__shfl((int)at, 0, 64);
                    if (big && cls == c)
                        list[isl_region(c, cap) + at + (uint32_t)__popcll(in & ((1ull << lane) - 1ull))] =
                            make_uint2(s, size);
                }
            }
        }
    }
}

__global__ void k_iota(uint32_t* __restrict__ p, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = i;
}


// ---------------------------------------------------------------- solver
struct SB {
    f3 v, w, x;
    float im;
    s3 I;
    bool dyn;
};

// A body's solver state for the row preparation.  The world inverse inertia is formed
// here, for the bodies of manifolds only (sv.w > 0 exactly when the body is dynamic and
// awake this step), rather than stored for every body at the step start.
__device__ __forceinline__ void load_sb(const Bodies& B, uint32_t i, SB& s, bool want_x) {
    const float4 v = B.sv[i], w = B.sw[i];
    s.v = xyz(v);
    s.im = v.w;
    s.w = xyz(w);
    s.dyn = v.w > 0.0f;
    s.I = s.dyn ? world_inv_inertia(quat_to_mat(B.q[i]), xyz(B.ii[i])) : s3{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (want_x) s.x = xyz(B.x[i]);
}
__device__ __forceinline__ void zero_sb(SB& s) {
    s.v = s.w = s.x = f3{0.0f, 0.0f, 0.0f};
    s.im = 0.0f;
    s.I = s3{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    s.dyn = false;
}

__device__ __forceinline__ void apply_imp(SB& A, SB& Bd, f3 rA, f3 rB, f3 P) {
    if (A.dyn) {
        A.v = A.v - P * A.im;
        A.w = A.w - smul(A.I, cross(rA, P));
    }
    if (Bd.dyn) {
        Bd.v = Bd.v + P * Bd.im;
        Bd.w = Bd.w + smul(Bd.I, cross(rB, P));
    }
}
__device__ __forceinline__ f3 vrel(const SB& A, const SB& Bd, f3 rA, f3 rB) {
    return (Bd.v + cross(Bd.w, rB)) - (A.v + cross(A.w, rA));
}

// Prepares solve slot s; returns the warm-start hits and the algorithmic bytes of one
// sweep visit of the slot (the kernel sums them per wave).
__device__ __forceinline__ void prep_slot(const Bodies& B, const StepParams& sp, const uint32_t* __restrict__ order,
                                          uint32_t cap, const uint2* __restrict__ m_ab,
                                          const uint32_t* __restrict__ m_np, const float4* __restrict__ c_pt,
                                          const float4* __restrict__ c_nf, const SolverRows& R, const PrevCache& pc,
                                          const float4* __restrict__ warm_in, const uint32_t* __restrict__ col,
                                          const uint64_t* __restrict__ bmask, const uint32_t* __restrict__ bdeg,
                                          Counters* __restrict__ cnt, float* __restrict__ feat, uint32_t s,
                                          uint32_t& hits_out, unsigned long long& bytes_out) {
    const uint32_t m = order[s];
    const uint2 ab = m_ab[m];
    const uint32_t np = m_np[m];
    const bool plane = (ab.y & PLANE_BIT) != 0;
    SB A, Bd;
    load_sb(B, ab.x, A, true);
    if (plane) zero_sb(Bd); else load_sb(B, ab.y, Bd, true);
    R.hdr[s] = make_uint4(ab.x, ab.y, np, m);
    {
        // dependency words for the persistent sweep: deg << 8 | rank per dynamic body
        const uint32_t c = col[m];
        R.colour[s] = c;
        uint2 dp = make_uint2(UNSET, UNSET);
        // (more than 64 colours: no dependency words; the sweep hands the step to per-colour launches)
        if (c < 64u && cnt->max_colour <= 64u) {
            // a body's colour mask must hold one bit per manifold of the body, or the
            // persistent sweep's visit counts could never be reached
            const unsigned long long below = (1ull << c) - 1ull;
            if (A.dyn) {
                const unsigned long long mk = bmask[ab.x];
                if ((uint32_t)__popcll(mk) != bdeg[ab.x]) atomicOr(&cnt->sticky, STICKY_INTERNAL);
                dp.x = ((uint32_t)__popcll(mk) << 8) | (uint32_t)__popcll(mk & below);
            }
            if (Bd.dyn) {
                const unsigned long long mk = bmask[ab.y];
                if ((uint32_t)__popcll(mk) != bdeg[ab.y]) atomicOr(&cnt->sticky, STICKY_INTERNAL);
                dp.y = ((uint32_t)__popcll(mk) << 8) | (uint32_t)__popcll(mk & below);
            }
            // who visits which body in which colour: the sweep's visits pass velocities on by it
            if (A.dyn) B.vslot[(size_t)ab.x * 64u + c] = s << 1;
            if (Bd.dyn) B.vslot[(size_t)ab.y * 64u + c] = (s << 1) | 1u;
        }
        R.dep[s] = dp;
    }
    uint32_t ps = 0;
    const bool have_prev = pc.valid && prev_find(pc, ((uint64_t)ab.x << 32) | ab.y, ps);
    // the pair's friction and restitution: mu = sqrt(mu_A mu_B) (mu_A when equal), e = max(e_A, e_B);
    // a plane has the world's values
    float mu, rest_e;
    {
        const float4 ma = B.mat[ab.x];
        const float mub = plane ? sp.friction : B.mat[ab.y].x, eb = plane ? sp.restitution : B.mat[ab.y].y;
        mu = ma.x == mub ? ma.x : sqrtf(ma.x * mub);
        rest_e = ma.y > eb ? ma.y : eb;
    }
    uint32_t hits = 0;
    for (uint32_t k = 0; k < np; ++k) {
        const float4 pt = c_pt[(size_t)m * 4 + k], nf = c_nf[(size_t)m * 4 + k];
        const f3 p = xyz(pt), n = xyz(nf);
        const float depth = pt.w;
        const uint32_t fid = fbits(nf.w);
        const f3 rA = p - A.x;
        const f3 rB = plane ? f3{0.0f, 0.0f, 0.0f} : p - Bd.x;
        f3 t1, t2;
        tangents(n, t1, t2);
        const f3 dirs[3] = {n, t1, t2};
        float kk[3];
        f3 ja[3], jb[3], jia[3], jib[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            ja[d] = cross(rA, dirs[d]);
            jb[d] = cross(rB, dirs[d]);
            jia[d] = smul(A.I, ja[d]);
            jib[d] = smul(Bd.I, jb[d]);
            kk[d] = (A.im + Bd.im + dot(ja[d], jia[d]) + dot(jb[d], jib[d])) * sp.soft1;
        }
        const float mN = kk[0] > 0.0f ? 1.0f / kk[0] : 0.0f;
        const float mT1 = kk[1] > 0.0f ? 1.0f / kk[1] : 0.0f;
        const float mT2 = kk[2] > 0.0f ? 1.0f / kk[2] : 0.0f;
        const f3 vr = vrel(A, Bd, rA, rB);
        const float vn0 = dot(vr, n);
        float bias = 0.0f;
        if (depth > sp.slop) {
            bias = sp.baumgarte * (depth - sp.slop) * sp.inv_dt;
            if (bias > sp.max_bias) bias = sp.max_bias;
        } else if (depth < 0.0f) {
            bias = depth * sp.inv_dt;
        }
        if (vn0 < -sp.rest_threshold) {
            const float rb = -rest_e * vn0;
            if (rb > bias) bias = rb;
        }
        const size_t o = (size_t)k * cap + s;
        float4* J = R.J + (size_t)k * JROWS * cap + s;
        J[0 * (size_t)cap] = f4(n, mN);
        J[1 * (size_t)cap] = f4(ja[0], kk[0]);
        J[2 * (size_t)cap] = f4(jb[0], 0.0f);
        J[3 * (size_t)cap] = f4(jia[0], bias);
        J[4 * (size_t)cap] = f4(jib[0], 0.0f);
        J[5 * (size_t)cap] = f4(t1, mT1);
        J[6 * (size_t)cap] = f4(ja[1], kk[1]);
        J[7 * (size_t)cap] = f4(jb[1], 0.0f);
        J[9 * (size_t)cap] = f4(jib[1], 0.0f);
        J[10 * (size_t)cap] = f4(t2, mT2);
        J[11 * (size_t)cap] = f4(ja[2], kk[2]);
        J[12 * (size_t)cap] = f4(jb[2], 0.0f);
        J[13 * (size_t)cap] = f4(jia[2], 0.0f);
        J[14 * (size_t)cap] = f4(jib[2], 0.0f);
        R.fid[o] = fid;
        // previous step's impulse of the same feature (the cached warm start)
        float4 Lp = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        bool hit = false;
        if (have_prev) {
            const uint32_t pnp = pc.np[ps];
            for (uint32_t j = 0; j < pnp; ++j) {
                const size_t po = (size_t)j * pc.cap + ps;
                if (pc.fid[po] == fid) {
                    Lp = pc.lam[po];
                    hit = true;
                    ++hits;
                    break;
                }
            }
        }
        {
            // friction bound of this step: mu x the previous normal impulse of the same feature,
            // or for a new point the impulse that stops its approach on its own
            const float est = mN * (bias - vn0);
            const float nb = hit ? Lp.x : est;
            J[8 * (size_t)cap] = f4(jia[1], mu * (nb > 0.0f ? nb : 0.0f));
        }
        // the given warm start, if any, else the cached one (chosen by value: a choice of
        // address would place Lp in scratch memory)
        float4 L = Lp;
        if (warm_in) {
            const float4 wv = warm_in[(size_t)m * 4 + k];
            L.x = wv.x;
            L.y = wv.y;
            L.z = wv.z;
        }
        L.w = 0.0f;
        R.lam[o] = L;
        R.lam0[o] = L;
        if (feat) {
            // warm-start network inputs, contact frame, impulses in units of u = mN g dt
            const float gdt = MLP_G_REF * sp.dt;
            const float inv_gdt = 1.0f / gdt;
            const float u = mN * gdt;
            const float inv_u = u > 0.0f ? 1.0f / u : 0.0f;
            float4* fr = (float4*)(feat + ((size_t)4 * s + k) * MLP_IN);
            fr[0] = make_float4(n.x, n.y, n.z, depth * 20.0f);
            fr[1] = make_float4(vn0 * inv_gdt, dot(vr, t1) * inv_gdt, dot(vr, t2) * inv_gdt, dot(rA, n));
            fr[2] = make_float4(dot(rA, t1), dot(rA, t2), dot(rB, n), dot(rB, t1));
            fr[3] = make_float4(dot(rB, t2), A.im * mN, Bd.im * mN, mT1 * kk[0]);
            fr[4] = make_float4(mT2 * kk[0], bias * inv_gdt, Lp.x * inv_u, Lp.y * inv_u);
            fr[5] = make_float4(Lp.z * inv_u, hit ? 1.0f : 0.0f, (float)np * 0.25f, plane ? 1.0f : 0.0f);
        }
    }
    hits_out = hits;
    // algorithmic bytes one sweep visit of this manifold moves: header 16; per
    // point 15 Jacobian rows (9 against a plane, whose b / ib rows are not read)
    // and lambda read + write; each body's solver velocities read (32) and, when
    // dynamic, written back (32); a plane has no body
    unsigned long long bytes = 16ull + (plane ? 9ull * 16ull + 32ull : 15ull * 16ull + 32ull) * np + 32ull +
                               (A.dyn ? 32ull : 0ull);
    if (!plane) bytes += 32ull + (Bd.dyn ? 32ull : 0ull);
    bytes_out = bytes;
}
__global__ void __launch_bounds__(256) k_prep(Bodies B, StepParams sp, const uint32_t* __restrict__ order,
                                              uint32_t cap, const uint2* __restrict__ m_ab,
                                              const uint32_t* __restrict__ m_np, const float4* __restrict__ c_pt,
                                              const float4* __restrict__ c_nf, SolverRows R, PrevCache pc,
                                              const float4* __restrict__ warm_in, const uint32_t* __restrict__ col,
                                              const uint64_t* __restrict__ bmask, const uint32_t* __restrict__ bdeg,
                                              Counters* __restrict__ cnt, float* __restrict__ feat, PrepExtra X) {
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x, gsz = gridDim.x * blockDim.x;
    for (uint32_t i = gid; i < X.zero_n; i += gsz) X.zero[i] = 0u;
    // more colours than the colour offsets hold fail the step (as a sticky error, which
    // this launch sets itself, so it reads the condition rather than the bit)
    const bool colours_ok = cnt->max_colour <= X.max_k;
    // a failed step must not touch the impulse buffers
    const bool ok = cnt->sticky == 0u && colours_ok;
    if (gid == 0 && !colours_ok) atomicOr(&cnt->sticky, STICKY_COLOURS);
    if (ok) {
        if (X.ckey) {
            const uint32_t m = cnt->cache_m[X.cset];
            for (uint32_t i = gid; i < m; i += gsz) X.ckey[X.cpos[i]] = EMPTY_KEY;
        }
        if (X.col_off || X.list) sorted_keys_part(B, X.skey, X.col_off, X.list, cap, cnt, gid, gsz);
    }
    uint32_t hits = 0;
    unsigned long long bytes = 0;
    const uint32_t M = ok ? cnt->m_eff : 0u;
    for (uint32_t s = gid; s < M; s += gsz) {
        uint32_t h = 0;
        unsigned long long b = 0;
        prep_slot(B, sp, order, cap, m_ab, m_np, c_pt, c_nf, R, pc, warm_in, col, bmask, bdeg, cnt, feat, s, h, b);
        hits += h;
        bytes += b;
    }
    spread_add(cnt, &SpreadRow::warm_hits, hits);
    spread_add(cnt, &SpreadRow::pgs_bytes, bytes);
}

// Memory policy of the sweep: plain accesses when every colour is its own
// launch; agent-coherent accesses (sc1, coherent across XCD L2s) in the
// persistent kernel, where bodies and impulses written by one workgroup are read
// by another inside the same launch.
template <bool COH> struct Mem {
    static AXM_D float4 ld(const float4* p) {
        if constexpr (COH) {
            const unsigned long long* q = reinterpret_cast<const unsigned long long*>(p);
            const unsigned long long lo = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned long long hi = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return make_float4(__uint_as_float((uint32_t)lo), __uint_as_float((uint32_t)(lo >> 32)),
                               __uint_as_float((uint32_t)hi), __uint_as_float((uint32_t)(hi >> 32)));
        } else {
            return *p;
        }
    }
    static AXM_D void st(float4* p, float4 v) {
        if constexpr (COH) {
            unsigned long long* q = reinterpret_cast<unsigned long long*>(p);
            const unsigned long long lo = (unsigned long long)__float_as_uint(v.x) |
                                          ((unsigned long long)__float_as_uint(v.y) << 32);
            const unsigned long long hi = (unsigned long long)__float_as_uint(v.z) |
                                          ((unsigned long long)__float_as_uint(v.w) << 32);
            __hip_atomic_store(q, lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(q + 1, hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            *p = v;
        }
    }
};

// Solver velocities of a body (the sweep needs no inertia: I a and I b are in the rows).
template <bool COH> __device__ __forceinline__ void load_vel(const Bodies& B, uint32_t i, SB& s) {
    const float4 v = Mem<COH>::ld(B.sv + i), w = Mem<COH>::ld(B.sw + i);
    s.v = xyz(v);
    s.im = v.w;
    s.w = xyz(w);
    s.dyn = v.w > 0.0f;
}

// One constraint direction of a contact point: d, a = rA x d, b = rB x d, ia = IA a, ib = IB b.
struct Dir {
    f3 d, a, b, ia, ib;
};
// dot product with fused multiply-adds: x.z y.z + (x.y y.y + x.x y.x)
__device__ __forceinline__ float fdot(f3 x, f3 y) { return fmaf(x.z, y.z, fmaf(x.y, y.y, x.x * y.x)); }
// relative velocity along the direction: d.(vB - vA) + b.wB - a.wA
__device__ __forceinline__ float jvel(const Dir& J, const SB& A, const SB& Bd) {
    const float r = fdot(J.d, Bd.v - A.v) + fdot(J.b, Bd.w);
    return r - fdot(J.a, A.w);
}
// impulse `lam` along the direction: A gets -lam, B +lam
__device__ __forceinline__ void japply(const Dir& J, float lam, SB& A, SB& Bd) {
    if (A.dyn) {
        const float sa = -(lam * A.im);
        A.v = f3{fmaf(sa, J.d.x, A.v.x), fmaf(sa, J.d.y, A.v.y), fmaf(sa, J.d.z, A.v.z)};
        A.w = f3{fmaf(-lam, J.ia.x, A.w.x), fmaf(-lam, J.ia.y, A.w.y), fmaf(-lam, J.ia.z, A.w.z)};
    }
    if (Bd.dyn) {
        const float sb = lam * Bd.im;
        Bd.v = f3{fmaf(sb, J.d.x, Bd.v.x), fmaf(sb, J.d.y, Bd.v.y), fmaf(sb, J.d.z, Bd.v.z)};
        Bd.w = f3{fmaf(lam, J.ib.x, Bd.w.x), fmaf(lam, J.ib.y, Bd.w.y), fmaf(lam, J.ib.z, Bd.w.z)};
    }
}
// japply without a branch per side, for visits whose lanes differ in which sides are
// dynamic.  A side that is not dynamic has zero inverse mass and zero inverse-inertia
// rows (its world inverse inertia is zero), so for a finite impulse its velocity changes
// at most in the sign of a zero component; callers never store such a side back.
__device__ __forceinline__ void japply_both(const Dir& J, float lam, SB& A, SB& Bd) {
    const float sa = -(lam * A.im);
    A.v = f3{fmaf(sa, J.d.x, A.v.x), fmaf(sa, J.d.y, A.v.y), fmaf(sa, J.d.z, A.v.z)};
    A.w = f3{fmaf(-lam, J.ia.x, A.w.x), fmaf(-lam, J.ia.y, A.w.y), fmaf(-lam, J.ia.z, A.w.z)};
    const float sb = lam * Bd.im;
    Bd.v = f3{fmaf(sb, J.d.x, Bd.v.x), fmaf(sb, J.d.y, Bd.v.y), fmaf(sb, J.d.z, Bd.v.z)};
    Bd.w = f3{fmaf(lam, J.ib.x, Bd.w.x), fmaf(lam, J.ib.y, Bd.w.y), fmaf(lam, J.ib.z, Bd.w.z)};
}
// Direction `dir` (0 n, 1 t1, 2 t2) of the point whose rows start at J, consecutive
// rows `rs` float4 apart; the .w of the first row is returned in w0.  Against a plane
// b and ib are zero and not read.
__device__ __forceinline__ Dir load_dir(const float4* J, size_t rs, int dir, bool plane, float& w0, float& w1,
                                        float& w2, float& w3, float& w4) {
    const float4* q = J + (size_t)(5 * dir) * rs;
    const float4 r0 = q[0], r1 = q[rs], r3 = q[3 * rs];
    Dir D;
    D.d = xyz(r0);
    D.a = xyz(r1);
    D.ia = xyz(r3);
    w0 = r0.w;
    w1 = r1.w;
    w3 = r3.w;
    if (plane) {
        D.b = D.ib = f3{0.0f, 0.0f, 0.0f};
        w2 = w4 = 0.0f;
    } else {
        const float4 r2 = q[2 * rs], r4 = q[4 * rs];
        D.b = xyz(r2);
        D.ib = xyz(r4);
        w2 = r2.w;
        w4 = r4.w;
    }
    return D;
}

// The projections of a visit, one instruction each: x clamped to [-m, m]
// (m >= 0) and x clamped below at zero.  For finite x they give the values of
// x < -m ? -m : (x > m ? m : x) and x > 0 ? x : 0, except that a zero may come out with the
// other sign; every later use of the impulse is a sum, product or comparison, so no later
// value differs.
__device__ __forceinline__ float clamp_sym(float x, float m) { return __builtin_amdgcn_fmed3f(x, -m, m); }
// One visit of a manifold on registers: warm start (first sweep only), friction
// rows of every point, then normal rows.  Point k's rows start at J + k * ps, rows
// `rs` apart; L[k] holds the point impulses in and out.
__device__ __forceinline__ void solve_rows(const float4* J, size_t rs, size_t ps, uint32_t np, bool plane, float keep,
                                           bool first, SB& A, SB& Bd, float4 L[4]) {
    float w0, w1, w2, w3, w4;
    if (first) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            if (k >= np) break;
            const float4* P = J + (size_t)k * ps;
            const Dir Dn = load_dir(P, rs, 0, plane, w0, w1, w2, w3, w4);
            const Dir D1 = load_dir(P, rs, 1, plane, w0, w1, w2, w3, w4);
            const Dir D2 = load_dir(P, rs, 2, plane, w0, w1, w2, w3, w4);
            japply_both(Dn, L[k].x, A, Bd);
            japply_both(D1, L[k].y, A, Bd);
            japply_both(D2, L[k].z, A, Bd);
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        if (k >= np) break;
        const float4* P = J + (size_t)k * ps;
        float maxf;  // the step's friction bound (row 8's .w)
        {
            float mT1;
            const Dir D1 = load_dir(P, rs, 1, plane, mT1, w1, w2, maxf, w4);
            float nl = fmaf(-mT1, jvel(D1, A, Bd), keep * L[k].y);
            nl = clamp_sym(nl, maxf);
            const float d = nl - L[k].y;
            L[k].y = nl;
            japply_both(D1, d, A, Bd);
        }
        {
            float mT2;
            const Dir D2 = load_dir(P, rs, 2, plane, mT2, w1, w2, w3, w4);
            float nl = fmaf(-mT2, jvel(D2, A, Bd), keep * L[k].z);
            nl = clamp_sym(nl, maxf);
            const float d = nl - L[k].z;
            L[k].z = nl;
            japply_both(D2, d, A, Bd);
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        if (k >= np) break;
        const float4* P = J + (size_t)k * ps;
        float mN, x1, x2, tg, x4;
        const Dir Dn = load_dir(P, rs, 0, plane, mN, x1, x2, tg, x4);
        float nl = fmaf(mN, tg - jvel(Dn, A, Bd), keep * L[k].x);
        nl = fmaxf(nl, 0.0f);
        const float d = nl - L[k].x;
        L[k].x = nl;
        japply_both(Dn, d, A, Bd);
    }
}
// The same with every row of the visit already in registers (Jr[k][r]: row r of
// point k), so that a visit whose rows are not staged waits for one batch of loads
// instead of one per row group.  Same arithmetic, same results.  The b-side rows of a
// plane contact hold zeros (load_rows), the values the row loads above substitute, so
// no lane selects between the two.
__device__ __forceinline__ Dir dir_regs(const float4 (&Jr)[JROWS], int dir, float& w0, float& w3) {
    const float4 r0 = Jr[5 * dir], r1 = Jr[5 * dir + 1], r3 = Jr[5 * dir + 3];
    Dir D;
    D.d = xyz(r0);
    D.a = xyz(r1);
    D.ia = xyz(r3);
    w0 = r0.w;
    w3 = r3.w;
    D.b = xyz(Jr[5 * dir + 2]);
    D.ib = xyz(Jr[5 * dir + 4]);
    return D;
}
__device__ __forceinline__ void load_rows(const SolverRows& R, uint32_t s, uint32_t cap, uint32_t np, bool plane,
                                          float4 (&Jr)[4][JROWS]) {
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        if (k >= np) break;
        const float4* src = R.J + (size_t)k * JROWS * cap + s;
#pragma unroll
        for (uint32_t r = 0; r < JROWS; ++r) {
            const bool bside = (r % 5u) == 2u || (r % 5u) == 4u;  // b and IB b: not read against a plane
            Jr[k][r] = (bside && plane) ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : src[(size_t)r * cap];
        }
    }
}
__device__ __forceinline__ void solve_regs(const float4 (&Jr)[4][JROWS], uint32_t np, float keep,
                                           bool first, SB& A, SB& Bd, float4 L[4]) {
    float w0, w3;
    if (first) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            if (k >= np) break;
            const Dir Dn = dir_regs(Jr[k], 0, w0, w3);
            const Dir D1 = dir_regs(Jr[k], 1, w0, w3);
            const Dir D2 = dir_regs(Jr[k], 2, w0, w3);
            japply_both(Dn, L[k].x, A, Bd);
            japply_both(D1, L[k].y, A, Bd);
            japply_both(D2, L[k].z, A, Bd);
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        if (k >= np) break;
        float maxf;  // the step's friction bound (row 8's .w)
        {
            float mT1;
            const Dir D1 = dir_regs(Jr[k], 1, mT1, maxf);
            float nl = fmaf(-mT1, jvel(D1, A, Bd), keep * L[k].y);
            nl = clamp_sym(nl, maxf);
            const float d = nl - L[k].y;
            L[k].y = nl;
            japply_both(D1, d, A, Bd);
        }
        {
            float mT2;
            const Dir D2 = dir_regs(Jr[k], 2, mT2, w3);
            float nl = fmaf(-mT2, jvel(D2, A, Bd), keep * L[k].z);
            nl = clamp_sym(nl, maxf);
            const float d = nl - L[k].z;
            L[k].z = nl;
            japply_both(D2, d, A, Bd);
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        if (k >= np) break;
        float mN, tg;
        const Dir Dn = dir_regs(Jr[k], 0, mN, tg);
        float nl = fmaf(mN, tg - jvel(Dn, A, Bd), keep * L[k].x);
        nl = fmaxf(nl, 0.0f);
        const float d = nl - L[k].x;
        L[k].x = nl;
        japply_both(Dn, d, A, Bd);
    }
}
// The same with the rows of solve slot s in the SoA row arrays (row r of point k at
// J[(k * JROWS + r) * cap + s]).
__device__ __forceinline__ void solve_core(const SolverRows& R, uint32_t s, uint32_t cap, uint32_t np, bool plane,
                                           float keep, bool first, SB& A, SB& Bd, float4 L[4]) {
    solve_rows(R.J + s, cap, (size_t)JROWS * cap, np, plane, keep, first, A, Bd, L);
}

// One visit of the manifold in solve slot s with plain loads and stores (one
// launch per colour: every visit of a launch touches distinct bodies).
__device__ __forceinline__ void solve_slot(const Bodies& B, const StepParams& sp, const SolverRows& R, uint4 h,
                                           uint32_t s, uint32_t cap, bool first) {
    const uint32_t a = h.x, b = h.y, np = h.z;
    const bool plane = (b & PLANE_BIT) != 0;
    SB A, Bd;
    load_vel<false>(B, a, A);
    if (plane) zero_sb(Bd); else load_vel<false>(B, b, Bd);
    float4 L[4];
    // over a fixed 4 so that L stays in registers
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
        if (k < np) L[k] = R.lam[(size_t)k * cap + s];
    solve_core(R, s, cap, np, plane, sp.keep, first, A, Bd, L);
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
        if (k < np) R.lam[(size_t)k * cap + s] = make_float4(L[k].x, L[k].y, L[k].z, 0.0f);
    if (A.dyn) {
        B.sv[a] = f4(A.v, A.im);
        B.sw[a] = f4(A.w, 0.0f);
    }
    if (Bd.dyn) {
        B.sv[b] = f4(Bd.v, Bd.im);
        B.sw[b] = f4(Bd.w, 0.0f);
    }
}

__global__ void __launch_bounds__(256) k_pgs(Bodies B, StepParams sp, SolverRows R, uint32_t s0, uint32_t s1,
                                             uint32_t cap, uint32_t first) {
    const uint32_t s = s0 + blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= s1) return;
    solve_slot(B, sp, R, R.hdr[s], s, cap, first != 0);
}

// Persistent sweep kernel.  An item is the visit of one manifold slot in one
// sweep.  It may run once every earlier visit of its dynamic bodies is complete:
// the visit of slot s in sweep k is visit number k * deg(x) + rank(x, s) of body
// x, with rank = colours of x's manifolds below s's colour (the per-body colour
// masks of the colouring), so each body sees exactly the update sequence of the
// colour-by-colour sweep without a grid-wide barrier.
//
// Ownership: the slots are cut into chunks of 64; workgroup g (one wave) owns
// chunks g, g + G, g + 2G, ... and lane l of it slot 64 * chunk + l, in every
// sweep.  A lane walks its own items in increasing (sweep, slot) order on its
// own, so the smallest unfinished item of the launch always has its
// dependencies complete and the walk cannot deadlock while all G waves are
// resident (the host sizes G from the occupancy of the kernel).  Because a lane
// is the only one to visit its slots, the Jacobian rows and the impulses of its
// points are staged once per launch into LDS (up to `ppl` points per lane, the
// rest is read from and written to the row arrays) and never go back to memory
// between sweeps; only body velocities move between waves.
//
// Inboxes: during the launch a body's solver velocity travels from one visit of
// the body to the next.  Each slot has an inbox of 8 64-bit words (64 bytes) holding,
// for the slot's next visit, body a's velocity (v, w: 192 bits) in words 0..3 and
// body b's in words 4..7, each word 48 value bits under a 16-bit version: the body's
// visits completed, modulo 2^16.  An inbox only ever holds the version before the
// one its reader waits for (deg visits earlier, deg <= 64) or that one, so 16 bits
// never alias.  A visit waits until its inbox words carry the visit numbers it needs
// (a 64-bit word is single-copy atomic, so matching versions mean matching values),
// solves, and writes each dynamic body's new velocity into the inbox of that body's
// next visit (the manifold of the next colour in the body's colour mask, or its first
// one for the next sweep) with plain stores (two 16-byte ones where the inboxes lie
// within 2 GiB).  The last word of each side (3 for a, 7 for b, in the last store a
// writer makes) is a hint: a poll reads the two hints and loads the rest once both are
// in; the full load checks every version itself.
// A bounded wait sets STICKY_TIMEOUT instead of hanging.
constexpr uint32_t IB_WORDS = INBOX_WORDS;  // inbox words per slot
constexpr uint32_t IB_SIDE = 4;     // words per body
constexpr uint32_t IB_HINT = 3;     // word 3 of each side (polled first), stored with word 2
constexpr uint32_t OWN_WAVE = 64;   // threads per workgroup of the sweep kernel
// residual check word: workgroups arrived in the low 16 bits, workgroups above the tolerance above them
constexpr uint32_t CHECK_ABOVE = 1u << 16;
constexpr uint32_t NO_VISIT = 0xFFFFFFFFu;  // version no visit count reaches

// A velocity (v, w) as four inbox words under version ver (low 16 bits): the six
// floats' 192 bits in 48-bit pieces, x0 | x1[0:16], x1[16:32] | x2, x3 | x4[0:16],
// x4[16:32] | x5.
__device__ __forceinline__ void vpack4(f3 v, f3 w, uint32_t ver, uint64_t (&o)[4]) {
    const uint64_t V = (uint64_t)(ver & 0xFFFFu) << 48;
    const uint32_t x0 = __float_as_uint(v.x), x1 = __float_as_uint(v.y), x2 = __float_as_uint(v.z);
    const uint32_t x3 = __float_as_uint(w.x), x4 = __float_as_uint(w.y), x5 = __float_as_uint(w.z);
    o[0] = V | ((uint64_t)(x1 & 0xFFFFu) << 32) | x0;
    o[1] = V | ((uint64_t)x2 << 16) | (x1 >> 16);
    o[2] = V | ((uint64_t)(x4 & 0xFFFFu) << 32) | x3;
    o[3] = V | ((uint64_t)x5 << 16) | (x4 >> 16);
}
// The same words as (low, high) dword pairs: the version of a word is high >> 16.
__device__ __forceinline__ uint32_t vver2(uint2 x) { return x.y >> 16; }
__device__ __forceinline__ void vunpack4(uint2 a, uint2 b, uint2 c, uint2 d, f3& v, f3& w) {
    v = f3{__uint_as_float(a.x), __uint_as_float((a.y & 0xFFFFu) | (b.x << 16)),
           __uint_as_float((b.x >> 16) | (b.y << 16))};
    w = f3{__uint_as_float(c.x), __uint_as_float((c.y & 0xFFFFu) | (d.x << 16)),
           __uint_as_float((d.x >> 16) | (d.y << 16))};
}
__device__ __forceinline__ uint2 vsplit(uint64_t x) { return make_uint2((uint32_t)x, (uint32_t)(x >> 32)); }
__device__ __forceinline__ uint64_t vload(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void vstore(uint64_t* p, uint64_t w) {
    __hip_atomic_store(p, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Word k (0..3) of side `side` of the inbox of slot s.
__device__ __forceinline__ size_t vin_word(uint32_t s, uint32_t side, uint32_t k) {
    return (size_t)s * IB_WORDS + side * IB_SIDE + k;
}
// Writes a velocity into side `side` of slot s's inbox, the hint word last.  With
// `wide` (inboxes within 2 GiB) words 0-1 and 2-3 go out as one 16-byte store each,
// with the cache policy of a device-scope store: two writes instead of four.  Every
// word carries its own version, so a reader that sees one half of a pair before the
// other only waits.
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void vin_store(uint64_t* inbox, uint32_t s, uint32_t side, uint32_t ver, f3 v, f3 w,
                                          bool wide) {
    uint64_t o[4];
    vpack4(v, w, ver, o);
    if (wide) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(inbox, 0, 0x7FFFFFFF, 0x00020000);
        const uint32_t base = s * (IB_WORDS * 8u) + side * (IB_SIDE * 8u);  // byte offset of word 0 of this side
        const u32x4_t q0 = {(uint32_t)o[0], (uint32_t)(o[0] >> 32), (uint32_t)o[1], (uint32_t)(o[1] >> 32)};
        const u32x4_t q1 = {(uint32_t)o[2], (uint32_t)(o[2] >> 32), (uint32_t)o[3], (uint32_t)(o[3] >> 32)};
        // aux: sc1, as the device-scope atomic store below
        __builtin_amdgcn_raw_buffer_store_b128(q0, rs, (int)base, 0, 16);
        __builtin_amdgcn_raw_buffer_store_b128(q1, rs, (int)(base + 16u), 0, 16);
        return;
    }
#pragma unroll
    for (uint32_t k = 0; k < IB_SIDE; ++k) vstore(inbox + vin_word(s, side, k), o[k]);
}
// Words k and k + 1 of slot s's inbox in one coherent 16-byte access, as (value,
// version) dword pairs; every word is checked against its own version, so a load
// that sees one word before the other only delays the visit.  Inboxes within 2 GiB.
__device__ __forceinline__ uint4 vin_quad(const uint64_t* inbox, uint32_t s, uint32_t k) {
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint64_t*>(inbox), 0, 0x7FFFFFFF, 0x00020000);
    // aux: sc0 | sc1, the cache policy of a system-coherent load (bypasses the non-coherent caches)
    const auto r = __builtin_amdgcn_raw_buffer_load_b128(rs, s * (IB_WORDS * 8u) + k * 8u, 0, 1 | 16);
    return make_uint4(r[0], r[1], r[2], r[3]);
}
// The visit after the one of colour c of a body with colour mask mk: the next
// colour up, or the body's first colour (next sweep).
__device__ __forceinline__ uint32_t next_colour(unsigned long long mk, uint32_t c) {
    const unsigned long long above = c >= 63u ? 0ull : mk & ~((2ull << c) - 1ull);
    return (uint32_t)__ffsll(above ? above : mk) - 1u;
}

// Before a launch, per slot of [s0, s1): the next visit of each dynamic body, and the inbox
// words: a body's first visit (rank 0) gets the body's solver velocity with version 0, every
// other inbox a version no visit waits for.  The rows exist only when this step's preparation
// ran.  (Thread gid of gsz.)
__device__ __forceinline__ void flow_init_part(const Bodies& B, const SolverRows& R, const uint64_t* __restrict__ bmask,
                                               uint32_t s0, uint32_t s1, uint32_t gid, uint32_t gsz) {
    for (uint32_t s = s0 + gid; s < s1; s += gsz) {
    const uint4 h = R.hdr[s];
    const uint2 dp = R.dep[s];
    const uint32_t c = R.colour[s];
    uint2 nx = make_uint2(UNSET, UNSET);
    f3 va = {0.0f, 0.0f, 0.0f}, wa = va, vb = va, wb = va;
    uint32_t ra = NO_VISIT, rb = NO_VISIT;
    if (dp.x != UNSET) {
        nx.x = B.vslot[(size_t)h.x * 64u + next_colour(bmask[h.x], c)];
        if ((dp.x & 0xFFu) == 0u) ra = 0u;
        va = xyz(B.sv[h.x]);
        wa = xyz(B.sw[h.x]);
    }
    if (dp.y != UNSET) {
        nx.y = B.vslot[(size_t)h.y * 64u + next_colour(bmask[h.y], c)];
        if ((dp.y & 0xFFu) == 0u) rb = 0u;
        vb = xyz(B.sv[h.y]);
        wb = xyz(B.sw[h.y]);
    }
    R.next[s] = nx;
    // the whole inbox (words 0-3 and 4-7 as laid out by vin_word) in four 16-byte
    // stores; the sweep kernel, a later launch, sees them after the launch boundary
    uint64_t oa[4], ob[4];
    vpack4(va, wa, ra, oa);
    vpack4(vb, wb, rb, ob);
    uint4* q = reinterpret_cast<uint4*>(R.inbox + (size_t)s * IB_WORDS);
    q[0] = make_uint4((uint32_t)oa[0], (uint32_t)(oa[0] >> 32), (uint32_t)oa[1], (uint32_t)(oa[1] >> 32));
    q[1] = make_uint4((uint32_t)oa[2], (uint32_t)(oa[2] >> 32), (uint32_t)oa[3], (uint32_t)(oa[3] >> 32));
    q[2] = make_uint4((uint32_t)ob[0], (uint32_t)(ob[0] >> 32), (uint32_t)ob[1], (uint32_t)(ob[1] >> 32));
    q[3] = make_uint4((uint32_t)ob[2], (uint32_t)(ob[2] >> 32), (uint32_t)ob[3], (uint32_t)(ob[3] >> 32));
    }
}
// The large islands' slots and, when the register sweep takes them, those of the islands of the
// largest class, whose arrival words start from zero.  G: the workgroups of the solve launch.
__global__ void __launch_bounds__(256) k_flow_init(Bodies B, SolverRows R, const uint64_t* __restrict__ bmask,
                                                   const Counters* __restrict__ cnt, const uint2* __restrict__ list,
                                                   unsigned long long* __restrict__ isl_arrive, uint32_t G) {
    if (cnt->sticky != 0u) return;
    flow_init_part(B, R, bmask, 0u, cnt->m_glob, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
    if (!list || wide_pieces(cnt, G) == 0u) return;
    for (uint32_t i = blockIdx.x; i < cnt->isl_n[0]; i += gridDim.x) {
        flow_init_part(B, R, bmask, list[i].x, list[i].x + list[i].y, threadIdx.x, blockDim.x);
        if (threadIdx.x < 2u) isl_arrive[(size_t)i * ISL_ARRIVE_WORDS + threadIdx.x * (ISL_ARRIVE_WORDS / 2u)] = 0ull;
    }
}
// Residual of one contact point: the largest velocity-space change (impulse change
// times the row's effective mass inverse) that one more visit would make along the
// normal or either friction direction, from the current velocities and impulses L.
// J points at the point's first Jacobian row, rs is the row stride.
__device__ __forceinline__ float point_residual(const float4* J, size_t rs, bool plane, float keep, const SB& A,
                                                const SB& Bd, const float4 L) {
    float mN, kN, tg, mT1, kT1, mT2, kT2, x2, x3, x4;
    const Dir Dn = load_dir(J, rs, 0, plane, mN, kN, x2, tg, x4);
    float maxf;  // the step's friction bound (row 8's .w)
    const Dir D1 = load_dir(J, rs, 1, plane, mT1, kT1, x2, maxf, x4);
    const Dir D2 = load_dir(J, rs, 2, plane, mT2, kT2, x2, x3, x4);
    float nl = fmaf(mN, tg - jvel(Dn, A, Bd), keep * L.x);
    nl = fmaxf(nl, 0.0f);
    float e = fabsf(nl - L.x) * kN;
    float q1 = fmaf(-mT1, jvel(D1, A, Bd), keep * L.y);
    q1 = clamp_sym(q1, maxf);
    const float e1 = fabsf(q1 - L.y) * kT1;
    float q2 = fmaf(-mT2, jvel(D2, A, Bd), keep * L.z);
    q2 = clamp_sym(q2, maxf);
    const float e2 = fabsf(q2 - L.z) * kT2;
    if (e1 > e) e = e1;
    if (e2 > e) e = e2;
    return e;
}

// The same with the point's rows in registers (as solve_regs).
__device__ __forceinline__ float point_residual_regs(const float4 (&Jr)[JROWS], float keep, const SB& A,
                                                     const SB& Bd, const float4 L) {
    float mN, tg, mT1, maxf, mT2, x3;
    const Dir Dn = dir_regs(Jr, 0, mN, tg);
    const Dir D1 = dir_regs(Jr, 1, mT1, maxf);
    const Dir D2 = dir_regs(Jr, 2, mT2, x3);
    const float kN = Jr[1].w, kT1 = Jr[6].w, kT2 = Jr[11].w;
    float nl = fmaf(mN, tg - jvel(Dn, A, Bd), keep * L.x);
    nl = fmaxf(nl, 0.0f);
    float e = fabsf(nl - L.x) * kN;
    float q1 = fmaf(-mT1, jvel(D1, A, Bd), keep * L.y);
    q1 = clamp_sym(q1, maxf);
    const float e1 = fabsf(q1 - L.y) * kT1;
    float q2 = fmaf(-mT2, jvel(D2, A, Bd), keep * L.z);
    q2 = clamp_sym(q2, maxf);
    const float e2 = fabsf(q2 - L.z) * kT2;
    if (e1 > e) e = e1;
    if (e2 > e) e = e2;
    return e;
}

// What a visit needs of its slot besides the rows: the slot, body indices and point count,
// dependency words, the next visits of its bodies, inverse masses and the
// velocity of a static partner (constant during the sweep).
struct Item {
    uint32_t s;  // the slot
    uint4 h;
    uint2 dp, nx;
    float imA, imB;
    f3 sv, sw;  // static partner's velocity (at most one side of a manifold is static)
};
__device__ __forceinline__ Item item_global(const Bodies& B, const SolverRows& R, uint32_t s) {
    Item it;
    it.s = s;
    it.h = R.hdr[s];
    it.dp = R.dep[s];
    it.nx = R.next[s];
    const bool plane = (it.h.y & PLANE_BIT) != 0u;
    const float4 va = B.sv[it.h.x];
    const float4 vb = plane ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : B.sv[it.h.y];
    it.imA = va.w;
    it.imB = vb.w;
    const uint32_t st = it.dp.x == UNSET ? it.h.x : it.h.y;  // the static side, if any
    const bool has_static = it.dp.x == UNSET || (!plane && it.dp.y == UNSET);
    it.sv = has_static ? xyz(it.dp.x == UNSET ? va : vb) : f3{0.0f, 0.0f, 0.0f};
    it.sw = has_static ? xyz(B.sw[st]) : f3{0.0f, 0.0f, 0.0f};
    return it;
}
// staged slot record: 4 float4 at rec[r * 64], r = 0..3
__device__ __forceinline__ void item_put(float4* rec, const Item& it) {
    rec[0] = make_float4(__uint_as_float(it.h.x), __uint_as_float(it.h.y), __uint_as_float(it.h.z),
                         __uint_as_float(it.s));
    rec[OWN_WAVE] = make_float4(__uint_as_float(it.dp.x), __uint_as_float(it.dp.y), __uint_as_float(it.nx.x),
                                __uint_as_float(it.nx.y));
    rec[2 * OWN_WAVE] = make_float4(it.imA, it.imB, it.sv.x, it.sv.y);
    rec[3 * OWN_WAVE] = make_float4(it.sv.z, it.sw.x, it.sw.y, it.sw.z);
}
__device__ __forceinline__ Item item_get(const float4* rec) {
    const float4 r0 = rec[0], r1 = rec[OWN_WAVE], r2 = rec[2 * OWN_WAVE], r3 = rec[3 * OWN_WAVE];
    Item it;
    it.h = make_uint4(__float_as_uint(r0.x), __float_as_uint(r0.y), __float_as_uint(r0.z), 0u);
    it.s = __float_as_uint(r0.w);
    it.dp = make_uint2(__float_as_uint(r1.x), __float_as_uint(r1.y));
    it.nx = make_uint2(__float_as_uint(r1.z), __float_as_uint(r1.w));
    it.imA = r2.x;
    it.imB = r2.y;
    it.sv = f3{r2.z, r2.w, r3.x};
    it.sw = f3{r3.y, r3.z, r3.w};
    return it;
}

constexpr uint32_t OWN_SLOTS = 16;  // slots per lane with a staged record

// LDS of a wave: records of its first min(owned chunks, OWN_SLOTS) slots per lane
// (as many as fit; record j of a lane at lds[(j * 4 + r) * 64 + lane]), then the
// staged points of the slots chosen for staging, packed in slot order: point q of a
// lane keeps row r at lds[P0 + (r * ppl + q) * 64 + lane] (rows 0..JROWS-1 the
// Jacobian rows of R.J[(k * JROWS + r) * cap + s], row JROWS its impulses).  Slots
// and points not staged are read from the row arrays.  With stop.bits, the sweeps
// run in chunks of stop.every with a residual check after each chunk (every wave of
// the grid meets at one arrival count per check).
__global__ void __launch_bounds__(OWN_WAVE) k_pgs_own(Bodies B, StepParams sp, SolverRows R, Counters* cnt,
                                                      uint32_t cap, uint32_t nsweeps, uint32_t flow_max,
                                                      uint32_t lds_f4, uint32_t spin_limit, uint32_t tune,
                                                      const uint64_t* __restrict__ bmask, SweepStop stop) {
    extern __shared__ float4 own_lds[];
    const uint32_t lane = threadIdx.x;
    const uint32_t M = cnt->m_glob;  // the large islands' slots (the small ones are solved on their own)
    if (cnt->max_colour > 64u) {
        // dependency ranks come from 64-bit colour masks: hand the step back for per-colour launches
        if (blockIdx.x == 0 && lane == 0) atomicOr(&cnt->sticky, STICKY_FLOW_COLOURS);
        return;
    }
    if (cnt->sticky != 0u || nsweeps == 0u) return;
    if (M > 0u && M <= flow_max) return;  // flow_part ran them
    if (M == 0u && cnt->m_eff > 0u) {
        // every island was solved on its own: no sweep of the large ones runs
        if (blockIdx.x == 0 && lane == 0 && stop.bits) {
            __hip_atomic_store(&cnt->sweeps_run, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&cnt->tol_hit, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return;
    }
    uint32_t* err = &cnt->sticky;
    const uint32_t G = gridDim.x, g = blockIdx.x;
    const uint32_t nchunks = (M + OWN_WAVE - 1) / OWN_WAVE;
    const uint32_t own = g < nchunks ? (nchunks - 1 - g) / G + 1 : 0u;
    // owned slots of this lane: j < nv (only the last owned chunk can be partial)
    const uint32_t nv = own == 0u ? 0u : own - (((g + (own - 1) * G) * OWN_WAVE + lane) >= M ? 1u : 0u);
    // slot records that fit the LDS (the rest are read from the row arrays)
    const uint32_t nrec = min(min(own, OWN_SLOTS), lds_f4 / (4u * OWN_WAVE));
    const uint32_t p0 = nrec * 4u * OWN_WAVE;
    const uint32_t ppl = lds_f4 > p0 ? (lds_f4 - p0) / ((JROWS + 1u) * OWN_WAVE) : 0u;
    const size_t rs = (size_t)ppl * OWN_WAVE;  // LDS row stride of the points (float4)
    float4* recs = own_lds + lane;
    float4* mine = own_lds + p0 + lane;
    auto slot_of = [&](uint32_t jj) { return (g + jj * G) * OWN_WAVE + lane; };

    // stage slot records (only owned slots below M exist: j < nv)
    const uint32_t nr = min(nrec, nv);
    for (uint32_t j = 0; j < nr; ++j) item_put(recs + (size_t)j * 4u * OWN_WAVE, item_global(B, R, slot_of(j)));
    // Which owned slots get their rows and impulses staged (bit j of smask): as many
    // as fit, among the slots with a staged record those on the longest dependency
    // chains first (the larger visit count per sweep of their two bodies), then the
    // other slots in order.  Only a lane's first 64 slots can be staged.
    uint64_t smask = 0;
    {
        auto rec_np_crit = [&](uint32_t j, uint32_t& np, uint32_t& crit) {
            const float4 r0 = recs[(size_t)j * 4u * OWN_WAVE], r1 = recs[(size_t)(j * 4u + 1u) * OWN_WAVE];
            const uint32_t dx = __float_as_uint(r1.x), dy = __float_as_uint(r1.y);
            np = min(__float_as_uint(r0.z), 4u);
            crit = max(dx == UNSET ? 0u : dx >> 8, dy == UNSET ? 0u : dy >> 8);
        };
        uint32_t used = 0, level = 0xFFFFFFFFu;
        for (;;) {  // criticality levels, descending
            uint32_t next = 0;
            bool any = false;
            for (uint32_t j = 0; j < nr; ++j) {
                uint32_t np, c;
                rec_np_crit(j, np, c);
                if (c < level && (!any || c > next)) {
                    next = c;
                    any = true;
                }
            }
            if (!any) break;
            for (uint32_t j = 0; j < nr; ++j) {
                uint32_t np, c;
                rec_np_crit(j, np, c);
                if (c == next && used + np <= ppl) {
                    smask |= 1ull << j;
                    used += np;
                }
            }
            level = next;
        }
        for (uint32_t j = nr; j < min(nv, 64u); ++j) {
            const uint32_t np = min(R.hdr[slot_of(j)].z, 4u);
            if (used + np <= ppl) {
                smask |= 1ull << j;
                used += np;
            }
        }
    }
    auto staged_slot = [&](uint32_t j) { return j < 64u && ((smask >> j) & 1ull) != 0ull; };
    const bool all_staged = nv <= nrec && smask == (1ull << nv) - 1ull;  // nrec <= 16
    // stage the selected slots' rows and impulses, packed in slot order
    {
        uint32_t off = 0;
        for (uint32_t j = 0; j < nv; ++j) {
            if (!staged_slot(j)) continue;
            const uint32_t s = slot_of(j);
            const uint32_t np = min(j < nrec ? __float_as_uint(recs[(size_t)j * 4u * OWN_WAVE].z) : R.hdr[s].z, 4u);
            for (uint32_t k = 0; k < np; ++k) {
                const float4* src = R.J + (size_t)k * JROWS * cap + s;
                float4* dst = mine + (size_t)(off + k) * OWN_WAVE;
#pragma unroll
                for (uint32_t r = 0; r < JROWS; ++r) dst[r * rs] = src[(size_t)r * cap];
                dst[JROWS * rs] = R.lam[(size_t)k * cap + s];
            }
            off += np;
        }
    }
    // The visits of a wave whose slots and points are all in LDS read nothing but
    // the inbox words from memory; the general loop reads what is not staged from
    // the row arrays.  Two instances, so that the first never waits on a memory
    // load other than its poll (a wait for a load also waits for the stores before it).
    const float keep = sp.keep;
    // tune bits 4-6: poll back-off level; bit 1: poll the two hint words before the full load
    // (inboxes within 2 GiB); bit 2: adaptive back-off
    const uint32_t nap = (tune >> 4) & 7u;
    const bool wide = (uint64_t)cap * IB_WORDS * 8u <= 0x7FFFFFFFull;  // 16-byte inbox loads
    const bool hint = (tune & 2u) != 0u && wide, adaptive = (tune & 4u) != 0u;
    const uint64_t t_start = wall_clock64();
    const uint64_t t_limit = (uint64_t)spin_limit * 100ull;  // wall clock: 100 MHz

    // Final velocity of dynamic body `body` after `sweeps` sweeps: the inbox of its
    // first visit (lowest colour) once it holds version sweeps * deg.  No visit of a
    // later sweep runs before the check's grid barrier, so the words stay put.
    auto final_vel = [&](uint32_t body, uint32_t dpw, uint32_t sweeps, SB& X) -> bool {
        const uint32_t v0 = B.vslot[(size_t)body * 64u + (uint32_t)__ffsll((unsigned long long)bmask[body]) - 1u];
        const uint32_t want = (sweeps * (dpw >> 8)) & 0xFFFFu, vs = v0 >> 1, side = v0 & 1u;
        const uint64_t* ib = R.inbox;
        for (;;) {
            const uint2 a0 = vsplit(vload(ib + vin_word(vs, side, 0))), a1 = vsplit(vload(ib + vin_word(vs, side, 1))),
                        a2 = vsplit(vload(ib + vin_word(vs, side, 2))), a3 = vsplit(vload(ib + vin_word(vs, side, 3)));
            const uint32_t d = (vver2(a0) ^ want) | (vver2(a1) ^ want) | (vver2(a2) ^ want) | (vver2(a3) ^ want);
            if (d == 0u) {
                vunpack4(a0, a1, a2, a3, X.v, X.w);
                return true;
            }
            if (wall_clock64() - t_start > t_limit) {
                atomicOr(err, STICKY_TIMEOUT);
                return false;
            }
            __builtin_amdgcn_s_sleep(1);
        }
    };
    // Residual check after `sweeps` sweeps: the k_residual value over this lane's
    // slots (rows and impulses where they are staged), wave max, one atomic max per
    // wave into stop.bits[sweeps - 1] (the history the host reads), and one atomic
    // add per wave into its arrival row of the check that carries both the arrival
    // (low 16 bits) and whether this wave's maximum is above the tolerance (bit 16
    // up): the decision needs no second round trip for the maximum.  Once the rows
    // sum to every workgroup, the launch stops when no wave was above the tolerance
    // (the same test as maximum <= tol).  Everything the waves exchange here and in
    // the sweep goes through device-scope atomics, so the barrier needs no cache
    // writeback or invalidation.  Returns 1 to stop, 0 to go on, -1 on an error.
    auto check = [&](uint32_t sweeps) -> int {
        float res = 0.0f;
        uint32_t off = 0;
        for (uint32_t j = 0; j < nv; ++j) {
            const Item it = j < nrec ? item_get(recs + (size_t)j * 4u * OWN_WAVE) : item_global(B, R, slot_of(j));
            const bool plane = (it.h.y & PLANE_BIT) != 0u;
            const uint32_t np = min(it.h.z, 4u);
            SB A, Bd;
            zero_sb(A);
            zero_sb(Bd);
            A.v = it.sv;
            A.w = it.sw;
            if (!plane) {
                Bd.v = it.sv;
                Bd.w = it.sw;
            }
            bool got = true;
            if (it.dp.x != UNSET) got &= final_vel(it.h.x, it.dp.x, sweeps, A);
            if (it.dp.y != UNSET) got &= final_vel(it.h.y, it.dp.y, sweeps, Bd);
            if (!got) break;
            const bool staged = staged_slot(j);
            for (uint32_t k = 0; k < np; ++k) {
                const float4* J = staged ? mine + (size_t)(off + k) * OWN_WAVE : R.J + (size_t)k * JROWS * cap + it.s;
                const size_t jr = staged ? rs : (size_t)cap;
                const float4 L = staged ? J[JROWS * jr] : R.lam[(size_t)k * cap + it.s];
                const float e = point_residual(J, jr, plane, keep, A, Bd, L);
                if (e > res) res = e;
            }
            off += staged ? np : 0u;
        }
        uint32_t bits = __float_as_uint(res);
        for (int o = 32; o >= 1; o >>= 1) {
            const uint32_t ob = __shfl_xor(bits, o, 64);
            bits = ob > bits ? ob : bits;
        }
        uint32_t* arr = stop.arrive + (size_t)(sweeps - 1u) * CHECK_ROWS * CHECK_ROW_WORDS;
        if (lane == 0u) {
            atomicMax(stop.bits + sweeps - 1u, bits);
            const bool above = __uint_as_float(bits) > stop.tol;
            __hip_atomic_fetch_add(arr + (g % CHECK_ROWS) * CHECK_ROW_WORDS, 1u + (above ? CHECK_ABOVE : 0u),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        bool late = false;
        uint32_t seen;
        for (;;) {
            // the rows summed (arrivals stay below 2^16, so the halves add apart); uniform
            // loads, no cross-lane steps (the sweep loop's register allocation stays as it is)
            seen = 0u;
#pragma unroll
            for (uint32_t r = 0; r < CHECK_ROWS; ++r)
                seen += __hip_atomic_load(arr + r * CHECK_ROW_WORDS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((seen & (CHECK_ABOVE - 1u)) >= G) break;
            if (wall_clock64() - t_start > t_limit) {
                late = true;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        if (late) {
            if (lane == 0u) atomicOr(err, STICKY_TIMEOUT);
            return -1;
        }
        if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) return -1;
        return seen < CHECK_ABOVE ? 1 : 0;
    };
    const bool checks = stop.bits != nullptr;
    uint32_t chunk_end = checks ? min(stop.every, nsweeps) : nsweeps;  // in the end the sweeps run
    auto sweep_loop = [&]<bool STAGED>() -> bool {
        uint32_t total = nv * chunk_end;
        uint32_t done = 0, sw = 0, j = 0, off = 0;
        Item it;
        it.s = 0u;
        if (total > 0u) it = (STAGED || nrec > 0u) ? item_get(recs) : item_global(B, R, slot_of(0));
        uint32_t s = it.s;
        bool fresh = true;
        uint32_t tA = 0, tB = 0, np = 0;
        bool plane = false;
        SB A, Bd;
        zero_sb(A);
        zero_sb(Bd);
        uint32_t spins = 0, idle = 0;
        for (;;) {
            const bool pending = done < total;
            if (pending && fresh) {
                fresh = false;
                tA = it.dp.x == UNSET ? 0u : sw * (it.dp.x >> 8) + (it.dp.x & 0xFFu);
                tB = it.dp.y == UNSET ? 0u : sw * (it.dp.y >> 8) + (it.dp.y & 0xFFu);
                plane = (it.h.y & PLANE_BIT) != 0u;
                np = min(it.h.z, 4u);
                A.im = it.imA;
                A.dyn = it.dp.x != UNSET;
                Bd.im = plane ? 0.0f : it.imB;
                Bd.dyn = it.dp.y != UNSET;
                if (!A.dyn) {
                    A.v = it.sv;
                    A.w = it.sw;
                }
                if (plane) {
                    Bd.v = Bd.w = f3{0.0f, 0.0f, 0.0f};
                } else if (!Bd.dyn) {
                    Bd.v = it.sv;
                    Bd.w = it.sw;
                }
            }
            // poll = load: all words of both bodies in this slot's inbox (one line), issued together
            bool ok = false;
            bool ready = pending;
            if (pending && hint) {
                // the two hint words first; the full load below runs only for lanes
                // whose hint words are in
                const uint64_t ha = vload(R.inbox + vin_word(s, 0, IB_HINT)), hb = vload(R.inbox + vin_word(s, 1, IB_HINT));
                ready = ((vver2(vsplit(ha)) == (tA & 0xFFFFu)) | !A.dyn) & ((vver2(vsplit(hb)) == (tB & 0xFFFFu)) | !Bd.dyn);
            }
            if (ready) {
                // (low, high) dwords of the four words of each side
                uint2 a[4], b[4];
                if (wide) {
                    // 16-byte loads, two per side
                    const uint4 q0 = vin_quad(R.inbox, s, 0), q1 = vin_quad(R.inbox, s, 2),
                                q2 = vin_quad(R.inbox, s, 4), q3 = vin_quad(R.inbox, s, 6);
                    a[0] = make_uint2(q0.x, q0.y), a[1] = make_uint2(q0.z, q0.w);
                    a[2] = make_uint2(q1.x, q1.y), a[3] = make_uint2(q1.z, q1.w);
                    b[0] = make_uint2(q2.x, q2.y), b[1] = make_uint2(q2.z, q2.w);
                    b[2] = make_uint2(q3.x, q3.y), b[3] = make_uint2(q3.z, q3.w);
                } else {
                    const uint64_t* ib = R.inbox;
#pragma unroll
                    for (uint32_t k = 0; k < IB_SIDE; ++k) {
                        a[k] = vsplit(vload(ib + vin_word(s, 0, k)));
                        b[k] = vsplit(vload(ib + vin_word(s, 1, k)));
                    }
                }
                // branch-free: every loaded word is consumed here, so no later instruction
                // waits on the memory counter (which also counts the stores before it)
                const uint32_t tA16 = tA & 0xFFFFu, tB16 = tB & 0xFFFFu;
                const uint32_t da = (vver2(a[0]) ^ tA16) | (vver2(a[1]) ^ tA16) | (vver2(a[2]) ^ tA16) |
                                    (vver2(a[3]) ^ tA16);
                const uint32_t db = (vver2(b[0]) ^ tB16) | (vver2(b[1]) ^ tB16) | (vver2(b[2]) ^ tB16) |
                                    (vver2(b[3]) ^ tB16);
                ok = ((da == 0u) | !A.dyn) & ((db == 0u) | !Bd.dyn);
                const bool ta = ok & A.dyn, tb = ok & Bd.dyn;
                f3 av, aw, bv, bw;
                vunpack4(a[0], a[1], a[2], a[3], av, aw);
                vunpack4(b[0], b[1], b[2], b[3], bv, bw);
                A.v = f3{ta ? av.x : A.v.x, ta ? av.y : A.v.y, ta ? av.z : A.v.z};
                A.w = f3{ta ? aw.x : A.w.x, ta ? aw.y : A.w.y, ta ? aw.z : A.w.z};
                Bd.v = f3{tb ? bv.x : Bd.v.x, tb ? bv.y : Bd.v.y, tb ? bv.z : Bd.v.z};
                Bd.w = f3{tb ? bw.x : Bd.w.x, tb ? bw.y : Bd.w.y, tb ? bw.z : Bd.w.z};
            }
            if (ok) {
                const bool first = sw == 0u;
                float4 L[4];
                // the point loops run over a fixed 4 so that L stays in registers
                const bool stg = STAGED || staged_slot(j);
                if (stg) {
                    float4* P = mine + (size_t)off * OWN_WAVE;
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k)
                        if (k < np) L[k] = P[JROWS * rs + (size_t)k * OWN_WAVE];
                    solve_rows(P, rs, OWN_WAVE, np, plane, keep, first, A, Bd, L);
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k)
                        if (k < np) P[JROWS * rs + (size_t)k * OWN_WAVE] = L[k];
                } else {
                    float4 Jr[4][JROWS];
                    load_rows(R, s, cap, np, plane, Jr);
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k)
                        if (k < np) L[k] = R.lam[(size_t)k * cap + s];
                    solve_regs(Jr, np, keep, first, A, Bd, L);
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k)
                        if (k < np) R.lam[(size_t)k * cap + s] = make_float4(L[k].x, L[k].y, L[k].z, 0.0f);
                }
                // pass the velocities on to each body's next visit
                if (A.dyn) vin_store(R.inbox, it.nx.x >> 1, it.nx.x & 1u, tA + 1u, A.v, A.w, wide);
                if (Bd.dyn) vin_store(R.inbox, it.nx.y >> 1, it.nx.y & 1u, tB + 1u, Bd.v, Bd.w, wide);
                // next item of this lane: the next owned slot, or the first one of the next sweep
                ++done;
                off += stg ? np : 0u;
                if (++j == nv) {
                    j = 0;
                    ++sw;
                    off = 0;
                }
                fresh = true;
                if (done < total) {
                    it = (STAGED || j < nrec) ? item_get(recs + (size_t)j * 4u * OWN_WAVE)
                                              : item_global(B, R, slot_of(j));
                    s = it.s;
                }
            }
            if (!__ballot(done < total)) {
                if (!checks) return true;
                // every slot of this wave is through sweep chunk_end - 1
                const int r = check(chunk_end);
                if (r < 0) return false;
                if (r > 0 || chunk_end == nsweeps) {
                    if (g == 0u && lane == 0u) {
                        __hip_atomic_store(&cnt->sweeps_run, chunk_end, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        __hip_atomic_store(&cnt->tol_hit, r > 0 ? 1u : 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                    return true;
                }
                chunk_end = min(chunk_end + stop.every, nsweeps);
                total = nv * chunk_end;
                if (nv > 0u) {
                    it = (STAGED || nrec > 0u) ? item_get(recs) : item_global(B, R, slot_of(0));
                    s = it.s;
                }
                fresh = true;
                continue;
            }
            if ((++spins & 255u) == 0u) {
                bool quit = false;
                if (wall_clock64() - t_start > t_limit) {
                    if (done < total) atomicOr(err, STICKY_TIMEOUT);  // waited longer than spin_limit microseconds
                    quit = true;
                } else if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) {
                    quit = true;  // another wave already gave up: drain
                }
                if (quit) return false;
            }
            // adaptive back-off: a wave none of whose lanes got through sleeps longer each time
            if (adaptive) idle = __ballot(ok) ? 0u : min(idle + 1u, 4u);
            switch (min(nap + idle, 6u)) {
            case 0: break;
            case 1: __builtin_amdgcn_s_sleep(1); break;
            case 2: __builtin_amdgcn_s_sleep(2); break;
            case 3: __builtin_amdgcn_s_sleep(4); break;
            case 4: __builtin_amdgcn_s_sleep(8); break;
            case 5: __builtin_amdgcn_s_sleep(16); break;
            default: __builtin_amdgcn_s_sleep(32); break;
            }
        }
    };
    const bool finished = __ballot(!all_staged) == 0ull ? sweep_loop.template operator()<true>()
                                                        : sweep_loop.template operator()<false>();
    if (!finished) return;

    // each dynamic body's velocity after the last sweep, by the lane of its first visit
    for (uint32_t j = 0; j < nv; ++j) {
        const Item it = j < nrec ? item_get(recs + (size_t)j * 4u * OWN_WAVE) : item_global(B, R, slot_of(j));
        SB X;
        if (it.dp.x != UNSET && (it.dp.x & 0xFFu) == 0u && final_vel(it.h.x, it.dp.x, chunk_end, X)) {
            B.sv[it.h.x] = f4(X.v, it.imA);
            B.sw[it.h.x] = f4(X.w, 0.0f);
        }
        if (it.dp.y != UNSET && (it.dp.y & 0xFFu) == 0u && final_vel(it.h.y, it.dp.y, chunk_end, X)) {
            B.sv[it.h.y] = f4(X.v, it.imB);
            B.sw[it.h.y] = f4(X.w, 0.0f);
        }
    }
    // impulses of the staged points back to the rows
    uint32_t woff = 0;
    for (uint32_t jj = 0; jj < nv; ++jj) {
        const uint32_t ss = slot_of(jj);
        if (!staged_slot(jj)) continue;
        const uint32_t n = min(jj < nrec ? __float_as_uint(recs[(size_t)jj * 4u * OWN_WAVE].z) : R.hdr[ss].z, 4u);
        for (uint32_t k = 0; k < n; ++k) {
            const float4 L = mine[(JROWS * rs) + (size_t)(woff + k) * OWN_WAVE];
            R.lam[(size_t)k * cap + ss] = make_float4(L.x, L.y, L.z, 0.0f);
        }
        woff += n;
    }
}

__global__ void __launch_bounds__(256) k_residual(Bodies B, StepParams sp, SolverRows R, const Counters* cnt,
                                                  uint32_t cap, uint32_t* __restrict__ out_bits) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t M = cnt->m_glob;  // the large islands' slots (the small ones report their own)
    float res = 0.0f;
    if (s < M && cnt->sticky == 0u) {  // rows exist only when the preparation ran
        uint4 h = R.hdr[s];
        h.z = min(h.z, 4u);
        const bool plane = (h.y & PLANE_BIT) != 0;
        SB A, Bd;
        load_vel<false>(B, h.x, A);
        if (plane) zero_sb(Bd); else load_vel<false>(B, h.y, Bd);
        for (uint32_t k = 0; k < h.z; ++k) {
            const float e = point_residual(R.J + (size_t)k * JROWS * cap + s, cap, plane, sp.keep, A, Bd,
                                           R.lam[(size_t)k * cap + s]);
            if (e > res) res = e;
        }
    }
    // wave max, then one atomic per wave (non-negative floats order as their bits)
    uint32_t bits = __float_as_uint(res);
    for (int o = 32; o >= 1; o >>= 1) {
        const uint32_t ob = __shfl_xor(bits, o, 64);
        bits = ob > bits ? ob : bits;
    }
    if ((threadIdx.x & 63) == 0) atomicMax(out_bits, bits);
}

// ---------------------------------------------------------------- islands solved on their own
// The manifolds of an island of at most ISLAND_LOCAL_MAX manifolds share no dynamic body
// with any other island, so the island is solved by itself: sweeps over its slots in
// solve order (colour, then manifold), and with a tolerance it stops after the first
// sweep that leaves its own residual <= tol.  Without a tolerance it runs every sweep, and
// the result is bit-identical to sweeping all islands together colour by colour.

// Residual of solve slot s (the k_residual value of its points).
__device__ __forceinline__ float slot_residual(const Bodies& B, float keep, const SolverRows& R, uint32_t s,
                                               uint32_t cap) {
    const uint4 h = R.hdr[s];
    const uint32_t np = min(h.z, 4u);
    const bool plane = (h.y & PLANE_BIT) != 0;
    SB A, Bd;
    load_vel<false>(B, h.x, A);
    if (plane) zero_sb(Bd); else load_vel<false>(B, h.y, Bd);
    float res = 0.0f;
    for (uint32_t k = 0; k < np; ++k) {
        const float e = point_residual(R.J + (size_t)k * JROWS * cap + s, cap, plane, keep, A, Bd,
                                       R.lam[(size_t)k * cap + s]);
        if (e > res) res = e;
    }
    return res;
}
// Results of the islands a thread reports: the most sweeps, the largest final residual
// (bits), whether one missed the tolerance, contact points and contact points x sweeps.
struct IslandAcc {
    uint32_t sweeps, res_bits, miss, pts;
    unsigned long long point_sweeps;
    __device__ void add(uint32_t sw, float res, bool missed, uint32_t p) {
        sweeps = max(sweeps, sw);
        res_bits = max(res_bits, __float_as_uint(res));
        miss |= missed ? 1u : 0u;
        pts += p;
        point_sweeps += (unsigned long long)p * sw;
    }
};
// Folds a wave's results into the counters: once per wave and launch, since every atomic
// here is on a word all waves share.
__device__ __forceinline__ void island_flush(Counters* cnt, IslandAcc a, bool islands_kernel = true) {
    for (int o = 32; o >= 1; o >>= 1) {
        a.sweeps = max(a.sweeps, (uint32_t)__shfl_xor((int)a.sweeps, o, 64));
        a.res_bits = max(a.res_bits, (uint32_t)__shfl_xor((int)a.res_bits, o, 64));
        a.miss |= (uint32_t)__shfl_xor((int)a.miss, o, 64);
        a.pts += (uint32_t)__shfl_xor((int)a.pts, o, 64);
        a.point_sweeps += __shfl_xor(a.point_sweeps, o, 64);
    }
    if ((threadIdx.x & 63u) != 0u || a.pts == 0u) return;
    atomicMax(&cnt->loc_sweeps, a.sweeps);
    atomicMax(&cnt->loc_res_bits, a.res_bits);
    if (a.miss) atomicOr(&cnt->loc_miss, 1u);
    atomicAdd(&cnt->loc_points, a.pts);
    atomicAdd(&cnt->loc_point_sweeps, a.point_sweeps);
    if (islands_kernel) atomicAdd(&cnt->bundle_point_sweeps, a.point_sweeps);
}
// Orders a wave's LDS accesses before and after this point (a wave's LDS operations execute
// in order, so no wait is needed, only that the compiler moves none across).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
constexpr uint32_t ISL_THREADS = 512, ISL_WAVES = ISL_THREADS / 64u;
// Block-wide maximum and sum over the workgroup's waves (red: two words of LDS per wave);
// every thread gets both.
__device__ __forceinline__ void block_max_sum(uint32_t& mx, uint32_t& sum, uint32_t* red) {
    for (int o = 32; o >= 1; o >>= 1) {
        const uint32_t om = __shfl_xor(mx, o, 64), os = __shfl_xor(sum, o, 64);
        mx = om > mx ? om : mx;
        sum += os;
    }
    if ((threadIdx.x & 63u) == 0u) {
        red[2u * (threadIdx.x >> 6)] = mx;
        red[2u * (threadIdx.x >> 6) + 1u] = sum;
    }
    __syncthreads();
    mx = sum = 0u;
#pragma unroll
    for (uint32_t w = 0; w < ISL_WAVES; ++w) {
        mx = max(mx, red[2u * w]);
        sum += red[2u * w + 1u];
    }
    __syncthreads();
}
// The small islands' kernel: one workgroup of eight waves per CU, two waves per SIMD.  A sweep
// of an island is a chain of dependent visits, colour after colour, and each visit a chain of
// three row updates per contact point.  What binds is that chain, so what a sweep touches
// stays on chip: rows and impulses in registers (a lane visits the same slot in every sweep),
// body velocities in LDS.  Velocities and impulses go back to memory once per island.  Above
// 256 manifolds a CU no longer holds the rows (240 B per point): those islands run across CUs in
// the large islands' register sweep (flow_part), or, when there are too many (wide_pieces), here
// with the rows read at each visit.
//
// Work is taken largest first, so that the long solves start early and the short ones fill
// the tail.  The workgroups first share the islands of more than 64 manifolds, one island at
// a time; then each wave on its own takes islands of the smaller classes, several to a wave
// in blocks of 64, 32 or 16 lanes, and last the windows of the islands of at most
// ISLAND_LANE_MAX manifolds: those whose first slot lies in one run of BUNDLE_SLOTS slots, one
// lane per slot (at most BUNDLE_SLOTS + ISLAND_LANE_MAX - 1 lanes).
//
// Each sweep runs phases: in phase p every island of the wave (or the workgroup's island)
// visits the slots of its p-th colour, all at once (within an island a colour's slots share no
// dynamic body, and islands share none at all); then each island's residual is the maximum
// over its lanes, and an island that is done stops while the others go on.  The visits are the
// arithmetic of solve_slot.  A body's velocity has one home in LDS, that of its first visit in
// a sweep (the lowest colour of its mask, whose slot the row preparation recorded in vslot).
//
// Per step, before (a workgroup of 256 threads per island of 9 to 4096 manifolds, rows and
// velocities in memory; a kernel of its own for the smaller ones) and now: 1000 bodies at
// residual 1e-4 (76 sweeps, largest island 154 manifolds) 1.55 -> 0.47 ms; 256 worlds at 1e-4
// (159k manifolds, 119 sweeps) 7.2 -> 2.8 ms; 4096 worlds at ten sweeps (1.7M manifolds)
// 11.3 -> 1.1 ms.
constexpr uint32_t BUNDLE_SLOTS = 56;
static_assert(BUNDLE_SLOTS + ISLAND_LANE_MAX - 1u <= 64u, "a bundle fits one wave");
// LDS of a wave's own work
constexpr uint32_t LAST_ROWS = JROWS - 1u;
struct WaveLds {
    float4 vel[256];              // v of the homes (64 * side + lane), then w
    float4 last[LAST_ROWS * 64];  // rows of every lane's fourth point (the last row in spare .w)
    uint32_t res[2][64];          // per island (its first lane): residual bits, two sweeps
    uint32_t pts[64];             // per island: contact points
    uint2 ab[64];
};
// LDS of a workgroup's island: this, then (above 256 manifolds) the tables, then the velocities
struct GroupLds {
    uint32_t off[66];  // first slot (island-relative) of colour >= c
    uint32_t red[2 * ISL_WAVES];
    unsigned long long mask;  // the island's colours
    uint32_t bodies, next;
};
constexpr uint32_t ISL_LDS_BYTES = 160u * 1024u;
constexpr uint32_t ISL_HEAD = (sizeof(GroupLds) + 15u) / 16u * 16u;
constexpr uint32_t ISL_TABLE_BYTES = 5u * ISLAND_LOCAL_MAX;  // 16-bit homes of both sides, points of every slot
static_assert(ISL_HEAD + ISL_TABLE_BYTES + 32u * (ISLAND_LOCAL_MAX + 1u) <= ISL_LDS_BYTES,
              "the velocities of any island's dynamic bodies fit");
static_assert(ISL_WAVES * sizeof(WaveLds) <= ISL_LDS_BYTES, "the waves' parts fit");
// homes of a side without a dynamic body: a plane, a static body
constexpr uint32_t PLANE_HOME = 0xFFFEu, NO_HOME = 0xFFFFu;

__device__ __forceinline__ void vel_load(const float4* v, const float4* w, uint32_t h, SB& X) {
    const float4 a = v[h], b = w[h];
    X.v = xyz(a);
    X.im = a.w;
    X.w = xyz(b);
    X.dyn = a.w > 0.0f;
}
__device__ __forceinline__ void vel_store(float4* v, float4* w, uint32_t h, const SB& X) {
    v[h] = f4(X.v, X.im);
    w[h] = f4(X.w, 0.0f);
}
__device__ __forceinline__ void vel_out(const Bodies& B, uint32_t body, const SB& X) {
    B.sv[body] = f4(X.v, X.im);
    B.sw[body] = f4(X.w, 0.0f);
}
// The first visit of a dynamic body in a sweep: slot << 1 | side.
__device__ __forceinline__ uint32_t first_visit(const Bodies& B, const uint64_t* __restrict__ bmask, uint32_t body) {
    return B.vslot[(size_t)body * 64u + (uint32_t)__ffsll((unsigned long long)bmask[body]) - 1u];
}
// Row updates of a point: relative velocity, projection, impulse.
__device__ __forceinline__ void friction_row(const Dir& D, float m, float maxf, float keep, float& l, SB& A, SB& Bd) {
    float nl = fmaf(-m, jvel(D, A, Bd), keep * l);
    nl = clamp_sym(nl, maxf);
    const float d = nl - l;
    l = nl;
    japply_both(D, d, A, Bd);
}
__device__ __forceinline__ void normal_row(const Dir& D, float m, float tg, float keep, float& l, SB& A, SB& Bd) {
    float nl = fmaf(m, tg - jvel(D, A, Bd), keep * l);
    nl = fmaxf(nl, 0.0f);
    const float d = nl - l;
    l = nl;
    japply_both(D, d, A, Bd);
}
__device__ __forceinline__ void friction_regs(const float4 (&J)[JROWS], float keep, float4& L, SB& A, SB& Bd) {
    float m1, m2, maxf, w3;
    const Dir D1 = dir_regs(J, 1, m1, maxf);
    friction_row(D1, m1, maxf, keep, L.y, A, Bd);
    const Dir D2 = dir_regs(J, 2, m2, w3);
    friction_row(D2, m2, maxf, keep, L.z, A, Bd);
}
__device__ __forceinline__ void normal_regs(const float4 (&J)[JROWS], float keep, float4& L, SB& A, SB& Bd) {
    float m, tg;
    const Dir D = dir_regs(J, 0, m, tg);
    normal_row(D, m, tg, keep, L.x, A, Bd);
}
__device__ __forceinline__ void start_regs(const float4 (&J)[JROWS], const float4& L, SB& A, SB& Bd) {
    float w0, w3;
    japply_both(dir_regs(J, 0, w0, w3), L.x, A, Bd);
    japply_both(dir_regs(J, 1, w0, w3), L.y, A, Bd);
    japply_both(dir_regs(J, 2, w0, w3), L.z, A, Bd);
}
// The fourth point's rows in LDS: row r of a lane at last[r * 64]; the last row rides in the
// unused .w of rows 2, 4 and 7.
__device__ __forceinline__ void last_put(float4* last, const float4 (&J)[JROWS]) {
#pragma unroll
    for (uint32_t r = 0; r < LAST_ROWS; ++r) {
        float4 x = J[r];
        if (r == 2u) x.w = J[LAST_ROWS].x;
        if (r == 4u) x.w = J[LAST_ROWS].y;
        if (r == 7u) x.w = J[LAST_ROWS].z;
        last[r * 64u] = x;
    }
}
__device__ __forceinline__ void last_get(const float4* last, float4 (&J)[JROWS]) {
    // an opaque zero: each use reads the rows it needs, none is kept in registers for the next
    uint32_t zero = 0u;
    asm volatile("" : "+v"(zero));
    last += zero;
#pragma unroll
    for (uint32_t r = 0; r < LAST_ROWS; ++r) J[r] = last[r * 64u];
    J[LAST_ROWS] = make_float4(J[2].w, J[4].w, J[7].w, 0.0f);
}
// The rows of point k of slot s (zeros for the b side of a plane contact).
__device__ __forceinline__ void point_rows(const SolverRows& R, uint32_t s, uint32_t cap, uint32_t k, bool plane,
                                           float4 (&J)[JROWS]) {
#pragma unroll
    for (uint32_t r = 0; r < JROWS; ++r) {
        const bool bside = (r % 5u) == 2u || (r % 5u) == 4u;
        J[r] = bside && plane ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : R.J[((size_t)k * JROWS + r) * cap + s];
    }
}

// Islands of one wave, one lane per slot: the lane's slot s (when mine), its island's first
// lane li and its colour.  search: the homes are found among the island's lanes instead of by
// the bodies' first visits (few lanes, or more colours than a mask holds).
__device__ __forceinline__ void wave_islands(const Bodies& B, float keep, const SolverRows& R, uint32_t cap, float tol,
                                             uint32_t max_sweeps, const uint64_t* __restrict__ bmask, WaveLds& W,
                                             bool mine, uint32_t s, uint32_t li, uint32_t colour, bool search,
                                             IslandAcc& acc) {
    const uint32_t lane = threadIdx.x & 63u;
    const bool tol_mode = tol > 0.0f;
    float4 *vv = W.vel, *vw = W.vel + 128, *last = W.last + lane;
    const uint4 h = mine ? R.hdr[s] : make_uint4(UNSET, UNSET, 0u, 0u);
    const uint32_t np = min(h.z, 4u);
    const bool plane = (h.y & PLANE_BIT) != 0u;
    W.ab[lane] = make_uint2(h.x, h.y);
    W.res[0][lane] = 0u;
    W.res[1][lane] = 0u;
    W.pts[lane] = 0u;
    // the slot's impulses and the rows of its first three points in registers
    float4 Jr[3][JROWS];
    float4 L[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) L[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    // a plane's side holds zeros (velocity, inverse mass): it loads as a static body
    float4 va = make_float4(0.0f, 0.0f, 0.0f, 0.0f), wa = va, vb = va, wb = va;
    if (mine) {
        va = B.sv[h.x];
        wa = B.sw[h.x];
        if (!plane) {
            vb = B.sv[h.y];
            wb = B.sw[h.y];
        }
        if (np > 3u) {
            float4 J[JROWS];
            point_rows(R, s, cap, 3u, plane, J);
            last_put(last, J);
        }
#pragma unroll
        for (uint32_t k = 0; k < 3; ++k)
            if (k < np) point_rows(R, s, cap, k, plane, Jr[k]);
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
            if (k < np) L[k] = R.lam[(size_t)k * cap + s];
    }
    const bool dyn_a = va.w > 0.0f, dyn_b = vb.w > 0.0f;
    wave_sync();
    // home of each side; the lane's phase: the colours of its island below its own (an
    // island's slots ascend by colour)
    uint32_t home_a = lane, home_b = 64u + lane;
    const uint32_t before = (uint32_t)__shfl_up((int)colour, 1, 64);
    const uint64_t heads = __ballot(mine && lane != li && before != colour);
    const uint64_t upto = (2ull << lane) - 1ull, from = ~((2ull << li) - 1ull);
    const uint32_t phase = (uint32_t)__popcll(heads & upto & from);
    if (mine) {
        if (search) {
            auto home_of = [&](uint32_t body, uint32_t own) {
                for (uint32_t j = li; j <= lane; ++j) {
                    const uint2 o = W.ab[j];
                    if (o.x == body) return j;
                    if (o.y == body) return 64u + j;
                }
                return own;
            };
            home_a = home_of(h.x, lane);
            if (!plane) home_b = home_of(h.y, 64u + lane);
        } else {
            const uint32_t s0 = s - (lane - li);
            if (dyn_a) {
                const uint32_t f = first_visit(B, bmask, h.x);
                home_a = (f & 1u) * 64u + (((f >> 1) - s0 + li) & 63u);
            }
            if (dyn_b) {
                const uint32_t f = first_visit(B, bmask, h.y);
                home_b = (f & 1u) * 64u + (((f >> 1) - s0 + li) & 63u);
            }
        }
        vv[lane] = va;
        vw[lane] = make_float4(wa.x, wa.y, wa.z, 0.0f);
        vv[64u + lane] = vb;
        vw[64u + lane] = make_float4(wb.x, wb.y, wb.z, 0.0f);
        atomicAdd(&W.pts[li], np);
    }
    uint32_t phases = mine ? phase + 1u : 0u;
    for (int o = 32; o >= 1; o >>= 1) phases = max(phases, (uint32_t)__shfl_xor((int)phases, o, 64));
    wave_sync();
    bool active = mine;
    uint32_t sweeps = 0;
    float res = 0.0f;
    for (uint32_t it = 0; it < max_sweeps; ++it) {
        if (__ballot(active) == 0ull) break;
        for (uint32_t c = 0; c < phases; ++c) {
            if (active && phase == c) {
                SB A, Bd;
                vel_load(vv, vw, home_a, A);
                vel_load(vv, vw, home_b, Bd);
                if (it == 0u) {
#pragma unroll
                    for (uint32_t k = 0; k < 3; ++k) {
                        if (k >= np) break;
                        start_regs(Jr[k], L[k], A, Bd);
                    }
                    if (np > 3u) {
                        float4 J[JROWS];
                        last_get(last, J);
                        start_regs(J, L[3], A, Bd);
                    }
                }
#pragma unroll
                for (uint32_t k = 0; k < 3; ++k) {
                    if (k >= np) break;
                    friction_regs(Jr[k], keep, L[k], A, Bd);
                }
                if (np > 3u) {
                    float4 J[JROWS];
                    last_get(last, J);
                    friction_regs(J, keep, L[3], A, Bd);
                }
#pragma unroll
                for (uint32_t k = 0; k < 3; ++k) {
                    if (k >= np) break;
                    normal_regs(Jr[k], keep, L[k], A, Bd);
                }
                if (np > 3u) {
                    float4 J[JROWS];
                    last_get(last, J);
                    normal_regs(J, keep, L[3], A, Bd);
                }
                if (A.dyn) vel_store(vv, vw, home_a, A);
                if (Bd.dyn) vel_store(vv, vw, home_b, Bd);
            }
            wave_sync();
        }
        if (tol_mode || it + 1u == max_sweeps) {
            uint32_t* cur = W.res[it & 1u];
            W.res[(it + 1u) & 1u][lane] = 0u;  // the next sweep's words (not read in this one)
            if (active) {
                SB A, Bd;
                vel_load(vv, vw, home_a, A);
                vel_load(vv, vw, home_b, Bd);
                float r = 0.0f;
#pragma unroll
                for (uint32_t k = 0; k < 3; ++k) {
                    if (k >= np) break;
                    const float e = point_residual_regs(Jr[k], keep, A, Bd, L[k]);
                    if (e > r) r = e;
                }
                if (np > 3u) {
                    float4 J[JROWS];
                    last_get(last, J);
                    const float e = point_residual_regs(J, keep, A, Bd, L[3]);
                    if (e > r) r = e;
                }
                atomicMax(&cur[li], __float_as_uint(r));
            }
            wave_sync();
            if (active) {
                res = __uint_as_float(cur[li]);
                if ((tol_mode && res <= tol) || it + 1u == max_sweeps) {
                    sweeps = it + 1u;
                    active = false;
                }
            }
        }
    }
    wave_sync();
    if (mine) {
        // impulses and the velocities of the bodies whose home this lane holds back to memory
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
            if (k < np) R.lam[(size_t)k * cap + s] = make_float4(L[k].x, L[k].y, L[k].z, 0.0f);
        SB X;
        if (dyn_a && home_a == lane) {
            vel_load(vv, vw, lane, X);
            vel_out(B, h.x, X);
        }
        if (dyn_b && home_b == 64u + lane) {
            vel_load(vv, vw, 64u + lane, X);
            vel_out(B, h.y, X);
        }
        if (lane == li) acc.add(sweeps, res, tol_mode && !(res <= tol), W.pts[li]);
    }
    wave_sync();
}

// ---- an island of 65 to 256 manifolds: two lanes of the workgroup per slot, one per body
// A visit is a chain of row updates, each 32 instructions with both bodies in one lane.  Two
// neighbouring lanes share them: the even lane holds body a's velocity and rows, the odd lane
// body b's, and the relative velocity is put together by DPP exchanges inside the adds.  That is
// 22 instructions per row, and half the registers, so every row of four points stays in them.
// The odd lane keeps -d, the even lane -a and -IA a: with these signs both lanes run the same
// instructions, and every product, sum and rounding is that of solve_rows (zeros may differ in
// sign).
template <int CTRL> __device__ __forceinline__ float dpp(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xF, 0xF, true));
}
constexpr int DPP_SWAP = 0xB1, DPP_EVEN = 0xA0, DPP_ODD = 0xF5;  // quad_perm [1,0,3,2], [0,0,2,2], [1,1,3,3]
struct HalfDir {
    f3 d, a, ia;
};
struct HalfPoint {
    HalfDir n, t1, t2;
    float mN, kN, tg, mT1, kT1, maxf, mT2, kT2;
};
struct HalfBody {
    f3 v, w;
    float im;
};
__device__ __forceinline__ float half_jvel(const HalfDir& D, const HalfBody& X) {
    const f3 dv = f3{dpp<DPP_SWAP>(X.v.x) - X.v.x, dpp<DPP_SWAP>(X.v.y) - X.v.y, dpp<DPP_SWAP>(X.v.z) - X.v.z};
    const float ang = fdot(D.a, X.w);
    const float r = fdot(D.d, dv) + dpp<DPP_ODD>(ang);
    return r + dpp<DPP_EVEN>(ang);
}
__device__ __forceinline__ void half_apply(const HalfDir& D, float lam, HalfBody& X) {
    const float s = -(lam * X.im);
    X.v = f3{fmaf(s, D.d.x, X.v.x), fmaf(s, D.d.y, X.v.y), fmaf(s, D.d.z, X.v.z)};
    X.w = f3{fmaf(lam, D.ia.x, X.w.x), fmaf(lam, D.ia.y, X.w.y), fmaf(lam, D.ia.z, X.w.z)};
}
__device__ __forceinline__ void half_friction(const HalfDir& D, float m, float maxf, float keep, float& l, HalfBody& X) {
    float nl = fmaf(-m, half_jvel(D, X), keep * l);
    nl = clamp_sym(nl, maxf);
    const float d = nl - l;
    l = nl;
    half_apply(D, d, X);
}
__device__ __forceinline__ void half_normal(const HalfDir& D, float m, float tg, float keep, float& l, HalfBody& X) {
    float nl = fmaf(m, tg - half_jvel(D, X), keep * l);
    nl = fmaxf(nl, 0.0f);
    const float d = nl - l;
    l = nl;
    half_apply(D, d, X);
}
// point_residual_regs of the pair (both lanes get it).
__device__ __forceinline__ float half_residual(const HalfPoint& P, float keep, const HalfBody& X, float ln, float l1,
                                               float l2) {
    float nl = fmaf(P.mN, P.tg - half_jvel(P.n, X), keep * ln);
    nl = fmaxf(nl, 0.0f);
    float e = fabsf(nl - ln) * P.kN;
    float q1 = fmaf(-P.mT1, half_jvel(P.t1, X), keep * l1);
    q1 = clamp_sym(q1, P.maxf);
    const float e1 = fabsf(q1 - l1) * P.kT1;
    float q2 = fmaf(-P.mT2, half_jvel(P.t2, X), keep * l2);
    q2 = clamp_sym(q2, P.maxf);
    const float e2 = fabsf(q2 - l2) * P.kT2;
    if (e1 > e) e = e1;
    if (e2 > e) e = e2;
    return e;
}
__device__ __forceinline__ void half_rows(const SolverRows& R, uint32_t s, uint32_t cap, uint32_t k, bool odd, bool plane,
                                          HalfPoint& P) {
    const float4* J = R.J + (size_t)k * JROWS * cap + s;
    auto dir = [&](uint32_t r0, HalfDir& D, float& m, float& kk, float& w3) {
        const float4 d = J[(size_t)r0 * cap], ra = J[(size_t)(r0 + 1u) * cap], ria = J[(size_t)(r0 + 3u) * cap];
        m = d.w;
        kk = ra.w;
        w3 = ria.w;
        // the b-side rows of a plane contact are not there: zeros
        float4 rb = make_float4(0.0f, 0.0f, 0.0f, 0.0f), rib = rb;
        if (odd && !plane) {
            rb = J[(size_t)(r0 + 2u) * cap];
            rib = J[(size_t)(r0 + 4u) * cap];
        }
        D.d = odd ? f3{-d.x, -d.y, -d.z} : xyz(d);
        D.a = odd ? xyz(rb) : f3{-ra.x, -ra.y, -ra.z};
        D.ia = odd ? xyz(rib) : f3{-ria.x, -ria.y, -ria.z};
    };
    float w3;
    dir(0u, P.n, P.mN, P.kN, P.tg);
    dir(5u, P.t1, P.mT1, P.kT1, P.maxf);
    dir(10u, P.t2, P.mT2, P.kT2, w3);
}
constexpr uint32_t PAIR_SLOTS = ISL_THREADS / 2u;
__device__ __forceinline__ void pair_island(const Bodies& B, float keep, const SolverRows& R, uint32_t cap, float tol,
                                            uint32_t max_sweeps, const uint64_t* __restrict__ bmask,
                                            const uint32_t* __restrict__ skey, unsigned char* lds, uint2 e,
                                            IslandAcc& acc) {
    GroupLds& G = *reinterpret_cast<GroupLds*>(lds);
    float4* vv = reinterpret_cast<float4*>(lds + ISL_HEAD);  // home of (slot, side): 2 * slot + side
    float4* vw = vv + 2u * PAIR_SLOTS;
    const uint32_t t = threadIdx.x, u = t >> 1, s0 = e.x, s = s0 + u;
    const bool odd = (t & 1u) != 0u, mine = u < e.y, tol_mode = tol > 0.0f;
    const uint32_t colour = mine ? skey[s] & 63u : 0u;
    if (t == 0u) G.mask = 0ull;
    const uint4 h = mine ? R.hdr[s] : make_uint4(UNSET, UNSET, 0u, 0u);
    const uint32_t np = min(h.z, 4u);
    const bool plane = (h.y & PLANE_BIT) != 0u;
    const uint32_t body = odd ? h.y : h.x;
    HalfPoint P[4];
    float ln[4], l1[4], l2[4];
    float4 v4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), w4 = v4;
    uint32_t home = t;
    if (mine) {
        if (!(odd && plane)) {
            v4 = B.sv[body];
            w4 = B.sw[body];
        }
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
            if (k < np) {
                half_rows(R, s, cap, k, odd, plane, P[k]);
                const float4 L = R.lam[(size_t)k * cap + s];
                ln[k] = L.x;
                l1[k] = L.y;
                l2[k] = L.z;
            }
        if (v4.w > 0.0f) home = min(first_visit(B, bmask, body) - 2u * s0, 2u * PAIR_SLOTS - 1u);
        vv[t] = v4;
        vw[t] = make_float4(w4.x, w4.y, w4.z, 0.0f);
    }
    const bool dyn = v4.w > 0.0f;
    HalfBody X;
    X.im = v4.w;
    auto get = [&]() {
        const float4 a = vv[home], b = vw[home];
        X.v = xyz(a);
        X.w = xyz(b);
    };
    __syncthreads();
    if (mine && !odd) atomicOr(&G.mask, 1ull << colour);
    __syncthreads();
    const uint64_t mask = G.mask;
    const uint32_t phases = (uint32_t)__popcll(mask);
    const uint32_t phase = mine ? (uint32_t)__popcll(mask & ((1ull << colour) - 1ull)) : UNSET;
    uint32_t it = 0;
    float res = 0.0f;
    for (; it < max_sweeps; ++it) {
        for (uint32_t c = 0; c < phases; ++c) {
            if (phase == c) {
                get();
                if (it == 0u) {
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k) {
                        if (k >= np) break;
                        half_apply(P[k].n, ln[k], X);
                        half_apply(P[k].t1, l1[k], X);
                        half_apply(P[k].t2, l2[k], X);
                    }
                }
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {
                    if (k >= np) break;
                    half_friction(P[k].t1, P[k].mT1, P[k].maxf, keep, l1[k], X);
                    half_friction(P[k].t2, P[k].mT2, P[k].maxf, keep, l2[k], X);
                }
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {
                    if (k >= np) break;
                    half_normal(P[k].n, P[k].mN, P[k].tg, keep, ln[k], X);
                }
                if (dyn) {
                    vv[home] = f4(X.v, X.im);
                    vw[home] = f4(X.w, 0.0f);
                }
            }
            __syncthreads();
        }
        if (tol_mode || it + 1u == max_sweeps) {
            float r = 0.0f;
            if (mine) {
                get();
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {
                    if (k >= np) break;
                    const float q = half_residual(P[k], keep, X, ln[k], l1[k], l2[k]);
                    if (q > r) r = q;
                }
            }
            uint32_t mx = __float_as_uint(r), unused = 0u;
            block_max_sum(mx, unused, G.red);
            res = __uint_as_float(mx);
            if (tol_mode && res <= tol) {
                ++it;
                break;
            }
        }
    }
    if (mine) {
        if (!odd) {
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
                if (k < np) R.lam[(size_t)k * cap + s] = make_float4(ln[k], l1[k], l2[k], 0.0f);
        }
        if (dyn && home == t) {
            get();
            B.sv[body] = f4(X.v, X.im);
            B.sw[body] = f4(X.w, 0.0f);
        }
    }
    uint32_t mx = 0u, pts = odd ? 0u : np;
    block_max_sum(mx, pts, G.red);
    if (t == 0u) acc.add(it, res, tol_mode && !(res <= tol), pts);
}

// ---- an island of more than 256 manifolds, one workgroup
// The dynamic bodies' velocities are packed in LDS, their homes numbered as their first visits
// claim them (at most one more than the manifolds); the rows, more than a CU holds, are read
// from the row arrays at each visit.  A lane asks for the rows of its next visit's first point
// before it waits at the barrier, and within a visit for the next point's rows before it works
// on this one's, so that most of their latency passes behind other work.
struct PointT {  // the friction rows of a point
    float4 r[10];
};
struct PointN {  // its normal rows
    float4 r[5];
};
__device__ __forceinline__ void rows_t(const SolverRows& R, uint32_t s, uint32_t cap, uint32_t k, bool plane, PointT& T) {
    const float4* J = R.J + ((size_t)k * JROWS + 5u) * cap + s;
#pragma unroll
    for (uint32_t r = 0; r < 10u; ++r) {
        const bool bside = r % 5u == 2u || r % 5u == 4u;
        T.r[r] = bside && plane ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : J[(size_t)r * cap];
    }
}
__device__ __forceinline__ void rows_n(const SolverRows& R, uint32_t s, uint32_t cap, uint32_t k, bool plane, PointN& N) {
    const float4* J = R.J + (size_t)k * JROWS * cap + s;
#pragma unroll
    for (uint32_t r = 0; r < 5u; ++r) {
        const bool bside = r == 2u || r == 4u;
        N.r[r] = bside && plane ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : J[(size_t)r * cap];
    }
}
__device__ __forceinline__ Dir dir_of(const float4* r) {
    return Dir{xyz(r[0]), xyz(r[1]), xyz(r[2]), xyz(r[3]), xyz(r[4])};
}
__device__ __forceinline__ void friction_t(const PointT& T, float keep, float4& L, SB& A, SB& Bd) {
    const float maxf = T.r[3].w;
    friction_row(dir_of(T.r), T.r[0].w, maxf, keep, L.y, A, Bd);
    friction_row(dir_of(T.r + 5), T.r[5].w, maxf, keep, L.z, A, Bd);
}
__device__ __forceinline__ void normal_n(const PointN& N, float keep, float4& L, SB& A, SB& Bd) {
    normal_row(dir_of(N.r), N.r[0].w, N.r[3].w, keep, L.x, A, Bd);
}
__device__ __forceinline__ void stream_island(const Bodies& B, float keep, const SolverRows& R, uint32_t cap, float tol,
                                              uint32_t max_sweeps, const uint64_t* __restrict__ bmask,
                                              const uint32_t* __restrict__ skey, unsigned char* lds, uint2 e,
                                              IslandAcc& acc) {
    GroupLds& G = *reinterpret_cast<GroupLds*>(lds);
    const uint32_t t = threadIdx.x, s0 = e.x, n = e.y;
    uint16_t* home = reinterpret_cast<uint16_t*>(lds + ISL_HEAD);
    uint8_t* pts_of = reinterpret_cast<uint8_t*>(home + 2u * ISLAND_LOCAL_MAX);
    float4* const vv = reinterpret_cast<float4*>(lds + ISL_HEAD + ISL_TABLE_BYTES);
    float4* const vw = vv + (ISLAND_LOCAL_MAX + 1u);
    const bool tol_mode = tol > 0.0f;
    if (t == 0u) G.bodies = 0u;
    const uint32_t c_end = (skey[s0 + n - 1u] & 0xFFu) + 1u;  // the island's colours lie below c_end (<= 64)
    __syncthreads();
    // colour offsets; points; homes of the bodies whose first visit is here, with their velocities
    for (uint32_t i = t; i < n; i += ISL_THREADS) {
        const uint32_t c = skey[s0 + i] & 0xFFu;
        for (uint32_t q = i ? (skey[s0 + i - 1u] & 0xFFu) + 1u : 0u; q <= c; ++q) G.off[q] = i;
        if (i == n - 1u) G.off[c_end] = n;
        const uint4 h = R.hdr[s0 + i];
        pts_of[i] = (uint8_t)min(h.z, 4u);
        auto claim = [&](uint32_t body, uint32_t at) {
            uint32_t id = (body & PLANE_BIT) ? PLANE_HOME : NO_HOME;
            if (id == NO_HOME) {
                const float4 v = B.sv[body];
                if (v.w > 0.0f && first_visit(B, bmask, body) == 2u * s0 + at) {
                    id = min(atomicAdd(&G.bodies, 1u), ISLAND_LOCAL_MAX);
                    const float4 w = B.sw[body];
                    vv[id] = v;
                    vw[id] = make_float4(w.x, w.y, w.z, 0.0f);
                }
            }
            home[at] = (uint16_t)id;
        };
        claim(h.x, 2u * i);
        claim(h.y, 2u * i + 1u);
    }
    __syncthreads();
    // the other visits' homes (a claimed entry is only read here)
    for (uint32_t i = t; i < n; i += ISL_THREADS) {
        const uint4 h = R.hdr[s0 + i];
        auto side = [&](uint32_t body, uint32_t at) {
            if (home[at] == NO_HOME && B.sv[body].w > 0.0f)
                home[at] = home[min(first_visit(B, bmask, body) - 2u * s0, 2u * n - 1u)];
        };
        side(h.x, 2u * i);
        side(h.y, 2u * i + 1u);
    }
    __syncthreads();
    // static partners are read from memory (planes: zeros)
    auto load_side = [&](uint32_t id, uint32_t i, uint32_t side, SB& X) {
        if (id < PLANE_HOME) {
            vel_load(vv, vw, id, X);
        } else {
            zero_sb(X);
            if (id == NO_HOME) load_vel<false>(B, side ? R.hdr[s0 + i].y : R.hdr[s0 + i].x, X);
        }
    };
    // this lane's visits in order: in colour c the slots off[c] + t, off[c] + t + 512, ...
    PointT T0;
    PointN N0;
    float4 L0;
    auto ask = [&](uint32_t c, uint32_t i) {
        // the first point of the visit after slot i of colour c (i UNSET: of the first one from
        // colour c on)
        uint32_t nx = UNSET;
        if (i != UNSET && i + ISL_THREADS < G.off[c + 1u]) {
            nx = i + ISL_THREADS;
        } else {
            for (uint32_t q = i == UNSET ? c : c + 1u; q < c_end; ++q)
                if (G.off[q] + t < G.off[q + 1u]) {
                    nx = G.off[q] + t;
                    break;
                }
        }
        if (nx != UNSET) {
            const bool plane = home[2u * nx + 1u] == PLANE_HOME;
            rows_t(R, s0 + nx, cap, 0u, plane, T0);
            rows_n(R, s0 + nx, cap, 0u, plane, N0);
            L0 = R.lam[s0 + nx];
        }
    };
    uint32_t it = 0;
    float res = 0.0f;
    for (; it < max_sweeps; ++it) {
        ask(0u, UNSET);
        for (uint32_t c = 0; c < c_end; ++c) {
            const uint32_t a = G.off[c], b = G.off[c + 1u];
            if (a == b) continue;
            for (uint32_t i = a + t; i < b; i += ISL_THREADS) {
                const uint32_t s = s0 + i, ia = home[2u * i], ib = home[2u * i + 1u], np = pts_of[i];
                const bool plane = ib == PLANE_HOME;
                SB A, Bd;
                load_side(ia, i, 0u, A);
                load_side(ib, i, 1u, Bd);
                float4 L[4];
                L[0] = L0;
                PointT Ta, Tb;
                PointN Na, Nb;
                if (np > 1u) {
                    rows_t(R, s, cap, 1u, plane, Ta);
#pragma unroll
                    for (uint32_t k = 1; k < 4; ++k)
                        if (k < np) L[k] = R.lam[(size_t)k * cap + s];
                }
                if (it == 0u) {
                    // the warm start (rows read again below)
                    japply_both(dir_of(N0.r), L[0].x, A, Bd);
                    japply_both(dir_of(T0.r), L[0].y, A, Bd);
                    japply_both(dir_of(T0.r + 5), L[0].z, A, Bd);
#pragma unroll
                    for (uint32_t k = 1; k < 4; ++k) {
                        if (k >= np) break;
                        rows_t(R, s, cap, k, plane, Tb);
                        rows_n(R, s, cap, k, plane, Nb);
                        japply_both(dir_of(Nb.r), L[k].x, A, Bd);
                        japply_both(dir_of(Tb.r), L[k].y, A, Bd);
                        japply_both(dir_of(Tb.r + 5), L[k].z, A, Bd);
                    }
                }
                friction_t(T0, keep, L[0], A, Bd);
                if (np > 1u) {
                    if (np > 2u) rows_t(R, s, cap, 2u, plane, Tb);
                    else rows_n(R, s, cap, 1u, plane, Na);
                    friction_t(Ta, keep, L[1], A, Bd);
                }
                if (np > 2u) {
                    if (np > 3u) rows_t(R, s, cap, 3u, plane, Ta);
                    rows_n(R, s, cap, 1u, plane, Na);
                    friction_t(Tb, keep, L[2], A, Bd);
                }
                if (np > 3u) friction_t(Ta, keep, L[3], A, Bd);
                if (np > 2u) rows_n(R, s, cap, 2u, plane, Nb);
                normal_n(N0, keep, L[0], A, Bd);
                if (np > 1u) normal_n(Na, keep, L[1], A, Bd);
                if (np > 3u) rows_n(R, s, cap, 3u, plane, Na);
                if (np > 2u) normal_n(Nb, keep, L[2], A, Bd);
                if (np > 3u) normal_n(Na, keep, L[3], A, Bd);
                if (ia < PLANE_HOME) vel_store(vv, vw, ia, A);
                if (ib < PLANE_HOME) vel_store(vv, vw, ib, Bd);
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k)
                    if (k < np) R.lam[(size_t)k * cap + s] = make_float4(L[k].x, L[k].y, L[k].z, 0.0f);
                ask(c, i);
            }
            __syncthreads();
        }
        if (tol_mode || it + 1u == max_sweeps) {
            float r = 0.0f;
            for (uint32_t i = t; i < n; i += ISL_THREADS) {
                SB A, Bd;
                load_side(home[2u * i], i, 0u, A);
                load_side(home[2u * i + 1u], i, 1u, Bd);
                const bool plane = home[2u * i + 1u] == PLANE_HOME;
                const uint32_t np = pts_of[i];
                for (uint32_t k = 0; k < np; ++k) {
                    const float q = point_residual(R.J + (size_t)k * JROWS * cap + s0 + i, cap, plane, keep, A, Bd,
                                                   R.lam[(size_t)k * cap + s0 + i]);
                    if (q > r) r = q;
                }
            }
            uint32_t mx = __float_as_uint(r), unused = 0u;
            block_max_sum(mx, unused, G.red);
            res = __uint_as_float(mx);
            if (tol_mode && res <= tol) {
                ++it;
                break;
            }
        }
    }
    uint32_t pts = 0;
    for (uint32_t i = t; i < n; i += ISL_THREADS) {
        pts += pts_of[i];
        const uint4 h = R.hdr[s0 + i];
        auto out = [&](uint32_t body, uint32_t at) {
            const uint32_t id = home[at];
            if (id >= PLANE_HOME || first_visit(B, bmask, body) != 2u * s0 + at) return;
            SB X;
            vel_load(vv, vw, id, X);
            vel_out(B, body, X);
        };
        out(h.x, 2u * i);
        out(h.y, 2u * i + 1u);
    }
    uint32_t mx = 0u;
    block_max_sum(mx, pts, G.red);
    if (t == 0u) acc.add(it, res, tol_mode && !(res <= tol), pts);
}

// An island with rows and velocities in memory (more colours than a body's colour mask holds).
// A colour's slots share no dynamic body, so the workgroup visits them together and meets at a
// barrier before the next colour (the velocities are visible within the workgroup after it).
__device__ __forceinline__ void memory_island(const Bodies& B, const StepParams& sp, const SolverRows& R, uint32_t cap,
                                              float tol, uint32_t max_sweeps, const uint32_t* __restrict__ skey,
                                              uint32_t* red, uint2 e, IslandAcc& acc) {
    const uint32_t s0 = e.x, s1 = e.x + e.y, t = threadIdx.x;
    const uint32_t k0 = skey[s0], k1 = skey[s1 - 1u];
    const bool tol_mode = tol > 0.0f;
    uint32_t it = 0;
    float res = 0.0f;
    for (; it < max_sweeps; ++it) {
        uint32_t a = s0;
        for (uint32_t c = k0 & 0xFFu; c <= (k1 & 0xFFu); ++c) {
            // [a, b): the island's slots of colour c (the keys ascend, equal above the colour)
            const uint32_t kc = (k0 & ~0xFFu) | c;
            uint32_t lo = a, hi = s1;
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                if (skey[mid] <= kc) lo = mid + 1u; else hi = mid;
            }
            if (lo > a) {
                for (uint32_t s = a + t; s < lo; s += blockDim.x) solve_slot(B, sp, R, R.hdr[s], s, cap, it == 0u);
                __syncthreads();
            }
            a = lo;
        }
        if (tol_mode || it + 1u == max_sweeps) {
            float r = 0.0f;
            for (uint32_t s = s0 + t; s < s1; s += blockDim.x) {
                const float q = slot_residual(B, sp.keep, R, s, cap);
                if (q > r) r = q;
            }
            uint32_t mx = __float_as_uint(r), unused = 0u;
            block_max_sum(mx, unused, red);
            res = __uint_as_float(mx);
            if (tol_mode && res <= tol) {
                ++it;
                break;
            }
        }
    }
    uint32_t pts = 0, mx = 0u;
    for (uint32_t s = s0 + t; s < s1; s += blockDim.x) pts += min(R.hdr[s].z, 4u);
    block_max_sum(mx, pts, red);
    if (t == 0u) acc.add(it, res, tol_mode && !(res <= tol), pts);
}

// wide: the register sweep takes the islands of the largest class.  The workgroups below `late`
// have swept large islands first: the others share the work out among themselves at the start,
// they take what is left.
__device__ __forceinline__ void islands_part(const Bodies& B, const StepParams& sp, const SolverRows& R, Counters* cnt,
                                             uint32_t cap, const uint2* __restrict__ list,
                                             const uint32_t* __restrict__ skey, float tol, uint32_t max_sweeps,
                                             const uint64_t* __restrict__ bmask, bool wide, uint32_t late,
                                             unsigned char* isl_lds) {
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t first = gridDim.x - late;  // workgroups that start with the islands
    const bool is_late = blockIdx.x < late;
    // the row preparation records no first visits when there are more colours than mask bits
    const bool masks = cnt->max_colour <= 64u;
    IslandAcc acc = {0u, 0u, 0u, 0u, 0ull};
    GroupLds& G = *reinterpret_cast<GroupLds*>(isl_lds);
    const uint32_t n0 = wide ? 0u : cnt->isl_n[0], n1 = cnt->isl_n[1], n2 = cnt->isl_n[2], n3 = cnt->isl_n[3], n4 = cnt->isl_n[4];

    // ---- islands of one workgroup each (without masks: every island of the list)
    const uint32_t n_wg = masks ? n0 + n1 : n0 + n1 + n2 + n3 + n4;
    uint32_t w0 = blockIdx.x - late;
    if (is_late) {
        if (t == 0u) G.next = first + (n_wg ? atomicAdd(&cnt->isl_wg_next, 1u) : 0u);
        __syncthreads();
        w0 = G.next;
        __syncthreads();
    }
    for (uint32_t w = w0; w < n_wg;) {
        uint32_t c = 0, i = w;
        if (i >= n0) c = 1u, i -= n0;
        if (c == 1u && i >= n1) c = 2u, i -= n1;
        if (c == 2u && i >= n2) c = 3u, i -= n2;
        if (c == 3u && i >= n3) c = 4u, i -= n3;
        const uint2 e = list[isl_region(c, cap) + i];
        if (!masks) memory_island(B, sp, R, cap, tol, max_sweeps, skey, G.red, e, acc);
        else if (c == 0u) stream_island(B, sp.keep, R, cap, tol, max_sweeps, bmask, skey, isl_lds, e, acc);
        else pair_island(B, sp.keep, R, cap, tol, max_sweeps, bmask, skey, isl_lds, e, acc);
        if (t == 0u) G.next = first + atomicAdd(&cnt->isl_wg_next, 1u);
        __syncthreads();
        w = G.next;
        __syncthreads();
    }
    __syncthreads();

    // ---- the rest, by waves
    WaveLds& W = reinterpret_cast<WaveLds*>(isl_lds)[t >> 6];
    const uint32_t M = min(cap, cnt->m_eff), M0 = cnt->m_glob;
    const uint32_t n64 = masks ? n2 : 0u, n32 = masks ? (n3 + 1u) / 2u : 0u, n16 = masks ? (n4 + 3u) / 4u : 0u;
    const uint32_t n_win = M > M0 ? (M - M0 + BUNDLE_SLOTS - 1u) / BUNDLE_SLOTS : 0u;
    const uint32_t n_wave = n64 + n32 + n16 + n_win;
    const uint32_t waves = first * ISL_WAVES;
    uint32_t v0 = blockIdx.x - late + first * (t >> 6);
    if (is_late) {
        uint32_t nx = 0;
        if (lane == 0u) nx = atomicAdd(&cnt->isl_wave_next, 1u);
        v0 = waves + (uint32_t)__shfl((int)nx, 0, 64);
    }
    for (uint32_t w = v0; w < n_wave;) {
        // the next piece is asked for before this one is worked on
        uint32_t nx = 0;
        if (lane == 0u) nx = atomicAdd(&cnt->isl_wave_next, 1u);
        bool mine = false, search = false;
        uint32_t s = 0, li = 0, colour = 0;
        if (w < n64 + n32 + n16) {
            const uint32_t c = w < n64 ? 2u : (w < n64 + n32 ? 3u : 4u);
            const uint32_t T = 64u >> (c - 2u);  // lanes per island
            const uint32_t unit = c == 2u ? w : (c == 3u ? w - n64 : w - n64 - n32);
            const uint32_t i = unit * (64u / T) + lane / T, u = lane % T;
            if (i < (c == 2u ? n2 : (c == 3u ? n3 : n4))) {
                const uint2 e = list[isl_region(c, cap) + i];
                mine = u < e.y;
                s = e.x + u;
                li = lane - u;
                if (mine) colour = skey[s] & 0xFFu;
            }
        } else {
            // a lane's slot belongs to the window when its island is small and its first slot
            // lies in it
            const uint32_t w0 = M0 + (w - n64 - n32 - n16) * BUNDLE_SLOTS;
            s = w0 + lane;
            search = true;
            if (s < M) {
                const uint32_t k = skey[s];
                if (B.icnt[(k & ~LOCAL_KEY) >> 8] <= ISLAND_LANE_MAX) {
                    uint32_t st = s;
                    while (st > M0 && ((skey[st - 1u] ^ k) >> 8) == 0u) --st;  // at most ISLAND_LANE_MAX - 1 steps
                    mine = st >= w0 && st < w0 + BUNDLE_SLOTS;
                    li = mine ? st - w0 : 0u;
                    colour = k & 0xFFu;
                }
            }
        }
        if (__ballot(mine) != 0ull)
            wave_islands(B, sp.keep, R, cap, tol, max_sweeps, bmask, W, mine, s, li, colour, search, acc);
        w = waves + (uint32_t)__shfl((int)nx, 0, 64);
    }
    island_flush(cnt, acc);
}

// ---------------------------------------------------------------- large islands in registers
// The large islands' sweeps when every slot has two lanes of the GPU to itself (flow_slots
// slots at most; k_pgs_own takes more): the even lane of a pair holds body a's side of the
// slot's rows, the odd lane body b's (half_jvel), with the impulses, in registers for the whole
// solve.  Visits pass velocities on through the inboxes as in k_pgs_own; with one slot per pair
// a wave's lanes wait for nothing but their own bodies, and a visit reads only the 32 bytes of
// its inbox side from memory.  What binds is the chain of dependent visits: a handoff (store,
// poll) of about 0.5 us and three row updates of 22 instructions per point.  Slots are dealt
// out 32 to a wave, over as many workgroups as are free (k_pgs_solve), so that a visit holds up
// few others.
//
// Residual checks run one sweep behind: after s sweeps (a check point) a slot's residual needs
// its bodies' velocities after the sweep, which their first visits of the next sweep have in
// their inboxes; the pair reads them there, stores its residual, and goes on with its next
// visit while the other waves still arrive.  The visit keeps the impulses it replaces, so that
// when the check says stop, the one visit run ahead is taken back.  A pair passes a check point
// only after the check before it has been decided, so at most one visit is ever ahead, and an
// inbox is never overwritten before every reader of its velocity has passed (the body's next
// round of visits includes the reader's own).
//
// Islands of more than 256 manifolds solved on their own run here too, in as many rounds as they
// need (wide_pieces): each checks and stops for itself after every sweep.  With the rows read
// from memory by one workgroup an island of 1880 manifolds took 41 us per sweep, here 14.9.
// A pile of 19.1k manifolds in 18 colours: 44.5 us per sweep in k_pgs_own -> 21.8 us; with a check
// after every sweep 66 -> 28.9 us.  Fewer slots per wave (8 or 16, so that a visit holds up fewer
// others) change the first by less than 2 % and cost up to 5 % in arrivals; polling harder (no
// sleep, a tight loop, two polls in flight) gains nothing or loses.
__device__ __forceinline__ u32x4_t flow_quad(const uint64_t* inbox, uint32_t byte) {
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint64_t*>(inbox), 0, FLOW_INBOX_BYTES, 0x00020000);
    // aux: sc0 | sc1, as vin_quad
    return __builtin_amdgcn_raw_buffer_load_b128(rs, (int)byte, 0, 1 | 16);
}
//
// M: the slots of the large islands, wide: the pieces of the others, G: the workgroups that take
// part (this one does).
struct FlowLds {
    uint32_t arrived, above, max;
};
template <bool CHECKS>
__device__ __forceinline__ void flow_part(const Bodies& B, const StepParams& sp, const SolverRows& R, Counters* cnt,
                                          uint32_t cap, uint32_t nsweeps, uint32_t spin_limit,
                                          const uint64_t* __restrict__ bmask, const uint2* __restrict__ list,
                                          const SweepStop& stop, uint32_t M, uint32_t wide, uint32_t G, FlowLds& L) {
    uint32_t &s_arrived = L.arrived, &s_above = L.above, &s_max = L.max;
    const uint32_t C = G * FLOW_WAVES;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    // Piece v is slots 32 v on of the large islands, or, from piece nl on, 32 slots of an island
    // of the work list.  Wave w works on pieces w, w + C, ... in turn (C: the waves of the grid;
    // the large islands are in the first round).  An island's pieces wait only for each other,
    // and every wave comes to them through pieces of earlier islands, so none waits for ever.
    // Neighbouring waves (the same colour) lie on different CUs.
    const uint32_t nl = (M + FLOW_WAVE_SLOTS - 1u) / FLOW_WAVE_SLOTS, nw = nl + wide;
    const uint32_t wid = wave * G + blockIdx.x;
    const uint32_t wg_waves = blockIdx.x < nl ? (nl - blockIdx.x + G - 1u) / G : 0u;  // with slots of the large islands
    if (threadIdx.x == 0u) s_arrived = s_above = s_max = 0u;
    __syncthreads();
    for (uint32_t v = wid; v < nw; v += C) {
    // opaque per round, so that no row address is kept in registers through a solve for the next
    asm volatile("" : "+s"(cap));
    const bool island = v >= nl;
    uint32_t groups = min(G, nl), s0 = v * FLOW_WAVE_SLOTS, s1 = M;
    unsigned long long* arrive = nullptr;  // an island's arrivals: two words, of the odd and the even check points
    if (island) {
        uint32_t j = v - nl;
        for (uint32_t i0 = 0; i0 < cnt->isl_n[0]; i0 += 64u) {
            const uint2 e = i0 + lane < cnt->isl_n[0] ? list[i0 + lane] : make_uint2(0u, 0u);
            const uint32_t w = (e.y + FLOW_WAVE_SLOTS - 1u) / FLOW_WAVE_SLOTS;
            uint32_t inc = w;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t x = (uint32_t)__shfl_up((int)inc, o, 64);
                if (lane >= (uint32_t)o) inc += x;
            }
            const uint64_t past = __ballot(j < inc);
            if (past != 0ull) {
                const int l = __ffsll((unsigned long long)past) - 1;
                groups = (uint32_t)__shfl((int)w, l, 64);
                s0 = (uint32_t)__shfl((int)e.x, l, 64);
                s1 = s0 + (uint32_t)__shfl((int)e.y, l, 64);
                s0 += (j - ((uint32_t)__shfl((int)inc, l, 64) - groups)) * FLOW_WAVE_SLOTS;
                arrive = stop.isl_arrive + (size_t)(i0 + (uint32_t)l) * ISL_ARRIVE_WORDS;
                break;
            }
            j -= (uint32_t)__shfl((int)inc, 63, 64);
        }
    }
    const uint32_t pair = lane >> 1, s = s0 + pair;
    const bool odd = (lane & 1u) != 0u, active = s < s1;
    // an island checks after every sweep
    const uint32_t every = CHECKS ? (island ? 1u : max(stop.every, 1u)) : nsweeps;
    const float keep = sp.keep, tol = stop.tol;
    uint32_t* err = &cnt->sticky;

    // ---- the slot: rows, impulses, this side's body
    HalfPoint P[4];
    float ln[4], l1[4], l2[4], pn[4], p1[4], p2[4];  // impulses, and those before the last visit
    HalfBody X;
    X.v = X.w = f3{0.0f, 0.0f, 0.0f};
    X.im = 0.0f;
    HalfBody F = X;  // the body's velocity at the last check point (or after the last sweep)
    uint32_t np = 0, body = 0, deg = 0, rank = 0, own = 0, from = 0, to = 0;
    bool dyn = false;
    if (active) {
        const uint4 h = R.hdr[s];
        const uint2 dp = R.dep[s], nx = R.next[s];
        const bool plane = (h.y & PLANE_BIT) != 0u;
        const uint32_t d = odd ? dp.y : dp.x;
        np = min(h.z, 4u);
        body = odd ? h.y : h.x;
        dyn = d != UNSET;
        if (!(odd && plane)) {
            const float4 v = B.sv[body];
            X.im = v.w;
            if (!dyn) {
                X.v = xyz(v);
                X.w = xyz(B.sw[body]);
            }
        }
        if (dyn) {
            deg = d >> 8;
            rank = d & 0xFFu;
            own = (s << 1 | (odd ? 1u : 0u)) * 32u;  // bytes: four words per side
            from = first_visit(B, bmask, body) * 32u;
            to = (odd ? nx.y : nx.x) * 32u;
        }
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
            if (k < np) {
                half_rows(R, s, cap, k, odd, plane, P[k]);
                const float4 L = R.lam[(size_t)k * cap + s];
                ln[k] = L.x;
                l1[k] = L.y;
                l2[k] = L.z;
            }
    }
    F = X;
    // a check's velocities are the next visit's inputs when both sides visit first
    const bool first_both = (rank | (uint32_t)__shfl_xor((int)rank, 1, 64)) == 0u;
    uint32_t k = 0;                        // this pair's sweeps done
    uint32_t ver = 0;                      // its body's visits in them
    uint32_t cp = min(every, nsweeps);     // its next check point (the end without checks)
    uint32_t need = 0;                     // the check point before it, which must be decided first
    bool fin = false;                      // it waits at check point cp (else for its inputs of visit k)
    bool live = active;
    float res = 0.0f;                      // its residual at the last check point
    uint32_t arrived = 0;                  // the last check point this wave arrived at
    uint32_t decided = 0;                  // the last check point known not to stop
    uint32_t stop_at = UNSET;
    uint32_t spins = 0;
    // The wait gives up after spin_limit without progress, its own or (a wave may wait for those that
    // still work on earlier pieces) any other wave's: a wave that got on since it last looked stores
    // the clock, one that did not looks whether another has.
    uint64_t t_last = wall_clock64();
    const uint64_t t_limit = (uint64_t)spin_limit * 100ull;  // wall clock: 100 MHz
    uint32_t beat = 0;
    bool moved = false;
    auto stalled = [&]() -> bool {
        const uint64_t now = wall_clock64();
        if (moved) {
            moved = false;
            t_last = now;
            if (lane == 0u)
                __hip_atomic_store(&cnt->flow_beat, (uint32_t)now, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
        const uint32_t b = __hip_atomic_load(&cnt->flow_beat, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (b != beat) {
            beat = b;
            t_last = now;
            return false;
        }
        return now - t_last > t_limit;
    };
    bool failed = false;
    // Whether all have arrived at check point c; then whether one is above the tolerance.  The
    // large islands count in words of their own per check point, an island in two words for
    // good (arrivals low, above the tolerance high): nobody reaches the check point after next
    // before every wave has seen this one decided.
    uint32_t above_seen[2] = {0u, 0u};
    auto arrivals = [&](uint32_t c, bool& above) -> bool {
        if (island) {
            const unsigned long long v =
                __hip_atomic_load(arrive + (c & 1u) * (ISL_ARRIVE_WORDS / 2u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((uint32_t)v < ((c + 1u) / 2u) * groups) return false;
            const uint32_t n = (uint32_t)(v >> 32), seen = (c & 1u) ? above_seen[1] : above_seen[0];
            above = n != seen;
            if (c & 1u) above_seen[1] = n;
            else above_seen[0] = n;
            return true;
        }
        uint32_t* arr = stop.arrive + (size_t)(c - 1u) * CHECK_ROWS * CHECK_ROW_WORDS;
        uint32_t seen = 0;
        if (lane < CHECK_ROWS)
            seen = __hip_atomic_load(arr + lane * CHECK_ROW_WORDS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (uint32_t o = CHECK_ROWS / 2u; o >= 1u; o >>= 1) seen += (uint32_t)__shfl_xor((int)seen, (int)o, 64);
        seen = (uint32_t)__builtin_amdgcn_readfirstlane((int)seen);
        above = seen >= CHECK_ABOVE;
        return (seen & (CHECK_ABOVE - 1u)) >= groups;
    };
    for (;;) {
        bool ok = live && need <= decided;
        if (ok && dyn) {
            const uint32_t at = fin ? from : own, want = (fin ? ver : ver + rank) & 0xFFFFu;
            const u32x4_t a = flow_quad(R.inbox, at), b = flow_quad(R.inbox, at + 16u);
            ok = (((a[1] >> 16) ^ want) | ((a[3] >> 16) ^ want) | ((b[1] >> 16) ^ want) | ((b[3] >> 16) ^ want)) == 0u;
            // X counts only in the pass in which every version matches
            vunpack4(make_uint2(a[0], a[1]), make_uint2(a[2], a[3]), make_uint2(b[0], b[1]), make_uint2(b[2], b[3]), X.v,
                     X.w);
        }
        const uint64_t oks = __ballot(ok);
        const uint64_t got = oks & (((oks >> 1) & 0x5555555555555555ull) | ((oks << 1) & 0xAAAAAAAAAAAAAAAAull));
        ok = ((got >> lane) & 1ull) != 0ull;
        bool passed = false, ahead = false;
        if (ok) {
            passed = fin;
            if (fin) {
                F = X;
                fin = false;
                live = k < nsweeps;
            }
            if (live && (!passed || first_both)) {
                ahead = true;
                if (CHECKS) {
#pragma unroll
                    for (uint32_t q = 0; q < 4; ++q) {
                        pn[q] = ln[q];
                        p1[q] = l1[q];
                        p2[q] = l2[q];
                    }
                }
                if (k == 0u) {
#pragma unroll
                    for (uint32_t q = 0; q < 4; ++q) {
                        if (q >= np) break;
                        half_apply(P[q].n, ln[q], X);
                        half_apply(P[q].t1, l1[q], X);
                        half_apply(P[q].t2, l2[q], X);
                    }
                }
#pragma unroll
                for (uint32_t q = 0; q < 4; ++q) {
                    if (q >= np) break;
                    half_friction(P[q].t1, P[q].mT1, P[q].maxf, keep, l1[q], X);
                    half_friction(P[q].t2, P[q].mT2, P[q].maxf, keep, l2[q], X);
                }
#pragma unroll
                for (uint32_t q = 0; q < 4; ++q) {
                    if (q >= np) break;
                    half_normal(P[q].n, P[q].mN, P[q].tg, keep, ln[q], X);
                }
                if (dyn) {
                    uint64_t o[4];
                    vpack4(X.v, X.w, ver + rank + 1u, o);
                    const __amdgpu_buffer_rsrc_t rs =
                        __builtin_amdgcn_make_buffer_rsrc(R.inbox, 0, FLOW_INBOX_BYTES, 0x00020000);
                    const u32x4_t q0 = {(uint32_t)o[0], (uint32_t)(o[0] >> 32), (uint32_t)o[1], (uint32_t)(o[1] >> 32)};
                    const u32x4_t q1 = {(uint32_t)o[2], (uint32_t)(o[2] >> 32), (uint32_t)o[3], (uint32_t)(o[3] >> 32)};
                    // aux: sc1, as vin_store
                    __builtin_amdgcn_raw_buffer_store_b128(q0, rs, (int)to, 0, 16);
                    __builtin_amdgcn_raw_buffer_store_b128(q1, rs, (int)(to + 16u), 0, 16);
                }
                if (k == cp) {  // the visit goes past a check point
                    need = cp;
                    cp = min(cp + every, nsweeps);
                }
                ++k;
                ver += deg;
                fin = k == cp;
            }
            // the residual at the check point, after the visit that others wait for (its impulses
            // are those before that visit)
            if ((CHECKS || island) && passed) {
                res = 0.0f;
#pragma unroll
                for (uint32_t q = 0; q < 4; ++q) {
                    if (q >= np) break;
                    const float e = half_residual(P[q], keep, F, ahead ? pn[q] : ln[q], ahead ? p1[q] : l1[q],
                                                  ahead ? p2[q] : l2[q]);
                    if (e > res) res = e;
                }
            }
        }
        // ---- the wave: arrival at a check point once all its pairs have passed it (no pair is
        // further than the next one), decisions, the end
        if (CHECKS) {
            if (__ballot(passed) != 0ull) {
                const uint32_t next = min(arrived + every, nsweeps);
                // a pair short of the check point has yet to reach it or waits there
                if (__ballot(active && (k < next || (k == next && fin))) == 0ull) {
                    arrived = next;
                    uint32_t bits = active ? __float_as_uint(res) : 0u;
                    for (int o = 32; o >= 1; o >>= 1) bits = max(bits, (uint32_t)__shfl_xor((int)bits, o, 64));
                    if (lane == 0u && island) {
                        const bool up = !(__uint_as_float(bits) <= tol);
                        __hip_atomic_fetch_add(arrive + (next & 1u) * (ISL_ARRIVE_WORDS / 2u), up ? (1ull << 32) + 1ull : 1ull,
                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    } else if (lane == 0u) {
                        // the last wave of the workgroup to arrive sends all; the words are free again
                        // before any wave can reach the next check point (it needs this one decided)
                        atomicMax(&s_max, bits);
                        if (__uint_as_float(bits) > tol) atomicOr(&s_above, 1u);
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                        const uint32_t n = atomicAdd(&s_arrived, 1u);
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                        if (n == wg_waves - 1u) {
                            const uint32_t mx = s_max, ab = s_above;
                            s_max = s_above = s_arrived = 0u;
                            // a wave that sees this arrival finds the words cleared
                            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                            atomicMax(stop.bits + next - 1u, mx);
                            __hip_atomic_fetch_add(
                                stop.arrive + ((size_t)(next - 1u) * CHECK_ROWS + blockIdx.x % CHECK_ROWS) * CHECK_ROW_WORDS,
                                1u + (ab ? CHECK_ABOVE : 0u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        }
                    }
                }
            }
            // the outstanding decision, when a pair waits for it or no pair got on (the inputs of a
            // visit past the check point never come when the check stops the others)
            if (decided < arrived && (got == 0ull || __ballot(live && need > decided) != 0ull)) {
                bool above;
                const uint32_t c = min(decided + every, nsweeps);
                if (arrivals(c, above)) {
                    if (!above) {
                        stop_at = c;
                        break;
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");  // the arrival words in LDS
                    decided = c;
                }
            }
        }
        if (got != 0ull) {
            if (__ballot(live) == 0ull) break;
            moved = true;
            continue;
        }
        __builtin_amdgcn_s_sleep(1);
        if ((++spins & 255u) == 0u) {
            if (stalled()) {
                if (lane == 0u) atomicOr(err, STICKY_TIMEOUT);
                failed = true;
                break;
            }
            if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) {
                failed = true;  // another wave gave up
                break;
            }
        }
    }
    if (failed) return;
    // the step's sweeps and whether they met the tolerance
    if (CHECKS && v == 0u && !island) {
        bool hit = stop_at != UNSET;
        if (!hit) {
            bool above = true, all = false;
            t_last = wall_clock64();
            while (!(all = arrivals(nsweeps, above))) {
                if ((++spins & 255u) == 0u && stalled()) break;
                __builtin_amdgcn_s_sleep(1);
            }
            if (!all) {
                if (lane == 0u) atomicOr(err, STICKY_TIMEOUT);
                return;
            }
            hit = !above;
        }
        if (lane == 0u) {
            __hip_atomic_store(&cnt->sweeps_run, stop_at != UNSET ? stop_at : nsweeps, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&cnt->tol_hit, hit ? 1u : 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (island) {
        IslandAcc acc = {0u, 0u, 0u, 0u, 0ull};
        if (active && !odd) acc.add(stop_at != UNSET ? stop_at : nsweeps, res, CHECKS && !(res <= tol), np);
        island_flush(cnt, acc, false);
    }
    if (!active) continue;
    const bool back = CHECKS && stop_at != UNSET && k > stop_at;  // a visit ran ahead of the stop
    if (!odd) {
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q)
            if (q < np)
                R.lam[(size_t)q * cap + s] =
                    make_float4(back ? pn[q] : ln[q], back ? p1[q] : l1[q], back ? p2[q] : l2[q], 0.0f);
    }
    if (dyn && rank == 0u) {
        B.sv[body] = f4(F.v, X.im);
        B.sw[body] = f4(F.w, 0.0f);
    }
    }
}
// Both: the large islands by the first workgroups, the others by the rest, and by the first
// when they are done (parts: 1 the large islands, 2 the others, 3 both at once).  Neither fills
// the chip for its whole length: the sweeps of the large islands are one chain, and the others end
// in a tail of the slowest.  One after the other and at once: 100000 bodies (20 sweeps, 21k slots
// in large islands and 55k in others) 585 -> 471 us, 256 worlds at 1e-4 2050 -> 1170.
template <bool CHECKS>
__global__ void __launch_bounds__(FLOW_THREADS, 2)
k_pgs_solve(Bodies B, StepParams sp, SolverRows R, Counters* cnt, uint32_t cap, uint32_t nsweeps, uint32_t spin_limit,
            const uint64_t* __restrict__ bmask, const uint2* __restrict__ list, const uint32_t* __restrict__ skey,
            float tol, uint32_t parts, uint32_t wide_on, SweepStop stop) {
    static_assert(FLOW_THREADS == ISL_THREADS, "one launch shape");
    extern __shared__ __align__(16) unsigned char isl_lds[];
    if (cnt->sticky != 0u || nsweeps == 0u) return;
    const uint32_t G = gridDim.x;
    const uint32_t wide = list && wide_on ? wide_pieces(cnt, G) : 0u;
    uint32_t flows = 0;  // workgroups that sweep the large islands
    if ((parts & 1u) && cnt->max_colour <= 64u) {
        const uint32_t M = cnt->m_glob <= flow_slots(G) ? cnt->m_glob : 0u;  // more: k_pgs_own
        const uint32_t nw = (M + FLOW_WAVE_SLOTS - 1u) / FLOW_WAVE_SLOTS + wide;
        // as thinly as the chip allows (a visit's wave holds up the others of its SIMD: 19.1k slots
        // on 75 workgroups take 24 us per sweep, on 256 21), but with a workgroup left for every 490
        // slots of the other islands, which take about as long then (a slot costs a workgroup 42
        // ns per sweep, a sweep of the large islands is 20 us)
        const uint32_t other = min(cnt->m_eff, cap) - min(min(cnt->m_eff, cap), M + wide * FLOW_WAVE_SLOTS);
        const uint32_t least = (nw + FLOW_WAVES - 1u) / FLOW_WAVES;
        flows = min(min(G, nw), max(least, G - min(G, (parts & 2u) ? (other + 489u) / 490u : 0u)));
        if (blockIdx.x < flows)
            flow_part<CHECKS>(B, sp, R, cnt, cap, nsweeps, spin_limit, bmask, list, stop, M, wide, flows,
                              *reinterpret_cast<FlowLds*>(isl_lds));
    }
    if (!(parts & 2u)) return;
    if (blockIdx.x < flows) {
        // every wave is done with its pieces; a sweep that gave up ends the launch here
        uint32_t* bad = reinterpret_cast<uint32_t*>(isl_lds);
        __syncthreads();
        if (threadIdx.x == 0u) *bad = __hip_atomic_load(&cnt->sticky, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*bad != 0u) return;
        __syncthreads();
    }
    islands_part(B, sp, R, cnt, cap, list, skey, tol, nsweeps, bmask, wide != 0u, flows, isl_lds);
}
// Allows the solve launch its LDS and returns how many of its workgroups fit on one CU (0 on error).
int pgs_solve_setup() {
    int nb = 0;
    if (hipFuncSetAttribute((const void*)k_pgs_solve<true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)ISL_LDS_BYTES) != hipSuccess ||
        hipFuncSetAttribute((const void*)k_pgs_solve<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)ISL_LDS_BYTES) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_pgs_solve<true>, FLOW_THREADS, ISL_LDS_BYTES) != hipSuccess)
        return 0;
    return nb;
}

// Previous-step lookup table for the warm start: (a, b) -> slot.
// Each entry's table position goes to pos[slot], so that the next build of this table
// clears only the entries it holds (cache_m of them) instead of the whole table.
__device__ __forceinline__ void cache_build_part(const SolverRows& R, Counters* cnt, const CacheTable& C,
                                                 uint32_t gid, uint32_t gsz) {
    uint64_t* __restrict__ key = C.key;
    uint32_t* __restrict__ slot = C.slot;
    uint32_t* __restrict__ np_out = C.np_out;
    uint32_t* __restrict__ pos = C.pos;
    const uint32_t mask = C.mask;
    const uint32_t M = cnt->m_eff;
    if (gid == 0) cnt->cache_m[C.set] = M;
    for (uint32_t s = gid; s < M; s += gsz) {
        np_out[s] = R.hdr[s].z;
        const uint4 h = R.hdr[s];
        const uint64_t k = ((uint64_t)h.x << 32) | h.y;
        uint32_t q = (uint32_t)mix64(k) & mask;
        bool placed = false;
        for (uint32_t probe = 0; probe <= mask && !placed; ++probe) {
            const unsigned long long prev =
                atomicCAS((unsigned long long*)&key[q], (unsigned long long)EMPTY_KEY, (unsigned long long)k);
            if (prev == EMPTY_KEY || prev == k) {
                slot[q] = s;
                pos[s] = q;
                placed = true;
            }
            q = (q + 1) & mask;
        }
        if (!placed) atomicOr(&cnt->sticky, STICKY_INTERNAL);  // table full: never expected (sized >= 2x the slots)
    }
}
__global__ void __launch_bounds__(256) k_cache_build(const SolverRows R, Counters* cnt, CacheTable C) {
    if (cnt->sticky != 0u) return;
    cache_build_part(R, cnt, C, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

// Moves the entries of an (a, b) -> slot table into a larger empty one.
__global__ void __launch_bounds__(256) k_cache_rehash(const uint64_t* __restrict__ okey,
                                                      const uint32_t* __restrict__ oslot, uint32_t on,
                                                      uint64_t* __restrict__ key, uint32_t* __restrict__ slot,
                                                      uint32_t mask, Counters* __restrict__ cnt,
                                                      uint32_t* __restrict__ pos) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= on) return;
    const uint64_t k = okey[i];
    if (k == EMPTY_KEY) return;
    const uint32_t v = oslot[i];
    uint32_t q = (uint32_t)mix64(k) & mask;
    for (uint32_t probe = 0; probe <= mask; ++probe) {
        const unsigned long long prev =
            atomicCAS((unsigned long long*)&key[q], (unsigned long long)EMPTY_KEY, (unsigned long long)k);
        if (prev == EMPTY_KEY || prev == k) {
            slot[q] = v;
            pos[v] = q;
            return;
        }
        q = (q + 1) & mask;
    }
    atomicOr(&cnt->sticky, STICKY_INTERNAL);
}



// Clears the per-step part of the control block and the meeting words.
__global__ void k_counters_begin(Counters* cnt, uint32_t* __restrict__ kinds, Meeting meet) {
    counters_reset(cnt, kinds, meet);
}

// Integration is skipped while any sticky error is set, so an overflowing step
// leaves the state exactly as it was.
__global__ void __launch_bounds__(256) k_integrate(Bodies B, StepParams sp, uint32_t n, Counters* cnt,
                                                   uint32_t sweeps, SolverRows R, CacheTable C) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (cnt->sticky != 0u) return;
    // the step's (a, b) -> slot table for the next step's warm start, in the same launch
    if (C.key) cache_build_part(R, cnt, C, i, gridDim.x * blockDim.x);
    if (i == 0) {
        cnt->steps_done += 1u;
        // sweeps of the large islands, and of the step (the most any island ran)
        const uint32_t swg = sweeps == SWEEPS_ON_DEVICE ? cnt->sweeps_run : sweeps;
        const uint32_t sw = max(swg, cnt->loc_sweeps);
        cnt->pgs_bytes_total += spread_sum(cnt, &SpreadRow::pgs_bytes) * (unsigned long long)sw;
        cnt->sweeps_total += sw;
        cnt->bundle_point_sweeps_total += cnt->bundle_point_sweeps;
        cnt->acc_steps += 1u;
        cnt->acc_reached += cnt->tol_hit != 0u && cnt->loc_miss == 0u ? 1u : 0u;
        cnt->acc_max_sweeps = max(cnt->acc_max_sweeps, sw);
        cnt->acc_sweeps += sw;
        cnt->acc_contact_sweeps +=
            (unsigned long long)(spread_sum(cnt, &SpreadRow::contacts) - cnt->loc_points) * swg + cnt->loc_point_sweeps;
        cnt->acc_local_contact_sweeps += cnt->loc_point_sweeps;
        cnt->acc_gjk_fail += cnt->gjk_fail;
        cnt->acc_epa_fail += cnt->epa_fail;
    }
    if (i >= n) return;
    const float4 v4 = B.sv[i];
    if (!(v4.w > 0.0f) && !(B.bfl[i].x & BODY_KINEMATIC)) return;
    const float4 w4 = B.sw[i];
    const float4 x4 = B.x[i];
    const float4 qv = B.q[i];
    const f3 v = xyz(v4), w = xyz(w4);
    const f3 x = xyz(x4) + v * sp.dt;
    const float hdt = 0.5f * sp.dt;
    const q4 q = {qv.x, qv.y, qv.z, qv.w};
    const q4 dq = qmul(q4{w.x, w.y, w.z, 0.0f}, q);
    const q4 nq = {q.x + dq.x * hdt, q.y + dq.y * hdt, q.z + dq.z * hdt, q.w + dq.w * hdt};
    const float len = sqrtf(nq.x * nq.x + nq.y * nq.y + nq.z * nq.z + nq.w * nq.w);
    const float inv = 1.0f / len;
    B.x[i] = make_float4(x.x, x.y, x.z, x4.w);
    B.q[i] = make_float4(nq.x * inv, nq.y * inv, nq.z * inv, nq.w * inv);
    B.vel[i] = v4;
    B.angv[i] = make_float4(w.x, w.y, w.z, 0.0f);
}

// ---------------------------------------------------------------- islands and sleeping
// Union-find over the step's manifolds between two awake dynamic bodies (uf_find).
__global__ void __launch_bounds__(256) k_isl_union(Bodies B, const uint2* __restrict__ m_ab, uint32_t cap,
                                                   uint32_t n, const Counters* __restrict__ cnt) {
    if (cnt->sticky != 0u) return;
    const uint32_t M = min(cap, cnt->m_eff);
    const uint32_t stamp = cnt->steps_done + 1u;  // runs before the integration counts this step
    for (uint32_t m = blockIdx.x * blockDim.x + threadIdx.x; m < M; m += gridDim.x * blockDim.x) {
        const uint2 ab = m_ab[m];
        if (ab.y & PLANE_BIT) continue;
        const bool da = B.sv[ab.x].w > 0.0f, db = B.sv[ab.y].w > 0.0f;
        if (da && db) {
            uint32_t ra = uf_find(B.upar, ab.x), rb = uf_find(B.upar, ab.y);
            while (ra != rb) {
                if (ra < rb) {
                    const uint32_t old = atomicCAS(B.upar + rb, rb, ra);
                    if (old == rb) break;
                    rb = uf_find(B.upar, old);
                } else {
                    const uint32_t old = atomicCAS(B.upar + ra, ra, rb);
                    if (old == ra) break;
                    ra = uf_find(B.upar, old);
                }
            }
        } else if (da || db) {
            // an awake dynamic body touches a sleeping one: its island wakes at the next step
            const uint32_t o = da ? ab.y : ab.x;
            const uint32_t y = B.slp[o].y;
            if ((y & ASLEEP_BIT) && (y & LABEL_MASK) < n) B.wake[y & LABEL_MASK] = stamp;
        }
    }
}
// The same by one workgroup with the parents in LDS, for worlds whose bodies fit: a step of a
// walk is an LDS access instead of a coherent load from memory, which other workgroups'
// links keep contended (19000 manifolds of 6000 bodies: 93 us, so 27; 1000 bodies: 11, so 5).
// Above the limit the one workgroup could not hold them; 100000 bodies take 130 us by
// k_isl_union.  The parents written back are the roots themselves.
constexpr uint32_t UNION_LDS_BODIES = 36864u;
constexpr int UNION_THREADS = 1024;
__device__ __forceinline__ uint32_t lds_find(uint32_t* par, uint32_t x) {
    auto ld = [par](uint32_t k) { return __hip_atomic_load(par + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
    uint32_t cur = ld(x);
    if (cur != x) {
        uint32_t prev = x, next;
        while (cur > (next = ld(cur))) {
            __hip_atomic_store(par + prev, next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            prev = cur;
            cur = next;
        }
    }
    return cur;
}
__global__ void __launch_bounds__(UNION_THREADS) k_isl_union_lds(Bodies B, const uint2* __restrict__ m_ab, uint32_t cap,
                                                                 uint32_t n, const Counters* __restrict__ cnt) {
    extern __shared__ uint32_t par[];
    if (cnt->sticky != 0u) return;
    const uint32_t M = min(cap, cnt->m_eff);
    const uint32_t stamp = cnt->steps_done + 1u;
    for (uint32_t i = threadIdx.x; i < n; i += UNION_THREADS) par[i] = B.sv[i].w > 0.0f ? i : UNSET;
    __syncthreads();
    auto edges = [&](auto&& link) {
        constexpr int U = 4;  // manifolds of a thread on the way at a time
        for (uint32_t m0 = threadIdx.x; m0 < M; m0 += U * UNION_THREADS) {
            uint2 e[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
                e[u] = m0 + u * UNION_THREADS < M ? m_ab[m0 + u * UNION_THREADS] : make_uint2(0u, PLANE_BIT);
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (!(e[u].y & PLANE_BIT)) link(e[u].x, e[u].y);
        }
    };
    // each body's first link is to the smallest it touches, without a walk: most of the manifolds
    // then find one root from both sides
    edges([&](uint32_t a, uint32_t b) {
        const bool da = par[a] != UNSET, db = par[b] != UNSET;  // never changes
        if (da && db) {
            atomicMin(par + max(a, b), min(a, b));
        } else if (da || db) {
            const uint32_t y = B.slp[da ? b : a].y;
            if ((y & ASLEEP_BIT) && (y & LABEL_MASK) < n) B.wake[y & LABEL_MASK] = stamp;
        }
    });
    __syncthreads();
    edges([&](uint32_t a, uint32_t b) {
        if (par[a] == UNSET || par[b] == UNSET) return;
        uint32_t ra = lds_find(par, a), rb = lds_find(par, b);
        while (ra != rb) {
            const uint32_t hi = max(ra, rb), lo = min(ra, rb);
            const uint32_t old = atomicCAS(par + hi, hi, lo);
            if (old == hi) break;
            ra = lds_find(par, old);
            rb = lo;
        }
    });
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += UNION_THREADS)
        if (par[i] != UNSET) B.upar[i] = lds_find(par, i);
}
int isl_union_setup() {
    return hipFuncSetAttribute((const void*)k_isl_union_lds, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)(4u * UNION_LDS_BODIES)) == hipSuccess ? 1 : 0;
}
// Labels, rest times and each island's smallest rest time; counts islands and sleeping bodies.
__global__ void __launch_bounds__(256) k_isl_label(Bodies B, StepParams sp, uint32_t n, Counters* cnt) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (cnt->sticky != 0u) return;
    uint32_t isl = 0, slp = 0;
    // each island's least rest time (rest times are >= 0: bit order = value order)
    struct Min {
        uint32_t* imin;
        __device__ uint32_t combine(uint32_t a, uint32_t b) const { return a < b ? a : b; }
        __device__ void apply(uint32_t r, uint32_t c) const { atomicMin(imin + r, c); }
    };
    const bool dyn = i < n && B.sv[i].w > 0.0f;
    uint32_t r = UNSET, tb = 0u;
    if (dyn) {
        r = uf_root(B.upar, i);
        const float4 v = B.vel[i], w = B.angv[i];
        const bool still = v.x * v.x + v.y * v.y + v.z * v.z < sp.sleep_lin2 &&
                           w.x * w.x + w.y * w.y + w.z * w.z < sp.sleep_ang2;
        const float t = still ? __uint_as_float(B.slp[i].x) + sp.dt : 0.0f;
        B.slp[i] = make_uint2(__float_as_uint(t), r);
        tb = __float_as_uint(t);
        isl = r == i ? 1u : 0u;
    }
    wave_by_island(dyn, r, tb, 0xFFFFFFFFu, Min{B.imin});
    if (i >= n) return;
    if (!dyn && B.vel[i].w > 0.0f) {
        // asleep (a static body has no inverse mass)
        const uint32_t y = B.slp[i].y;
        isl = (y & LABEL_MASK) == i ? 1u : 0u;
        slp = 1u;
    }
    const uint32_t row = (blockIdx.x * 4u + (threadIdx.x >> 6)) % SPREAD;
    const uint32_t wi = __popcll(__ballot(isl != 0u)), ws = __popcll(__ballot(slp != 0u));
    if ((threadIdx.x & 63u) == 0u) {
        if (wi) atomicAdd(&cnt->sp[row].islands, wi);
        if (ws) atomicAdd(&cnt->sp[row].sleeping, ws);
    }
}
// Islands whose bodies have all rested sleep_time seconds fall asleep.
__global__ void __launch_bounds__(256) k_isl_sleep(Bodies B, StepParams sp, uint32_t n, Counters* cnt) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (cnt->sticky != 0u || i >= n) return;
    bool now = false;
    if (sp.allow_sleep && B.sv[i].w > 0.0f) {
        const uint2 sl = B.slp[i];
        if (B.imin[sl.y] >= __float_as_uint(sp.sleep_time)) {
            B.slp[i] = make_uint2(sl.x, sl.y | ASLEEP_BIT);
            B.vel[i] = make_float4(0.0f, 0.0f, 0.0f, B.vel[i].w);
            B.angv[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            now = true;
        }
    }
    const uint32_t row = (blockIdx.x * 4u + (threadIdx.x >> 6)) % SPREAD;
    const uint32_t ws = __popcll(__ballot(now));
    if ((threadIdx.x & 63u) == 0u && ws) atomicAdd(&cnt->sp[row].sleeping, ws);
}

// ---------------------------------------------------------------- host launchers
static inline dim3 grid_for(uint32_t n, uint32_t b = 256) { return dim3((n + b - 1) / b ? (n + b - 1) / b : 1); }
// Kernels whose element count is read on the device stride over it with at most
// 1024 workgroups, so that a capacity far above the count launches few idle waves.
static inline dim3 grid_bounded(uint32_t cap, uint32_t max_groups = 1024u) {
    const uint32_t b = (cap + 255u) / 256u;
    return dim3(b == 0u ? 1u : (b > max_groups ? max_groups : b));
}


void launch_counters_begin(Counters* cnt, uint32_t* kinds, const Meeting& meet, hipStream_t s) {
    hipLaunchKernelGGL(k_counters_begin, dim3(1), dim3(64), 0, s, cnt, kinds, meet);
}
void launch_begin(const Bodies& B, const StepParams& sp, uint32_t n, uint64_t* key, uint32_t* key32, uint32_t* val,
                  uint64_t* bmax0,
                  uint64_t* bmax1, uint64_t* bmask, uint32_t* bdeg, Counters* cnt, uint32_t* kinds,
                  const Meeting& meet, const CellTable& ct, hipStream_t s) {
    const uint32_t m = std::max(n, ct.mbits ? ct.mlist_n : 0u);
    if (m)
        hipLaunchKernelGGL(k_begin, grid_for(m), dim3(256), 0, s, B, sp, n, key, key32, val, bmax0, bmax1, bmask, bdeg,
                           cnt, kinds, meet, ct);
    else
        launch_counters_begin(cnt, kinds, meet, s);
}
void launch_fill_u64(uint64_t* p, uint64_t v, uint32_t n, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_fill_u64, grid_for(n), dim3(256), 0, s, p, v, n);
}
void launch_fill_u32(uint32_t* p, uint32_t v, uint32_t n, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_fill_u32, grid_for(n), dim3(256), 0, s, p, v, n);
}
void launch_iota(uint32_t* p, uint32_t n, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_iota, grid_for(n), dim3(256), 0, s, p, n);
}
void launch_cell_clear(const CellTable& t, hipStream_t s) {
    if (t.mbits) return;  // k_begin cleared the bitmap words
    const uint32_t n = std::max(t.mask + 1u, (t.bmask >> 5) + 1u);
    hipLaunchKernelGGL(k_cell_clear, grid_for(n), dim3(256), 0, s, t);
}
void launch_cell_table(const Bodies& B, const SortedKeys& skey, const uint32_t* sval, uint32_t n, const CellTable& t,
                       Counters* cnt, uint32_t* scan_tmp, hipStream_t s) {
    if (!n) return;
    hipLaunchKernelGGL(k_cell_table, grid_for(n), dim3(256), 0, s, B, skey, sval, n, t, cnt);
    if (t.mbits) {
        scan_exclusive(t.crank, t.crank, n, scan_tmp, s, nullptr, nullptr, false, &cnt->sticky);
        hipLaunchKernelGGL(k_cell_rank, grid_for(n), dim3(256), 0, s, skey, n, t, cnt);
        return;
    }
    hipLaunchKernelGGL(k_cell_place, grid_for(n), dim3(256), 0, s, skey, n, t, cnt);
}
void launch_pair_count(const Bodies& B, const StepParams& sp, const SortedKeys& skey, const uint32_t* sval,
                       const CellTable& ct, uint32_t n, uint32_t* cnt, uint32_t* bsum, uint32_t* stash, Counters* ctr,
                       hipStream_t s) {
    if (!n) return;
    if (ct.mbits) {
        hipLaunchKernelGGL(k_pair_count<BP_RANK>, grid_for(BP_PARTS * n), dim3(256), 0, s, B, sp, skey, sval, ct, n,
                           cnt, bsum, stash, ctr);
        return;
    }
    hipLaunchKernelGGL(k_pair_count<BP_SPARSE>, grid_for(BP_PARTS * n), dim3(256), 0, s, B, sp, skey, sval, ct, n, cnt,
                       bsum, stash, ctr);
    hipLaunchKernelGGL(k_pair_count_dense, grid_for(BP_PARTS * n), dim3(256), 0, s, B, sp, skey, sval, ct, n, cnt,
                       bsum, stash, ctr);
}
void launch_pair_emit(const Bodies& B, const StepParams& sp, const SortedKeys& skey, const uint32_t* sval,
                      const CellTable& ct, uint32_t n, const uint32_t* pcnt, const uint32_t* boff, uint32_t cap,
                      uint32_t* pa, uint32_t* pb, Counters* cnt, const uint32_t* stash, hipStream_t s) {
    if (!n) return;
    if (ct.mbits) {
        hipLaunchKernelGGL(k_pair_emit<BP_RANK>, grid_for(BP_PARTS * n), dim3(256), 0, s, B, sp, skey, sval, ct, n, pcnt,
                           boff, cap, pa, pb, cnt, stash);
        return;
    }
    hipLaunchKernelGGL(k_pair_emit<BP_SPARSE>, grid_for(BP_PARTS * n), dim3(256), 0, s, B, sp, skey, sval, ct, n, pcnt,
                       boff, cap, pa, pb, cnt, stash);
    hipLaunchKernelGGL(k_pair_emit<BP_DENSE>, grid_for(BP_PARTS * n), dim3(256), 0, s, B, sp, skey, sval, ct, n, pcnt,
                       boff, cap, pa, pb, cnt, stash);
}
void launch_narrow(const Bodies& B, const StepParams& sp, const uint32_t* pa, const uint32_t* pb, uint32_t cap_pairs,
                   uint32_t* p_np, float4* p_pt, float4* p_nf, uint32_t* epa_list, uint32_t* p_kind, uint32_t* kinds,
                   uint32_t* order, uint32_t epa_groups, Counters* cnt, hipStream_t s) {
    // 256 workgroups: each adds its kind counts to the 16 shared counters once per pass
    hipLaunchKernelGGL(k_pair_kind, grid_bounded(cap_pairs, 256u), dim3(256), 0, s, B, pa, pb, p_kind, kinds, cnt);
    hipLaunchKernelGGL(k_pair_order, grid_bounded(cap_pairs, 256u), dim3(256), 0, s, p_kind, kinds, order, cnt);
    hipLaunchKernelGGL(k_narrow<false>, grid_bounded(cap_pairs), dim3(256), 0, s, B, sp, pa, pb, p_np, p_pt, p_nf,
                       epa_list, cnt, order, kinds);
    hipLaunchKernelGGL(k_narrow<true>, grid_bounded(cap_pairs), dim3(256), 0, s, B, sp, pa, pb, p_np, p_pt, p_nf,
                       epa_list, cnt, order, kinds);
    // the deep pairs are few: a fixed grid strides over the queue
    hipLaunchKernelGGL(k_narrow_epa, dim3(epa_groups), dim3(64), 0, s, B, sp, pa, pb, epa_list, cap_pairs, p_np, p_pt,
                       p_nf, cnt);
}
void launch_compact(const uint32_t* pa, const uint32_t* pb, uint32_t cap_pairs, const uint32_t* p_np,
                    const float4* p_pt, const float4* p_nf, const uint32_t* moff, uint32_t cap, uint2* m_ab,
                    uint32_t* m_np, float4* c_pt, float4* c_nf, Counters* cnt, hipStream_t s) {
    hipLaunchKernelGGL(k_compact, grid_bounded(cap_pairs), dim3(256), 0, s, pa, pb, p_np, p_pt, p_nf, moff, cap, m_ab,
                       m_np, c_pt, c_nf, cnt);
}
int colour_blocks_per_cu() {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_colour, 256, 0) != hipSuccess) return 1;
    return nb < 1 ? 1 : nb;
}
static PrevCache make_prev(const PrevCacheArgs& pca) {
    PrevCache pc;
    pc.key = pca.key;
    pc.slot = pca.slot;
    pc.mask = pca.mask;
    pc.lam = pca.lam;
    pc.fid = pca.fid;
    pc.np = pca.np;
    pc.colour = pca.colour;
    pc.cap = pca.cap;
    pc.valid = pca.valid;
    return pc;
}
void launch_colour(const Bodies& B, const uint2* m_ab, uint32_t cap_man, uint32_t* col, uint64_t* prio,
                   uint64_t* bmax0, uint64_t* bmax1, uint64_t* bmask, uint32_t* bdeg, uint32_t* list, GridBar* bar,
                   Counters* cnt, uint32_t blocks, const PrevCacheArgs& prev, uint32_t split, hipStream_t s) {
    constexpr uint32_t SMALL = 16384;  // longest list coloured by one workgroup
    hipLaunchKernelGGL(k_colour_keep, grid_bounded(cap_man), dim3(256), 0, s, B, m_ab, col, prio, bmax0, bmask, bdeg, list,
                       cnt, make_prev(prev), RECOLOUR_PERIOD, split ? cap_man : 0u);
    hipLaunchKernelGGL(k_colour_small, dim3(1), dim3(1024), 0, s, B, m_ab, col, prio, bmax0, bmax1, bmask, list, cnt,
                       65000u, SMALL);
    hipLaunchKernelGGL(k_colour, dim3(blocks), dim3(256), 0, s, B, m_ab, col, prio, bmax0, bmax1, bmask, list, bar,
                       cnt, 65000u, SMALL);
}
void launch_prep(const Bodies& B, const StepParams& sp, const uint32_t* order, uint32_t cap, const uint2* m_ab,
                 const uint32_t* m_np, const float4* c_pt, const float4* c_nf, const SolverRows& R,
                 const PrevCacheArgs& pca, const float4* warm_in, const uint32_t* col, const uint64_t* bmask,
                 const uint32_t* bdeg, Counters* cnt, float* feat, const PrepExtra& X, hipStream_t s) {
    const PrevCache pc = make_prev(pca);
    hipLaunchKernelGGL(k_prep, grid_bounded(cap), dim3(256), 0, s, B, sp, order, cap, m_ab, m_np, c_pt, c_nf, R, pc,
                       warm_in, col, bmask, bdeg, cnt, feat, X);
}

// Learned warm start: the network predicts the correction to the previous
// step's impulse of the same feature (already in the rows, zero for a new
// point) in units of u = mN g dt; lambda = previous + output * u, projected onto
// lambda_n >= 0 and the step's friction box |lambda_t| <= mu B.
__global__ void __launch_bounds__(256) k_mlp_apply(SolverRows R, const Counters* __restrict__ cnt, uint32_t cap,
                                                   const float* __restrict__ Y, StepParams sp) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= cnt->m_eff || cnt->sticky != 0u) return;
    const uint32_t np = R.hdr[s].z;
    const float gdt = MLP_G_REF * sp.dt;
    for (uint32_t k = 0; k < np; ++k) {
        const size_t o = (size_t)k * cap + s;
        const float u = R.J[(size_t)k * JROWS * cap + s].w * gdt;  // mN
        const float* y = Y + ((size_t)4 * s + k) * MLP_OUT;
        const float4 Lp = R.lam[o];
        // a non-finite output leaves the point exactly at its cached impulse (as the plain warm
        // start has it); finite outputs are capped at MLP_Y_MAX units, so any network gives a
        // finite start the sweeps then correct
        if (!(isfinite(y[0]) && isfinite(y[1]) && isfinite(y[2]))) continue;
        auto cap_y = [](float v) { return v < -MLP_Y_MAX ? -MLP_Y_MAX : (v > MLP_Y_MAX ? MLP_Y_MAX : v); };
        const float y0 = cap_y(y[0]), y1 = cap_y(y[1]), y2 = cap_y(y[2]);
        float ln = Lp.x + y0 * u;
        ln = ln > 0.0f ? ln : 0.0f;
        const float maxf = R.J[((size_t)k * JROWS + 8) * cap + s].w;  // the step's friction bound
        float t1 = Lp.y + y1 * u, t2 = Lp.z + y2 * u;
        t1 = t1 < -maxf ? -maxf : (t1 > maxf ? maxf : t1);
        t2 = t2 < -maxf ? -maxf : (t2 > maxf ? maxf : t2);
        const float4 L = make_float4(ln, t1, t2, 0.0f);
        R.lam[o] = L;
        R.lam0[o] = L;
    }
}
void launch_mlp_apply(const SolverRows& R, const Counters* cnt, uint32_t cap, const float* Y, const StepParams& sp,
                      hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_apply, grid_for(cap), dim3(256), 0, s, R, cnt, cap, Y, sp);
}
int pgs_own_setup(uint32_t max_lds_bytes, uint32_t lds_bytes) {
    if (hipFuncSetAttribute((const void*)k_pgs_own, hipFuncAttributeMaxDynamicSharedMemorySize, (int)max_lds_bytes) !=
        hipSuccess)
        return 0;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_pgs_own, OWN_WAVE, lds_bytes) != hipSuccess) return 0;
    return nb;
}
void launch_flow_init(const Bodies& B, const SolverRows& R, uint32_t cap, const uint64_t* bmask, const Counters* cnt,
                      const uint2* list, unsigned long long* isl_arrive, uint32_t cus, hipStream_t s) {
    hipLaunchKernelGGL(k_flow_init, grid_bounded(cap), dim3(256), 0, s, B, R, bmask, cnt, list, isl_arrive, cus);
}
void launch_pgs_solve(const Bodies& B, const StepParams& sp, const SolverRows& R, uint32_t cap, const uint64_t* bmask,
                      uint32_t nsweeps, Counters* cnt, uint32_t spin_limit, uint32_t cus, const uint32_t* skey,
                      const uint2* list, float tol, uint32_t parts, bool wide, const OwnShape& own, const SweepStop& stop,
                      hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
    if (!nsweeps) return;
    if (ev0) (void)hipEventRecord(ev0, s);
    if (stop.bits)
        hipLaunchKernelGGL(k_pgs_solve<true>, dim3(cus), dim3(FLOW_THREADS), ISL_LDS_BYTES, s, B, sp, R, cnt, cap, nsweeps,
                           spin_limit, bmask, list, skey, tol, parts, wide ? 1u : 0u, stop);
    else
        hipLaunchKernelGGL(k_pgs_solve<false>, dim3(cus), dim3(FLOW_THREADS), ISL_LDS_BYTES, s, B, sp, R, cnt, cap, nsweeps,
                           spin_limit, bmask, list, skey, tol, parts, wide ? 1u : 0u, stop);
    if (parts & SOLVE_LARGE)
        hipLaunchKernelGGL(k_pgs_own, dim3(own.groups ? own.groups : 1u), dim3(OWN_WAVE), own.lds_bytes, s, B, sp, R, cnt,
                           cap, nsweeps, flow_slots(cus), own.lds_bytes / (uint32_t)sizeof(float4),
                           spin_limit, own.tune, bmask, stop);
    if (ev1) (void)hipEventRecord(ev1, s);
}
void launch_pgs(const Bodies& B, const StepParams& sp, const SolverRows& R, uint32_t s0, uint32_t s1, uint32_t cap,
                uint32_t first, hipStream_t s) {
    if (s1 > s0) hipLaunchKernelGGL(k_pgs, grid_for(s1 - s0), dim3(256), 0, s, B, sp, R, s0, s1, cap, first);
}
void launch_residual(const Bodies& B, const StepParams& sp, const SolverRows& R, const Counters* cnt, uint32_t cap,
                     uint32_t* out_bits, hipStream_t s) {
    hipLaunchKernelGGL(k_residual, grid_for(cap), dim3(256), 0, s, B, sp, R, cnt, cap, out_bits);
}
// Empties the entries the table holds (the positions its last build recorded).
__global__ void k_cache_clear(uint64_t* __restrict__ key, const uint32_t* __restrict__ pos, const Counters* cnt,
                              uint32_t set) {
    if (cnt->sticky != 0u) return;
    const uint32_t m = cnt->cache_m[set];
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += gridDim.x * blockDim.x) key[pos[i]] = EMPTY_KEY;
}

void launch_cache_build(const SolverRows& R, Counters* cnt, uint32_t cap, uint64_t* key, uint32_t* slot,
                        uint32_t mask, uint32_t* np_out, uint32_t* pos, uint32_t set, hipStream_t s, bool clear) {
    if (clear) hipLaunchKernelGGL(k_cache_clear, grid_bounded(cap), dim3(256), 0, s, key, pos, cnt, set);
    hipLaunchKernelGGL(k_cache_build, grid_bounded(cap), dim3(256), 0, s, R, cnt,
                       CacheTable{key, slot, mask, np_out, pos, set});
}
void launch_cache_rehash(const uint64_t* okey, const uint32_t* oslot, uint32_t on, uint64_t* key, uint32_t* slot,
                         uint32_t mask, Counters* cnt, uint32_t* pos, hipStream_t s) {
    if (on)
        hipLaunchKernelGGL(k_cache_rehash, grid_for(on), dim3(256), 0, s, okey, oslot, on, key, slot, mask, cnt, pos);
}
void launch_integrate(const Bodies& B, const StepParams& sp, uint32_t n, Counters* cnt, uint32_t sweeps,
                      hipStream_t s, const SolverRows* R, const CacheTable* C) {
    const uint32_t g = std::max(n, 1u);
    hipLaunchKernelGGL(k_integrate, grid_for(g), dim3(256), 0, s, B, sp, n, cnt, sweeps, R ? *R : SolverRows{},
                       C ? *C : CacheTable{});
}

void launch_isl_union(const Bodies& B, uint32_t n, const uint2* m_ab, uint32_t cap_man, Counters* cnt,
                      hipStream_t s) {
    if (n == 0u) return;
    if (n <= UNION_LDS_BODIES)
        hipLaunchKernelGGL(k_isl_union_lds, dim3(1), dim3(UNION_THREADS), 4u * n, s, B, m_ab, cap_man, n, cnt);
    else
        hipLaunchKernelGGL(k_isl_union, grid_bounded(cap_man), dim3(256), 0, s, B, m_ab, cap_man, n, cnt);
}
void launch_islands(const Bodies& B, const StepParams& sp, uint32_t n, Counters* cnt, hipStream_t s) {
    if (!n) return;
    hipLaunchKernelGGL(k_isl_label, grid_for(n), dim3(256), 0, s, B, sp, n, cnt);
    hipLaunchKernelGGL(k_isl_sleep, grid_for(n), dim3(256), 0, s, B, sp, n, cnt);
}
}  // namespace axm
