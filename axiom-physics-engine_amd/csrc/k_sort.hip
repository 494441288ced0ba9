// Device-wide exclusive scan and stable LSD radix sort for gfx950 (wave64).
//
// Radix sort: digits of 8 bits with every pass in one launch, or, for more than 131072 keys read
// from memory, of up to 10 bits in three launches a pass (below).
// Scan: one pass, tiles chained by decoupled look-back (below).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "dev_islands.hpp"
#include "launch.hpp"

namespace axm {

constexpr int SC_THREADS = 256;
constexpr int SC_ITEMS = 16;
constexpr int SC_TILE = SC_THREADS * SC_ITEMS;
// workgroups of a scan launch (each takes tiles in turn): enough to keep many tiles in
// flight; fewer when the count is read on the device and usually far below the capacity
constexpr uint32_t SC_MAX_GROUPS = 512, SC_MAX_GROUPS_DEV = 64;

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

// Inclusive wave scan (wave64) of a u32.
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
    const uint32_t lane = lane_id();
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(v, o, 64);
        if (lane >= (uint32_t)o) v += t;
    }
    return v;
}

// Exclusive block scan (blockDim = 256 = 4 waves); returns the block total in `total`.
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t& total) {
    __shared__ uint32_t s_w[SC_THREADS / 64];
    const uint32_t lane = lane_id(), wv = threadIdx.x >> 6;
    const uint32_t inc = wave_incl_scan(v);
    if (lane == 63) s_w[wv] = inc;
    __syncthreads();
    uint32_t base = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < SC_THREADS / 64; ++w) {
        const uint32_t x = s_w[w];
        if ((uint32_t)w < wv) base += x;
        tot += x;
    }
    __syncthreads();
    total = tot;
    return base + inc - v;
}

// Single-pass exclusive scan with decoupled look-back.  Workgroup b starts with
// tile b; when there are more tiles than workgroups, the rest are taken in turn
// from a counter (so every lower tile is already held by a running workgroup).  A
// workgroup publishes its tile total, then reads the status words of the 64 tiles
// below it at once (one per lane of its first wave), moving down 64 at a time until
// it meets an inclusive prefix, and publishes its own.  Status word: bits 62-63
// state (0 none, 1 tile total, 2 inclusive prefix), bits 0-31 the value.  The
// launch is at most a few hundred workgroups, all resident together.  Atomics on
// one address (or line) queue one after another, so the finish count that finds the
// last workgroup is spread over SC_ROWS counters one line apart, each row's last
// arrival adding to one top counter; the last workgroup to finish clears the status
// words it used and the counters, so every call starts from zeros (the scratch is
// zeroed once when allocated).  Scratch layout (u32 words): [0] tile counter,
// [SC_ROW0 + 32 r] row r's finish count, [SC_TOP] rows finished, then from
// SC_STATUS the nb 64-bit status words.
constexpr uint64_t SC_AGG = 1ull << 62, SC_PRE = 2ull << 62;
constexpr uint32_t SC_ROWS = 16, SC_ROW0 = 32, SC_TOP = SC_ROW0 + 32 * SC_ROWS, SC_STATUS = SC_TOP + 32;

// With n_dev the element count is min(n, *n_dev), read on the device (nb, the
// tiles the scratch holds, is sized for n).  With flags, the input is read as
// (in[i] != 0).  `in` may equal `out` (each thread reads its elements before it
// writes them).
__global__ void __launch_bounds__(SC_THREADS) k_scan_1p(const uint32_t* in, uint32_t* out, uint32_t n_cap,
                                                         uint32_t* __restrict__ tmp, uint32_t nb,
                                                         uint32_t* __restrict__ total_out,
                                                         const uint32_t* __restrict__ n_dev, int flags,
                                                         uint32_t* __restrict__ err) {
    __shared__ uint32_t s_tile, s_prefix;
    uint64_t* st = reinterpret_cast<uint64_t*>(tmp + SC_STATUS);
    const uint32_t n = n_dev ? min(n_cap, *n_dev) : n_cap;
    const uint32_t nt = n == 0u ? 1u : (n + SC_TILE - 1u) / SC_TILE;  // tiles with elements (tile 0 always)
    // 16-byte loads and stores when both arrays allow them (whole items of a full tile)
    const bool vec = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0u;
    uint32_t tile = blockIdx.x;
    while (tile < nt) {
        // each thread owns SC_ITEMS consecutive elements of the tile
        const uint32_t base = tile * SC_TILE + threadIdx.x * SC_ITEMS;
        const bool whole = vec && base + SC_ITEMS <= n;
        uint32_t v[SC_ITEMS];
        if (whole) {
            const uint4* p = reinterpret_cast<const uint4*>(in + base);
#pragma unroll
            for (int q = 0; q < SC_ITEMS / 4; ++q) {
                const uint4 x = p[q];
                v[4 * q] = x.x;
                v[4 * q + 1] = x.y;
                v[4 * q + 2] = x.z;
                v[4 * q + 3] = x.w;
            }
        } else {
#pragma unroll
            for (int k = 0; k < SC_ITEMS; ++k) v[k] = base + k < n ? in[base + k] : 0u;
        }
        uint32_t sum = 0;
#pragma unroll
        for (int k = 0; k < SC_ITEMS; ++k) {
            if (flags) v[k] = v[k] != 0u ? 1u : 0u;
            sum += v[k];
        }
        uint32_t tot;
        const uint32_t ex = block_excl_scan(sum, tot);
        if (threadIdx.x < 64u) {
            // the first wave publishes the tile and looks back over 64 lower tiles at a time
            const uint32_t lane = threadIdx.x;
            uint32_t prefix = 0;
            if (tile == 0) {
                if (lane == 0u) __hip_atomic_store(&st[0], SC_PRE | tot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else {
                if (lane == 0u) __hip_atomic_store(&st[tile], SC_AGG | tot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                // lower tiles are held by running workgroups, so each publishes; the wall-clock
                // bound only keeps a broken invariant from hanging the device
                const uint64_t t0 = wall_clock64();
                int j0 = (int)tile - 1;  // window: tiles j0 - lane
                for (;;) {
                    const int j = j0 - (int)lane;
                    // below tile 0 reads as an inclusive prefix of 0 (tile 0 always publishes one first)
                    const uint64_t w =
                        j >= 0 ? __hip_atomic_load(&st[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : SC_PRE;
                    const uint32_t state = (uint32_t)(w >> 62);
                    const uint64_t pre = __ballot(state == 2u), none = __ballot(state == 0u);
                    // the nearest inclusive prefix, and every tile between it and this one published
                    const uint32_t first = pre ? (uint32_t)__ffsll((unsigned long long)pre) - 1u : 64u;
                    const uint64_t upto = first >= 63u ? ~0ull : (2ull << first) - 1ull;
                    if (none & upto) {
                        if (wall_clock64() - t0 > 200000000ull) {  // 2 s: report, do not hang
                            if (lane == 0u && err) atomicOr(err, STICKY_TIMEOUT);
                            break;
                        }
                        __builtin_amdgcn_s_sleep(1);
                        continue;
                    }
                    uint32_t val = lane <= first ? (uint32_t)w : 0u;
                    val = __shfl(wave_incl_scan(val), 63, 64);
                    prefix += val;
                    if (first < 64u) break;
                    j0 -= 64;
                }
                if (lane == 0u)
                    __hip_atomic_store(&st[tile], SC_PRE | (uint32_t)(prefix + tot), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            }
            if (lane == 0u) s_prefix = prefix;
        }
        __syncthreads();
        uint32_t run = s_prefix + ex;
        if (whole) {
            uint4* p = reinterpret_cast<uint4*>(out + base);
#pragma unroll
            for (int q = 0; q < SC_ITEMS / 4; ++q) {
                uint4 x;
                x.x = run;
                run += v[4 * q];
                x.y = run;
                run += v[4 * q + 1];
                x.z = run;
                run += v[4 * q + 2];
                x.w = run;
                run += v[4 * q + 3];
                p[q] = x;
            }
        } else {
#pragma unroll
            for (int k = 0; k < SC_ITEMS; ++k) {
                if (base + k < n) out[base + k] = run;
                run += v[k];
            }
        }
        if (tile == nt - 1 && threadIdx.x == SC_THREADS - 1) {
            out[n] = s_prefix + tot;
            if (total_out) *total_out = s_prefix + tot;
        }
        if (nt <= gridDim.x) break;  // every tile was a first tile
        if (threadIdx.x == 0) s_tile = gridDim.x + atomicAdd(&tmp[0], 1u);
        __syncthreads();  // s_prefix is rewritten by the next tile; the ticket is in
        tile = s_tile;
        __syncthreads();  // every thread has the ticket before thread 0 takes the next one
    }
    __shared__ bool s_last;
    if (threadIdx.x == 0) {
        // finish count: this workgroup's row, then the top counter once the row is complete
        const uint32_t G = gridDim.x, r = blockIdx.x % SC_ROWS;
        const uint32_t in_row = (G - r + SC_ROWS - 1u) / SC_ROWS, rows = G < SC_ROWS ? G : SC_ROWS;
        bool last = false;
        if (atomicAdd(&tmp[SC_ROW0 + 32u * r], 1u) == in_row - 1u) {
            // every member of the row has added
            __hip_atomic_store(&tmp[SC_ROW0 + 32u * r], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            last = atomicAdd(&tmp[SC_TOP], 1u) == rows - 1u;
        }
        s_last = last;
    }
    __syncthreads();
    if (s_last) {
        // every workgroup has finished its look-back: reset the scratch for the next call
        for (uint32_t k = threadIdx.x; k < nt; k += SC_THREADS)
            __hip_atomic_store(&st[k], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (threadIdx.x == 0) {
            __hip_atomic_store(&tmp[0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&tmp[SC_TOP], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

size_t scan_tmp_words(uint32_t n) { return SC_STATUS + 2 * (size_t)((n + SC_TILE - 1) / SC_TILE); }

__global__ void k_zero1(uint32_t* p, uint32_t* q) {
    *p = 0;
    if (q) *q = 0;
}

void scan_exclusive(const uint32_t* in, uint32_t* out, uint32_t n, uint32_t* tmp, hipStream_t s, uint32_t* total_out,
                    const uint32_t* n_dev, bool flags, uint32_t* err) {
    if (n == 0) {
        hipLaunchKernelGGL(k_zero1, dim3(1), dim3(1), 0, s, out, total_out);
        return;
    }
    const uint32_t nb = (n + SC_TILE - 1) / SC_TILE;
    const uint32_t groups = std::min<uint32_t>(nb, n_dev ? SC_MAX_GROUPS_DEV : SC_MAX_GROUPS);
    hipLaunchKernelGGL(k_scan_1p, dim3(groups), dim3(SC_THREADS), 0, s, in, out, n, tmp, nb, total_out, n_dev,
                       flags ? 1 : 0, err);
}

// ---------------------------------------------------------------- radix sort
// Stable LSD radix sort, 8-bit digits, every pass in one launch.  Workgroups of 16 waves take
// tiles of 2048 or 4096 keys, a wave consecutive ones: it ranks 64 at a time in index order (the
// lanes with one digit by a ballot per digit bit) on counters of its own in LDS, so a tile's
// ranks take no barrier; the waves' counts are then prefixed.  As long as one workgroup can hold
// the keys in registers (one_limit) it sorts alone, through LDS.  Beyond, each workgroup takes a
// run of tiles; per pass it publishes its run's digit counts, the grid meets, it finds its places
// from all counts, scatters, and the grid meets again.  The count may be read on the device:
// workgroups without keys leave at once, so the grid is sized for the capacity at no cost.
//
// The grid that meets must be resident as a whole: at most RS_GROUPS workgroups, half of what the
// chip holds (the steps of a device's worlds take turns, so no other grid that meets runs beside
// it).  200 and 1000 bodies: 14 us for the body
// keys and 7 to 8 for the solve order (with launches per pass 47, and 23 to 47 in tiles of 256
// threads whose ranks met at four barriers); 6000 bodies 27 and 30 (53 and 72); 100000 bodies 54
// and 47 (65 and 117); the solve order of 1.7M manifolds 320 (889, its keys' own launch 35).
constexpr int RS_THREADS = 1024, RS_WAVES = RS_THREADS / 64;
constexpr uint32_t RS_GROUPS = 128, RS_HDR = SORT_MEET_WORDS;

// Sort keys read from memory.
template <class K> struct KeysGiven {
    using Key = K;
    static constexpr int ITEMS = 4, ONE_ITEMS = 12;
    uint32_t n;
    int bits;
    __device__ uint32_t count() const { return n; }
    __device__ int key_bits() const { return bits; }
    __device__ K key(const K* k, uint32_t i) const { return k[i]; }
    __device__ uint32_t value(const uint32_t* v, uint32_t i) const { return v[i]; }
    __device__ K order(K k) const { return k; }
};
// The solve order's keys, made from the colours and islands: the colour, or with the split
// LOCAL_KEY | root << 8 | colour for a manifold of an island of at most ISLAND_LOCAL_MAX
// manifolds; the value is the manifold's index.  A stable sort then gives the solve order: the
// large islands' manifolds by colour, then the small islands one after another, each by colour
// (manifold index last).  Digits are taken from the key without the colour and root bits that no
// key of the step has (a pile of 6000 bodies: 19 bits, three passes instead of four).
struct KeysSolve {
    using Key = uint32_t;
    static constexpr int ITEMS = 2, ONE_ITEMS = 4;
    Bodies B;
    const uint2* m_ab;
    const uint32_t* col;
    const Counters* cnt;
    uint32_t cap, split;
    int root_bits, colour_bits;  // colour_bits: set by the kernel from the step's colours
    __device__ uint32_t count() const { return min(cap, cnt->m_eff); }
    __device__ int key_bits() const { return split ? colour_bits + root_bits + 1 : colour_bits; }
    __device__ uint32_t key(const uint32_t*, uint32_t m) const {
        uint32_t k = col[m];
        if (split) {
            const uint32_t r = man_root(B, m_ab[m]);
            if (r != UNSET && B.icnt[r] <= ISLAND_LOCAL_MAX) k |= LOCAL_KEY | (r << 8);
        }
        return k;
    }
    __device__ uint32_t value(const uint32_t*, uint32_t m) const { return m; }
    __device__ uint32_t order(uint32_t k) const {
        return (k & 0xFFu) | ((k & ~LOCAL_KEY) >> 8) << colour_bits |
               (split ? (k >> 31) << (colour_bits + root_bits) : 0u);
    }
};

// Barrier over the nb workgroups that take part (all resident): each wave's stores complete,
// then one thread per workgroup arrives (agent-scope release) and waits for the last arrival
// (agent-scope acquire); a bounded wait ORs STICKY_TIMEOUT into *err instead of hanging.
// bar[0] counts arrivals and returns to 0; bar[1] is the generation.
__device__ __forceinline__ void rs_sync(uint32_t* bar, uint32_t nb, uint32_t* err) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t g = __hip_atomic_load(&bar[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t arrived = __hip_atomic_fetch_add(&bar[0], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (arrived == nb - 1) {
            __hip_atomic_store(&bar[0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_fetch_add(&bar[1], 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            const uint64_t t0 = wall_clock64();
            while (__hip_atomic_load(&bar[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == g) {
                __builtin_amdgcn_s_sleep(1);
                if (wall_clock64() - t0 > 200000000ull) {  // 2 s: report, do not hang
                    if (err) atomicOr(err, STICKY_TIMEOUT);
                    break;
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
    }
    __syncthreads();
}

// Most keys of a sort in one workgroup, and the LDS they pass through.  Given keys: 6000 take 27 us
// alone and 37 in two workgroups.  Made keys are gathered through five arrays, which one CU does
// slowly: 9144 take 88 us alone, 35 in five workgroups.
template <class S> __host__ __device__ constexpr uint32_t one_limit() { return (uint32_t)RS_THREADS * S::ONE_ITEMS; }
template <class S> constexpr uint32_t one_bytes(uint32_t n) {
    return (uint32_t)sizeof(typename S::Key) * (n < one_limit<S>() ? n : one_limit<S>());
}
// Sorts into k0, v0.  Given keys start there, one tile per workgroup: the first pass may write over
// them, its workgroups hold their keys in registers by then.
template <class S>
__global__ void __launch_bounds__(RS_THREADS) k_radix_sort(S src, typename S::Key* k0, uint32_t* v0,
                                                           typename S::Key* k1, uint32_t* v1, uint32_t* tmp, uint32_t* err) {
    using K = typename S::Key;
    constexpr int ITEMS = S::ITEMS;
    constexpr uint32_t TILE = RS_THREADS * ITEMS;
    constexpr bool MADE = std::is_same<S, KeysSolve>::value;
    __shared__ uint32_t s_wc[RS_WAVES][256], s_base[256], s_red[8][256], s_part[4];
    extern __shared__ __align__(16) unsigned char s_stage[];
    const uint32_t n = src.count();
    const uint32_t nt = (n + TILE - 1u) / TILE;
    // tiles of a workgroup, workgroups with keys
    const bool one = n <= one_limit<S>();
    const uint32_t run = one ? nt : (nt + gridDim.x - 1u) / gridDim.x;
    const uint32_t ng = run ? (nt + run - 1u) / run : 0u;
    const uint32_t g = blockIdx.x;
    if (g >= ng) return;
    if constexpr (MADE) {
        src.colour_bits = 1;
        while (src.colour_bits < 8 && src.cnt->max_colour > (1u << src.colour_bits)) ++src.colour_bits;
    }
    const int passes = (src.key_bits() + 7) / 8;
    const uint32_t tid = threadIdx.x, lane = lane_id(), wv = tid >> 6;
    const uint64_t lt = (1ull << lane) - 1ull;
    uint32_t* const H = tmp + RS_HDR;
    auto index = [&](uint32_t t, int it) { return t * TILE + wv * (64u * ITEMS) + (uint32_t)it * 64u + lane; };
    auto digit = [&](K k, int p) { return (uint32_t)(src.order(k) >> (8 * p)) & 255u; };
    // the rank of a key among its digit's in the wave's keys so far, on the wave's counters
    uint32_t* const wc = s_wc[wv];
    auto clear = [&]() {
#pragma unroll
        for (int k = 0; k < 4; ++k) wc[64 * k + lane] = 0u;
        __builtin_amdgcn_wave_barrier();
    };
    auto rank1 = [&](bool valid, uint32_t d) -> uint32_t {
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint64_t bal = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? bal : ~bal;
        }
        const uint32_t r = (uint32_t)__popcll(peers & lt);
        const uint32_t before = wc[d];
        __builtin_amdgcn_wave_barrier();
        if (valid && r == 0u) wc[d] = before + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
        return before + r;
    };
    // all waves ranked: their counts turned into the counts of the waves before; threads below 256
    // return their digit's count
    auto prefix = [&]() -> uint32_t {
        __syncthreads();
        uint32_t tot = 0;
        if (tid < 256u) {
#pragma unroll
            for (int w = 0; w < RS_WAVES; ++w) {
                const uint32_t c = s_wc[w][tid];
                s_wc[w][tid] = tot;
                tot += c;
            }
        }
        return tot;
    };
    // s_base[d] = keys of smaller digits (c: the digit's count, threads below 256) + below
    auto place = [&](uint32_t c, uint32_t below) {
        const uint32_t inc = wave_incl_scan(tid < 256u ? c : 0u);
        if (tid < 256u && lane == 63u) s_part[wv] = inc;
        __syncthreads();
        if (tid < 256u) {
            uint32_t o = 0;
            for (uint32_t w = 0; w < wv; ++w) o += s_part[w];
            s_base[tid] = o + inc - c + below;
        }
        __syncthreads();
    };
    if (ng == 1u) {
        // the keys in registers, a wave's consecutive
        constexpr int ONE = S::ONE_ITEMS;
        K key[ONE];
        uint32_t val[ONE], rk[ONE];
        const int items = (int)((n + RS_THREADS - 1u) / RS_THREADS);  // at most ONE: one_limit
        const uint32_t first = wv * 64u * (uint32_t)items + lane;
        auto valid = [&](int it) { return it < items && first + 64u * (uint32_t)it < n; };
#pragma unroll
        for (int it = 0; it < ONE; ++it) {
            const uint32_t i = first + 64u * (uint32_t)it;
            key[it] = valid(it) ? src.key(k0, i) : (K)0;
            val[it] = valid(it) ? src.value(v0, i) : 0u;
        }
        for (int p = 0; p < passes; ++p) {
            clear();
#pragma unroll
            for (int it = 0; it < ONE; ++it) {
                rk[it] = 0u;
                if (it < items) rk[it] = rank1(valid(it), digit(key[it], p));
            }
            place(prefix(), 0u);
#pragma unroll
            for (int it = 0; it < ONE; ++it) {
                const uint32_t d = digit(key[it], p);
                rk[it] += s_base[d] + s_wc[wv][d];
            }
            if (p + 1 == passes) {
#pragma unroll
                for (int it = 0; it < ONE; ++it)
                    if (valid(it)) {
                        k0[rk[it]] = key[it];
                        v0[rk[it]] = val[it];
                    }
                return;
            }
            K* s_key = reinterpret_cast<K*>(s_stage);
            uint32_t* s_val = reinterpret_cast<uint32_t*>(s_stage);
#pragma unroll
            for (int it = 0; it < ONE; ++it)
                if (valid(it)) s_key[rk[it]] = key[it];
            __syncthreads();
#pragma unroll
            for (int it = 0; it < ONE; ++it) key[it] = valid(it) ? s_key[first + 64u * (uint32_t)it] : (K)0;
            __syncthreads();
#pragma unroll
            for (int it = 0; it < ONE; ++it)
                if (valid(it)) s_val[rk[it]] = val[it];
            __syncthreads();
#pragma unroll
            for (int it = 0; it < ONE; ++it) val[it] = valid(it) ? s_val[first + 64u * (uint32_t)it] : 0u;
            __syncthreads();
        }
        return;
    }
    K key[ITEMS];
    uint32_t val[ITEMS], rk[ITEMS];
    auto rank = [&](uint32_t t, int p) -> uint32_t {
        clear();
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) rk[it] = rank1(index(t, it) < n, digit(key[it], p));
        return prefix();
    };
    const uint32_t t0 = g * run, t1 = min(nt, t0 + run);
    for (int p = 0; p < passes; ++p) {
        const bool to1 = ((passes - 1 - p) & 1) != 0;
        K* ko = to1 ? k1 : k0;
        uint32_t* vo = to1 ? v1 : v0;
        // the pass's keys: given ones start in k0, made ones where the first pass does not write
        const bool from1 = p == 0 && !MADE ? false : !to1;
        K* ki = from1 ? k1 : k0;
        uint32_t* vi = from1 ? v1 : v0;
        uint32_t mine = 0;  // the run's keys with this thread's digit
        for (uint32_t t = t0; t < t1; ++t) {
#pragma unroll
            for (int it = 0; it < ITEMS; ++it) {
                const uint32_t i = index(t, it);
                if (p == 0) {
                    key[it] = i < n ? src.key(ki, i) : (K)0;
                    val[it] = i < n ? src.value(vi, i) : 0u;
                    if (MADE && run > 1u && i < n) {
                        ki[i] = key[it];
                        vi[i] = val[it];
                    }
                } else {
                    key[it] = i < n ? ki[i] : (K)0;
                    val[it] = i < n ? vi[i] : 0u;
                }
            }
            if (t != t0) __syncthreads();  // the counts of the tile before have been read
            mine += rank(t, p);
        }
        if (tid < 256u) H[256u * g + tid] = mine;
        rs_sync(tmp, ng, err);
        // digit d's keys in all runs and in the runs before this one: four threads a digit
        {
            const uint32_t d = tid & 255u, q = tid >> 8;
            uint32_t all = 0, below = 0;
            for (uint32_t r = q; r < ng; r += 32u) {
                uint32_t c[8];
#pragma unroll
                for (uint32_t u = 0; u < 8u; ++u) c[u] = r + 4u * u < ng ? H[256u * (r + 4u * u) + d] : 0u;
#pragma unroll
                for (uint32_t u = 0; u < 8u; ++u) {
                    all += c[u];
                    below += r + 4u * u < g ? c[u] : 0u;
                }
            }
            s_red[q][d] = all;
            s_red[4u + q][d] = below;
        }
        __syncthreads();
        uint32_t all = 0, below = 0;
        if (tid < 256u) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                all += s_red[q][tid];
                below += s_red[4 + q][tid];
            }
        }
        place(all, below);
        for (uint32_t t = t0; t < t1; ++t) {
            uint32_t tot = 0;
            if (run > 1u) {
#pragma unroll
                for (int it = 0; it < ITEMS; ++it) {
                    const uint32_t i = index(t, it);
                    key[it] = i < n ? ki[i] : (K)0;
                    val[it] = i < n ? vi[i] : 0u;
                }
                tot = rank(t, p);
                __syncthreads();
            }
#pragma unroll
            for (int it = 0; it < ITEMS; ++it) {
                if (index(t, it) >= n) continue;
                const uint32_t d = digit(key[it], p);
                const uint32_t pos = s_base[d] + s_wc[wv][d] + rk[it];
                if (pos < n) {
                    ko[pos] = key[it];
                    vo[pos] = val[it];
                }
            }
            if (run > 1u) {
                __syncthreads();
                if (tid < 256u) s_base[tid] += tot;
                __syncthreads();
            }
        }
        if (p + 1 < passes) rs_sync(tmp, ng, err);
    }
}

// ---------------------------------------------------------------- per-pass sort
// More given keys than RS_GIVEN: three launches a pass (per-tile digit counts, their scan, the
// scatter).  A grid that meets writes back and drops every XCD's L2 at each meeting, once per
// workgroup: 1M keys of 30 bits take 257 us so, 100000 52.  Digits of up to ten bits, so 30 bits
// take three passes.  The scatter is bound by its write requests (1M random keys are 2M of them
// a pass when each lane writes its own): a tile goes through LDS into digit order first and then
// out in runs.  1M keys of 30 bits: 79 us (8-bit digits, tiles of 1024 keys written by lane: 106;
// ten bits written by lane: 91); 600000 68 (83), 300000 65 (72), 140000 60 (65).
constexpr uint32_t RS_GIVEN = 131072u;
constexpr int RP_THREADS = 1024, RP_ITEMS = 4, RP_TILE = RP_THREADS * RP_ITEMS;
constexpr int RP_BITS = 10, RP_DIGITS = 1 << RP_BITS;

// Per-tile digit counts, digit-major: hist[d * tiles + tile].
template <class K>
__global__ void __launch_bounds__(RP_THREADS) k_rs_hist(const K* __restrict__ keys, uint32_t n, int shift, uint32_t mask,
                                                        uint32_t* __restrict__ hist) {
    __shared__ uint32_t h[RP_DIGITS];
    h[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * RP_TILE;
#pragma unroll
    for (int it = 0; it < RP_ITEMS; ++it) {
        const uint32_t i = base + it * RP_THREADS + threadIdx.x;
        if (i < n) atomicAdd(&h[(uint32_t)(keys[i] >> shift) & mask], 1u);
    }
    __syncthreads();
    hist[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = h[threadIdx.x];
}

template <class K>
__global__ void __launch_bounds__(RP_THREADS) k_rs_scatter(const K* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                           K* __restrict__ kout, uint32_t* __restrict__ vout, uint32_t n,
                                                           int shift, uint32_t mask, const uint32_t* __restrict__ offs) {
    constexpr int WAVES = RP_THREADS / 64;
    // the waves' digit counts (at most a tile: 16 bits), then the tile's keys in digit order
    __shared__ __align__(8) unsigned char s_mem[2 * WAVES * RP_DIGITS];
    static_assert(sizeof(K) * RP_TILE <= sizeof(s_mem), "keys lie where the counts were");
    __shared__ uint32_t s_val[RP_TILE], s_start[RP_DIGITS], s_delta[RP_DIGITS], s_w[WAVES];
    uint16_t* const s_wc = reinterpret_cast<uint16_t*>(s_mem);
    K* const s_key = reinterpret_cast<K*>(s_mem);
    const uint32_t tid = threadIdx.x, lane = lane_id(), wv = tid >> 6;
    const uint32_t off = offs[(size_t)tid * gridDim.x + blockIdx.x];  // this thread's digit
    const uint32_t base = blockIdx.x * RP_TILE, first = base + wv * (64u * RP_ITEMS) + lane;
    const uint64_t lt = (1ull << lane) - 1ull;
    K k[RP_ITEMS];
    uint32_t v[RP_ITEMS], rk[RP_ITEMS];
#pragma unroll
    for (int it = 0; it < RP_ITEMS; ++it) {
        const uint32_t i = first + 64u * it;
        k[it] = i < n ? kin[i] : (K)0;
        v[it] = i < n ? vin[i] : 0u;
    }
    uint16_t* const wc = s_wc + wv * RP_DIGITS;
#pragma unroll
    for (int q = 0; q < RP_DIGITS / 64; ++q) wc[64 * q + lane] = 0u;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int it = 0; it < RP_ITEMS; ++it) {
        const bool valid = first + 64u * it < n;
        const uint32_t d = (uint32_t)(k[it] >> shift) & mask;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < RP_BITS; ++b) {
            const uint64_t bal = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? bal : ~bal;
        }
        const uint32_t r = (uint32_t)__popcll(peers & lt);
        const uint32_t before = wc[d];
        __builtin_amdgcn_wave_barrier();
        if (valid && r == 0u) wc[d] = (uint16_t)(before + (uint32_t)__popcll(peers));
        __builtin_amdgcn_wave_barrier();
        rk[it] = before + r;
    }
    __syncthreads();
    // the waves' counts of a digit turned into the counts of the waves before, the digits' starts
    uint32_t tot = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        const uint32_t c = s_wc[w * RP_DIGITS + tid];
        s_wc[w * RP_DIGITS + tid] = (uint16_t)tot;
        tot += c;
    }
    const uint32_t inc = wave_incl_scan(tot);
    if (lane == 63u) s_w[wv] = inc;
    __syncthreads();
    uint32_t start = inc - tot;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) start += (uint32_t)w < wv ? s_w[w] : 0u;
    s_start[tid] = start;
    s_delta[tid] = off - start;
    __syncthreads();
#pragma unroll
    for (int it = 0; it < RP_ITEMS; ++it) {
        const uint32_t d = (uint32_t)(k[it] >> shift) & mask;
        rk[it] += s_start[d] + wc[d];
    }
    __syncthreads();  // the counts are read: keys take their place
#pragma unroll
    for (int it = 0; it < RP_ITEMS; ++it) {
        if (first + 64u * it >= n) continue;
        s_key[rk[it]] = k[it];
        s_val[rk[it]] = v[it];
    }
    __syncthreads();
    const uint32_t m = n - base < (uint32_t)RP_TILE ? n - base : (uint32_t)RP_TILE;
#pragma unroll
    for (int it = 0; it < RP_ITEMS; ++it) {
        const uint32_t j = (uint32_t)it * RP_THREADS + tid;
        if (j >= m) continue;
        const K key = s_key[j];
        const uint32_t pos = s_delta[(uint32_t)(key >> shift) & mask] + j;
        kout[pos] = key;
        vout[pos] = s_val[j];
    }
}

// Scratch of the per-pass sort: the histogram with the scan's total, then the scan's scratch.
static size_t hist_words(uint32_t nb) { return (size_t)RP_DIGITS * nb + 2; }
size_t radix_tmp_words(uint32_t n) {
    const uint32_t nb = (n + RP_TILE - 1) / RP_TILE;
    return hist_words(nb) + scan_tmp_words(RP_DIGITS * nb);
}
size_t radix_meet_words() { return RS_HDR + 256u * RS_GROUPS; }

template <class S> static uint32_t rs_groups(uint32_t n, uint32_t cus) {
    return std::max(1u, std::min({(n - 1u) / (RS_THREADS * S::ITEMS) + 1u, RS_GROUPS, cus}));
}
template <class K>
static int radix_sort_impl(K* keys, uint32_t* vals, K* keys_alt, uint32_t* vals_alt, uint32_t n, int end_bit,
                           uint32_t* tmp, uint32_t* meet, uint32_t cus, hipStream_t s, uint32_t* err) {
    if (n == 0 || end_bit <= 0) return 0;
    const uint32_t g = rs_groups<KeysGiven<K>>(n, cus);
    if (n <= RS_GIVEN && (uint64_t)g * RS_THREADS * KeysGiven<K>::ITEMS >= n) {
        const uint32_t lds = n <= one_limit<KeysGiven<K>>() ? one_bytes<KeysGiven<K>>(n) : 0u;
        hipLaunchKernelGGL(k_radix_sort<KeysGiven<K>>, dim3(g), dim3(RS_THREADS), lds, s, KeysGiven<K>{n, end_bit}, keys, vals,
                           keys_alt, vals_alt, meet, err);
        return 0;
    }
    const uint32_t nb = (n + RP_TILE - 1) / RP_TILE;
    uint32_t* hist = tmp;  // scanned in place
    uint32_t* scan_tmp = tmp + hist_words(nb);  // 8-byte aligned for the scan's status words
    // the fewest passes, their digits as narrow as they can be
    const int np = (end_bit + RP_BITS - 1) / RP_BITS, bits = (end_bit + np - 1) / np;
    const uint32_t mask = (1u << bits) - 1u;
    K* ki = keys;
    K* ko = keys_alt;
    uint32_t* vi = vals;
    uint32_t* vo = vals_alt;
    int passes = 0;
    for (int shift = 0; shift < end_bit; shift += bits) {
        hipLaunchKernelGGL(k_rs_hist<K>, dim3(nb), dim3(RP_THREADS), 0, s, ki, n, shift, mask, hist);
        scan_exclusive(hist, hist, RP_DIGITS * nb, scan_tmp, s, nullptr, nullptr, false, err);
        hipLaunchKernelGGL(k_rs_scatter<K>, dim3(nb), dim3(RP_THREADS), 0, s, ki, vi, ko, vo, n, shift, mask, hist);
        K* tk = ki; ki = ko; ko = tk;
        uint32_t* tv = vi; vi = vo; vo = tv;
        ++passes;
    }
    return passes & 1;
}

int radix_sort_u64(uint64_t* keys, uint32_t* vals, uint64_t* keys_alt, uint32_t* vals_alt, uint32_t n, int end_bit,
                   uint32_t* tmp, uint32_t* meet, uint32_t cus, hipStream_t s, uint32_t* err) {
    return radix_sort_impl<uint64_t>(keys, vals, keys_alt, vals_alt, n, end_bit, tmp, meet, cus, s, err);
}

int radix_sort_u32(uint32_t* keys, uint32_t* vals, uint32_t* keys_alt, uint32_t* vals_alt, uint32_t n, int end_bit,
                   uint32_t* tmp, uint32_t* meet, uint32_t cus, hipStream_t s, uint32_t* err) {
    return radix_sort_impl<uint32_t>(keys, vals, keys_alt, vals_alt, n, end_bit, tmp, meet, cus, s, err);
}

int radix_setup() {
    auto allow = [](const void* f, uint32_t bytes) {
        return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess;
    };
    return allow((const void*)k_radix_sort<KeysGiven<uint32_t>>, one_bytes<KeysGiven<uint32_t>>(~0u)) &&
                   allow((const void*)k_radix_sort<KeysGiven<uint64_t>>, one_bytes<KeysGiven<uint64_t>>(~0u)) &&
                   allow((const void*)k_radix_sort<KeysSolve>, one_bytes<KeysSolve>(~0u))
               ? 1 : 0;
}

void sort_solve_order(const Bodies& B, const uint2* m_ab, const uint32_t* col, uint32_t cap, uint32_t split, int root_bits,
                      uint32_t* key, uint32_t* val, uint32_t* key_alt, uint32_t* val_alt, uint32_t* meet, uint32_t cus,
                      Counters* cnt, hipStream_t s) {
    if (cap == 0) return;
    KeysSolve src{B, m_ab, col, cnt, cap, split, root_bits, 8};
    hipLaunchKernelGGL(k_radix_sort<KeysSolve>, dim3(rs_groups<KeysSolve>(cap, cus)), dim3(RS_THREADS),
                       one_bytes<KeysSolve>(cap), s, src, key, val, key_alt,
                       val_alt, meet, &cnt->sticky);
}

}  // namespace axm
