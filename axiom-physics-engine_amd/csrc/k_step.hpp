// Launch wrappers of the step kernels (k_step.hip) and the solver-row layout.
#pragma once
#include "launch.hpp"

namespace axm {

// Solver rows in solve order, slot-major.  Per contact point k of slot s, JROWS
// float4 at J[(k * JROWS + j) * cap + s] hold the three constraint directions
// d = n, t1, t2 with their angular Jacobians a = rA x d, b = rB x d and the
// inverse-inertia-weighted terms ia = IA a, ib = IB b (precomputed once per
// step, so a sweep's row update is dot products and fused multiply-adds):
//   j0 (n, mN)     j1 (aN, kN)   j2 (bN, -)  j3 (iaN, target)  j4 (ibN, -)
//   j5 (t1, mT1)   j6 (a1, kT1)  j7 (b1, -)  j8 (ia1, -)       j9 (ib1, -)
//   j10 (t2, mT2)  j11 (a2, kT2) j12 (b2, -) j13 (ia2, -)      j14 (ib2, -)
// (m = effective mass, k = 1 / m).  lam = (lambda_n, lambda_t1, lambda_t2, -) at
// k * cap + s, lam0 = its warm-start value, fid = feature id.
constexpr uint32_t JROWS = 15;
constexpr uint32_t INBOX_WORDS = 8;  // 64-bit inbox words per slot of the persistent sweep
struct SolverRows {
    uint4* hdr;  // (a, b, npts, manifold) per slot
    float4* J;
    float4* lam;
    float4* lam0;
    uint32_t* fid;
    uint2* dep;  // per slot: (deg << 8 | rank) of body a and body b in the colour order, UNSET if not dynamic
    uint32_t* colour;  // per slot: the manifold's colour (kept by the next step's incremental colouring)
    uint64_t* inbox;   // persistent sweep: per slot INBOX_WORDS words, velocities of body a (0..3) and b (4..7)
    uint2* next;       // persistent sweep: per slot, the next visit of body a and of b (slot << 1 | side)
};
// Steps between full recolourings (in between, persisting contacts keep their colour).
constexpr uint32_t RECOLOUR_PERIOD = 64;

struct PrevCacheArgs {
    const uint64_t* key;
    const uint32_t* slot;
    uint32_t mask;
    const float4* lam;
    const uint32_t* fid;
    const uint32_t* np;
    const uint32_t* colour;
    uint32_t cap;
    uint32_t valid;
};

// Clears the per-step counters, the step's meeting words and, when given, the 32 pair-kind
// counters.
void launch_counters_begin(Counters* cnt, uint32_t* kinds, const Meeting& meet, hipStream_t s);
// Start of a step: velocities, world inertia, AABBs, cell keys; clears the
// colouring's per-body words.
// The sorted cell keys of the broadphase: 32-bit in the Morton rank mode (one world, where
// a key is the cell's Morton code), else 64-bit (world << 30 | Morton code); one is set.
struct SortedKeys {
    const uint64_t* k64 = nullptr;
    const uint32_t* k32 = nullptr;
    __host__ __device__ uint64_t operator[](uint32_t s) const { return k32 ? (uint64_t)k32[s] : k64[s]; }
};
// Also resets the step's counters and meeting words (as launch_counters_begin).  The keys go to key32 (the
// Morton code) with the Morton bitmap, else to key.
void launch_begin(const Bodies& B, const StepParams& sp, uint32_t n, uint64_t* key, uint32_t* key32, uint32_t* val,
                  uint64_t* bmax0,
                  uint64_t* bmax1, uint64_t* bmask, uint32_t* bdeg, Counters* cnt, uint32_t* kinds,
                  const Meeting& meet, const CellTable& ct, hipStream_t s);
// Islands of the step, after the narrowphase: union-find over the manifolds between awake
// dynamic bodies (root = smallest body index), and wake requests for sleeping islands an
// awake body touched.
void launch_isl_union(const Bodies& B, uint32_t n, const uint2* m_ab, uint32_t cap_man, Counters* cnt,
                      hipStream_t s);
// End of a step (after the integration): island labels, rest times, and islands falling asleep.
void launch_islands(const Bodies& B, const StepParams& sp, uint32_t n, Counters* cnt, hipStream_t s);
void launch_fill_u64(uint64_t* p, uint64_t v, uint32_t n, hipStream_t s);
void launch_fill_u32(uint32_t* p, uint32_t v, uint32_t n, hipStream_t s);
void launch_iota(uint32_t* p, uint32_t n, hipStream_t s);
// Empties the cell hash table and its occupancy bits (nothing with the Morton bitmap,
// whose words k_begin clears).
void launch_cell_clear(const CellTable& t, hipStream_t s);
void launch_cell_table(const Bodies& B, const SortedKeys& skey, const uint32_t* sval, uint32_t n, const CellTable& t,
                       Counters* cnt, uint32_t* scan_tmp, hipStream_t s);
// Pairs per (body, z slice) part, BP_PARTS * n counts in canonical order (stashing
// the first PAIR_STASH partners of each part), then the emit pass into pa / pb at
// the scanned offsets.
// Pair counts per (body, z slice) part in cnt, and per 256-part workgroup in bsum (the
// emit pass takes the exclusive scan of bsum, with the total at [workgroups], as boff).
void launch_pair_count(const Bodies& B, const StepParams& sp, const SortedKeys& skey, const uint32_t* sval,
                       const CellTable& ct, uint32_t n, uint32_t* cnt, uint32_t* bsum, uint32_t* stash, Counters* ctr,
                       hipStream_t s);
void launch_pair_emit(const Bodies& B, const StepParams& sp, const SortedKeys& skey, const uint32_t* sval,
                      const CellTable& ct, uint32_t n, const uint32_t* pcnt, const uint32_t* boff, uint32_t cap,
                      uint32_t* pa, uint32_t* pb, Counters* cnt, const uint32_t* stash, hipStream_t s);
// Narrowphase of every pair: the pairs are first ordered by kind of test (p_kind,
// the 32 counters `kinds` cleared at the step start, `order`), then tested; deep
// box-capsule pairs queue for EPA, run by `epa_groups` workgroups of 64.
void launch_narrow(const Bodies& B, const StepParams& sp, const uint32_t* pa, const uint32_t* pb, uint32_t cap_pairs,
                   uint32_t* p_np, float4* p_pt, float4* p_nf, uint32_t* epa_list, uint32_t* p_kind, uint32_t* kinds,
                   uint32_t* order, uint32_t epa_groups, Counters* cnt, hipStream_t s);
void launch_compact(const uint32_t* pa, const uint32_t* pb, uint32_t cap_pairs, const uint32_t* p_np,
                    const float4* p_pt, const float4* p_nf, const uint32_t* moff, uint32_t cap, uint2* m_ab,
                    uint32_t* m_np, float4* c_pt, float4* c_nf, Counters* cnt, hipStream_t s);
int colour_blocks_per_cu();
// Jones-Plassmann colouring; `prev` (previous step's (a, b) -> slot table and colours,
// valid = a previous step exists) enables the incremental form between full recolourings.
// Colouring: the keep pass, then Jones-Plassmann rounds over the manifolds not
// kept (`list`), in one workgroup for a short list or on the whole grid.
// With split, the first launch also counts the manifolds per island (icnt, after the union
// kernel), which the colour sort input of the island split needs.
void launch_colour(const Bodies& B, const uint2* m_ab, uint32_t cap_man, uint32_t* col, uint64_t* prio,
                   uint64_t* bmax0, uint64_t* bmax1, uint64_t* bmask, uint32_t* bdeg, uint32_t* list, GridBar* bar,
                   Counters* cnt, uint32_t blocks, const PrevCacheArgs& prev, uint32_t split, hipStream_t s);
// Work the row preparation launch also does for the launches after it, each in a loop of
// its own over the grid: the colour offsets of the sorted keys skey (col_off[c] = first
// position whose key has colour >= c, c = 0..K, and m_glob = col_off[K], when col_off is
// set), the small islands' work list from the same keys (when list is set), clearing zero_n words (the sweep's residual words),
// and emptying the (a, b) -> slot table of row set cset (the entries its last build
// recorded, at the positions cpos holds; when ckey is set, the table's build is then made
// without clearing it).  More than max_k colours fail the step (STICKY_COLOURS).
struct PrepExtra {
    const uint32_t* skey = nullptr;
    uint32_t* col_off = nullptr;
    uint32_t max_k = 0xFFFFFFFFu;
    uint2* list = nullptr;
    uint32_t* zero = nullptr;
    uint32_t zero_n = 0;
    uint64_t* ckey = nullptr;
    const uint32_t* cpos = nullptr;
    uint32_t cset = 0;
};
void launch_prep(const Bodies& B, const StepParams& sp, const uint32_t* order, uint32_t cap, const uint2* m_ab,
                 const uint32_t* m_np, const float4* c_pt, const float4* c_nf, const SolverRows& R,
                 const PrevCacheArgs& pca, const float4* warm_in, const uint32_t* col, const uint64_t* bmask,
                 const uint32_t* bdeg, Counters* cnt, float* feat, const PrepExtra& X, hipStream_t s);
// Writes the learned warm start (network outputs Y, rows 4 * slot + point) into the impulse rows.
void launch_mlp_apply(const SolverRows& R, const Counters* cnt, uint32_t cap, const float* Y, const StepParams& sp,
                      hipStream_t s);
// Residual checks inside one persistent sweep launch: after every `every` sweeps and
// after the last one, the residual (the k_residual value) is written to
// bits[sweeps - 1]; the launch stops at the first check whose residual is <= tol
// (never when tol < 0) and stores the sweeps it ran in Counters::sweeps_run.
// The arrivals of the check after `sweeps` sweeps are counted in CHECK_ROWS words one
// line apart, arrive[((sweeps - 1) * CHECK_ROWS + r) * CHECK_ROW_WORDS] (workgroup g
// adds to row g mod CHECK_ROWS: atomics on one line queue one after another); both
// arrays start the step at zero.  bits == nullptr means no checks.
constexpr uint32_t CHECK_ROWS = 8, CHECK_ROW_WORDS = 32;
// The islands swept in the same launch count their arrivals in two 64-bit words each, 64 bytes
// apart, ISL_ARRIVE_WORDS per island of the work list's largest class (launch_flow_init clears
// them): isl_arrive_words for a manifold capacity.
constexpr uint32_t ISL_ARRIVE_WORDS = 16;
inline size_t isl_arrive_words(uint32_t cap_man) { return (size_t)ISL_ARRIVE_WORDS * (cap_man / 257u + 1u); }
// Words of a residual buffer for `cap` sweeps: the residual of each sweep, then the
// arrival rows of a check after each sweep.
inline uint32_t res_words(uint32_t cap) { return cap * (1u + CHECK_ROWS * CHECK_ROW_WORDS); }
struct SweepStop {
    uint32_t* bits = nullptr;
    uint32_t* arrive = nullptr;
    unsigned long long* isl_arrive = nullptr;
    float tol = -1.0f;
    uint32_t every = 1;
};
// Launch shape of the register sweep (flow_part).
constexpr uint32_t FLOW_THREADS = 512, FLOW_WAVES = FLOW_THREADS / 64u;
constexpr uint32_t FLOW_WAVE_SLOTS = 32;
// Most slots of large islands that it takes on G workgroups; the staged sweep takes more.
inline __host__ __device__ uint32_t flow_slots(uint32_t G) { return G * FLOW_WAVES * FLOW_WAVE_SLOTS; }
// It reaches the inboxes by 32-bit byte offsets into a buffer of this many bytes.
constexpr uint32_t FLOW_INBOX_BYTES = 0x7FFFFFFFu;
// Pieces of 32 slots of the islands of the largest class that the register sweep takes on G
// workgroups: all of them, or none, when one workgroup per island (stream_island) is faster.
// A sweep costs the register sweep its chain of visits (15 us at ten colours) while everything
// fits its waves, and about 0.5 ns per slot beyond (160k slots: 80 us); one workgroup takes
// about 25 ns per slot of its island, all islands at once on as many CUs (44 us for 1880 slots,
// 100 us for 3950).  None, too, when a step has more manifolds than its inboxes' offsets reach
// (33 million): these islands' slots come after the large ones', anywhere up to the last.
inline __host__ __device__ uint32_t wide_pieces(const Counters* cnt, uint32_t G) {
    const uint32_t nl = (cnt->m_glob + FLOW_WAVE_SLOTS - 1u) / FLOW_WAVE_SLOTS, w = cnt->isl_wide;
    if (cnt->max_colour > 64u) return 0u;
    if ((uint64_t)cnt->m_eff * INBOX_WORDS * 8u > FLOW_INBOX_BYTES) return 0u;
    const bool fits = nl <= G * FLOW_WAVES && nl + w <= G * FLOW_WAVES;
    return fits || (uint64_t)cnt->isl_most * 50u > (uint64_t)w * FLOW_WAVE_SLOTS ? w : 0u;
}
// Prepares the large islands' sweeps (after the row preparation): inboxes and next visits, with
// the work list also those of the islands of its largest class that the solve launch of `cus`
// workgroups will take (isl_arrive: their arrival words).
void launch_flow_init(const Bodies& B, const SolverRows& R, uint32_t cap, const uint64_t* bmask, const Counters* cnt,
                      const uint2* list, unsigned long long* isl_arrive, uint32_t cus, hipStream_t s);
// Shape of the staged sweep: `groups` workgroups of one wave, each with `lds_bytes` of LDS for
// its staged rows; all of them must be resident at once (see pgs_own_setup).
struct OwnShape {
    uint32_t groups, lds_bytes, tune;
};
// The solver's sweeps, in `cus` workgroups of 512 threads, all resident at once (see
// pgs_solve_setup).  SOLVE_LARGE: the large islands; up to cus x 256 slots run with one slot per
// pair of lanes, more in the staged sweep.  SOLVE_LIST: the islands of the work list and the small
// ones, which tol > 0 stops each at its own residual.  With `wide` the register sweep takes the
// islands of the list's largest class when that is faster (launch_flow_init has prepared them);
// parts in launches of their own name the same.  bmask holds the colouring's per-body colour
// masks.  spin_limit: microseconds after which a wait gives up, in the register sweep those without
// progress of any wave, in the staged sweep those from its start.  Events ev0 / ev1, when given, are
// recorded around the launch.
constexpr uint32_t SOLVE_LARGE = 1u, SOLVE_LIST = 2u;
void launch_pgs_solve(const Bodies& B, const StepParams& sp, const SolverRows& R, uint32_t cap, const uint64_t* bmask,
                      uint32_t nsweeps, Counters* cnt, uint32_t spin_limit, uint32_t cus, const uint32_t* skey,
                      const uint2* list, float tol, uint32_t parts, bool wide, const OwnShape& own, const SweepStop& stop,
                      hipStream_t s, hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr);
// Allows the solve launch its LDS; its workgroups that fit on one CU (0 on error).
int pgs_solve_setup();
// Raises the sweep kernel's dynamic-LDS limit to max_lds_bytes and returns how many of
// its workgroups with lds_bytes each fit on one CU (0 on error).
int pgs_own_setup(uint32_t max_lds_bytes, uint32_t lds_bytes);
// Allows the islands' union its LDS; 0 on failure.
int isl_union_setup();
void launch_pgs(const Bodies& B, const StepParams& sp, const SolverRows& R, uint32_t s0, uint32_t s1, uint32_t cap,
                uint32_t first, hipStream_t s);
void launch_residual(const Bodies& B, const StepParams& sp, const SolverRows& R, const Counters* cnt, uint32_t cap,
                     uint32_t* out_bits, hipStream_t s);
// An (a, b) -> slot table of one row set, for its build.
struct CacheTable {
    uint64_t* key = nullptr;
    uint32_t* slot = nullptr;
    uint32_t mask = 0;
    uint32_t* np_out = nullptr;
    uint32_t* pos = nullptr;
    uint32_t set = 0;
};
// Empties the (a, b) -> slot table of row set `set` (the entries its last build made, at
// the positions pos holds; skipped with clear = false, when the row preparation did it)
// and fills it with the step's slots.
void launch_cache_build(const SolverRows& R, Counters* cnt, uint32_t cap, uint64_t* key, uint32_t* slot,
                        uint32_t mask, uint32_t* np_out, uint32_t* pos, uint32_t set, hipStream_t s,
                        bool clear = true);
// Rehashes the `on`-slot table (okey, oslot) into the empty table (key, slot, mask), with the
// new positions in pos.
void launch_cache_rehash(const uint64_t* okey, const uint32_t* oslot, uint32_t on, uint64_t* key, uint32_t* slot,
                         uint32_t mask, Counters* cnt, uint32_t* pos, hipStream_t s);
// sweeps == SWEEPS_ON_DEVICE: the count is read from Counters::sweeps_run.
constexpr uint32_t SWEEPS_ON_DEVICE = 0xFFFFFFFFu;
// With R and C, the same launch also builds the (a, b) -> slot table C of the step's rows
// (as launch_cache_build with clear = false).
void launch_integrate(const Bodies& B, const StepParams& sp, uint32_t n, Counters* cnt, uint32_t sweeps, hipStream_t s,
                      const SolverRows* R = nullptr, const CacheTable* C = nullptr);

}  // namespace axm
