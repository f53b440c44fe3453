// Batched Leiden over G vertex-disjoint graphs: one level per call
// (ckv_batched_leiden, with COO aggregation and per-graph label densification
// beside it) and the whole multi-level run (ckv_leiden_run).  Restates the reference's graph/leiden/_csrc (leiden.cu
// 43-205, local_moving.cu 69-210, refinement.cu 71-300, csr.cu 20-271,
// aggregate.cu 24-184, helpers.cu 9-122) for MI355X:
//
//   * a vertex takes half a wave, a wave or a workgroup by the length of its
//     row, which its threads hold in registers; its neighbour communities
//     gather in an LDS table by compare-and-swap, in f64 sums of arbitrary
//     order (exact for weights within 29 bits of each other's range);
//   * the sweep loops run without host round trips: every sweep's kernels
//     are queued up front and read from a ring of marks, one per sweep in which
//     a vertex moved, where their phase stands (up or down moves, stalled,
//     ended); sweeps after the end hand on what they were given or return;
//   * the symmetric CSR of a list in any order is one stable radix sort of
//     (src, dst) keys, rows ordered by neighbour id.
//
// Move rules follow the reference: synchronous moves on a snapshot, gain
//   dQ = (k_v,new - k_v,old)/m + gamma k_v (Sigma_old - k_v - Sigma_new)/(2 m^2),
// neighbour-community weights rounded to float, the per-vertex jitter and the
// per-sweep rank of the reference's PCG hash (rng.cuh), the up/down gate in
// local moving, the well-connectedness gate and the independent-set commit in
// refinement.  Equal float scores are broken by the order in which the
// reference's 1024-slot table scan prefers a community's home slot, then by
// smaller id.  A vertex keeps at most TABLE_CAP distinct neighbour
// communities (the reference's table size), in order of first appearance.
//
// Launch sequence of ckv_batched_leiden (one stream, no host sync):
//   mirror_kernel, radix sort, row_ptr_kernel, col_kernel, degree_kernel, graph_sum_kernel (2m)
//   level_init_kernel, row_list_kernel
//   local moving x max_inner_iter: local_moving_kernel, local_moving_giant_kernel
//   pair_init_kernel
//   refinement x max_inner_iter: refine_propose_kernel, refine_propose_giant_kernel, refine_commit_kernel
//   sigma of the result, modularity_kernel, graph_sum_kernel, finish_kernel (labels, -1 for isolated)
//
// ckv_leiden_run keeps the graph as a CSR from level to level.  The first
// level's comes from the ascending edge list with one 32-bit sort of E keys
// (the lists of higher neighbours are the edge list itself; before, all 2E
// entries were sorted by 64-bit keys: 1.25 ms at 9.7 M edges, 0.45 ms now).  A
// level's result contracts the CSR row by row in LDS hash tables, where the
// edge list was relabelled, sorted by 64-bit keys, reduced, and sorted again
// into a CSR (2.0 ms at 9.7 M edges, 0.35 ms now).  Launch sequence per level:
//   level_init, row_list, sweeps as above (giants only where rows can be so long), rank_kernel
//   [the host reads the width], dense_chain_kernel (flag, scan, densify and chain kernels for graphs
//   of more than RANK_MOST vertices), agg_hist, scan, agg_fill (members by super-vertex), agg_list,
//   agg_short (one wave per row), agg_long (workgroup), agg_dense, graph_sum
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <stdint.h>

#include "ckv_amd.h"
#include "ckv_device.h"
#include "ckv_error.h"
#include "ckv_sort.h"
#include "ckv_table.h"

namespace ckv {
namespace {

constexpr int LWAVES = 4;        // vertices (waves) per workgroup
constexpr int LTHREADS = 64 * LWAVES;
constexpr int TABLE_CAP = 1024;  // distinct neighbour communities per vertex
constexpr int ETHREADS = 256;

// Control words of a level.  A sweep in which a vertex moves marks its slot of
// its phase's ring; the next sweeps read the ring themselves, so no kernel runs
// between sweeps to advance a state.  A slot is a word per XCD, each in a line
// of its own: with a mark per moved vertex on one word the first local-moving
// sweeps of 32 8k graphs' levels averaged 64 us, 31 now.  Every RING sweeps
// fold_kernel moves the ring's outcome to the base words.
constexpr int RING = 16;
constexpr int MARK_STRIDE = 32;              // words from one XCD's mark to the next
constexpr int SLOT_WORDS = 8 * MARK_STRIDE;  // a sweep's slot
enum { CTL_OVERFLOW = 0,  // nonzero when a workgroup table overflowed (a broken table bound)
       CTL_STALLS = 1,    // local moving: stalled sweeps before the ring, modulo 2
       CTL_LAST = 2,      // the last sweep before the ring stalled
       CTL_DONE = 3,      // the phase ended before the ring
       CTL_LM = MARK_STRIDE,                     // local moving's ring
       CTL_REFINE = CTL_LM + RING * SLOT_WORDS,  // refinement's ring
       CTL_WORDS = CTL_REFINE + RING * SLOT_WORDS };

// ----------------------------------------------------------------- hashing (rng.cuh)
__device__ __host__ inline uint32_t pcg_hash(uint32_t x) {
  const uint32_t state = x * 747796405u + 2891336453u;
  const uint32_t word = ((state >> ((state >> 28u) + 4u)) ^ state) * 277803737u;
  return (word >> 22u) ^ word;
}
// The reference's hash of (graph, vertex, c, d), each folded in by pcg_hash(h ^ x);
// the first two are the vertex's salt.
__device__ inline uint32_t salt_of(uint32_t g, uint32_t v) { return pcg_hash(pcg_hash(g) ^ v); }
__device__ inline uint32_t mix_salt(uint32_t salt, uint32_t c, uint32_t d) { return pcg_hash(pcg_hash(salt ^ c) ^ d); }
__device__ inline float unit_float(uint32_t h) { return (float)(h >> 8) * (1.0f / 16777216.0f); }
__device__ inline float rand_uniform(uint32_t salt, uint32_t level, uint32_t sweep, uint32_t seed) {
  return unit_float(mix_salt(salt, (level << 16) | sweep, seed));
}
__device__ inline float rand_uniform_pair(uint32_t salt, uint32_t c, uint32_t level, uint32_t sweep, uint32_t seed) {
  const uint32_t s = pcg_hash((sweep << 16) ^ c);
  return unit_float(mix_salt(salt, (level << 16) | (s & 0xFFFFu), seed));
}
__device__ inline float gumbel(float u) {
  u = fmaxf(u, 1.0e-7f);
  u = fminf(u, 1.0f - 1.0e-7f);
  return -logf(-logf(u));
}

// Tie preference among equal scores (larger wins): the reference scans home
// slot s = pcg_hash(c) & 1023 with thread s & 127 (slice index s >> 7, first
// strict maximum kept) and reduces lanes, then warps, with 32-lane
// shuffle-down trees that keep their own value on ties; then the smaller id.
__device__ inline uint32_t bitrev5(uint32_t x) { return __builtin_bitreverse32(x) >> 27; }
__device__ inline uint32_t cand_pref(int32_t c) {
  const uint32_t s = pcg_hash((uint32_t)c) & 1023u;
  const uint32_t key = (bitrev5((s >> 5) & 3u) << 8) | (bitrev5(s & 31u) << 3) | (s >> 7);
  return ((8191u - key) << 18) | (0x3FFFFu - ((uint32_t)c & 0x3FFFFu));
}
constexpr uint32_t STAY_PREF = 0xFFFFFFFFu;  // staying wins every tie
__device__ inline uint32_t ordered(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ inline uint64_t pack(float score, uint32_t pref) { return ((uint64_t)ordered(score) << 32) | pref; }

// ----------------------------------------------------------------- wave helpers
__device__ inline int first_lane(uint64_t m) { return __ffsll((long long)m) - 1; }

// Marks a sweep (its slot of the ring) in which a thread of the wave moved a
// vertex: once per wave at its end, and only while the XCD's word reads zero.
__device__ inline void mark_moved(int32_t* slot, bool moved) {
  int32_t* word = slot + (blockIdx.x & 7) * MARK_STRIDE;
  if (__ballot(moved) != 0 && lane() == 0 && *word == 0)
    __hip_atomic_store(word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Local moving before sweep `sweep` (wave-uniform): done after two stalled
// sweeps in a row; up or down moves, flipped by every stalled sweep
// (leiden.cu:113-135).
struct MoveState {
  bool done;
  int up;
};
struct RingState {
  bool done, last;
  int stalls;
};
// The state after the first n <= RING sweeps of a ring; a single stalled sweep
// ends refinement, two in a row local moving.
__device__ inline RingState ring_state(const int32_t* __restrict__ ctl, bool lm, int n) {
  RingState r{ctl[CTL_DONE] != 0, ctl[CTL_LAST] != 0, ctl[CTL_STALLS]};
  const int32_t* ring = ctl + (lm ? CTL_LM : CTL_REFINE);
  for (int s0 = 0; s0 < n; s0 += 8) {
    const int at = s0 * 8 + lane();
    const uint64_t marks = __ballot(at < 8 * n && ring[at * MARK_STRIDE] != 0);
    for (int k = s0; k < n && k < s0 + 8; ++k) {
      const bool stalled = ((marks >> (8 * (k - s0))) & 0xff) == 0;
      r.done = r.done || (stalled && (!lm || r.last));
      r.stalls ^= stalled ? 1 : 0;
      r.last = stalled;
    }
  }
  return r;
}
__device__ inline MoveState move_state(const int32_t* __restrict__ ctl, int sweep) {
  const RingState r = ring_state(ctl, true, sweep & (RING - 1));
  return MoveState{r.done, 1 ^ (r.stalls & 1)};
}
__device__ inline bool refine_done(const int32_t* __restrict__ ctl, int sweep) {
  return ring_state(ctl, false, sweep & (RING - 1)).done;
}
__device__ inline int32_t* mark_slot(int32_t* ctl, bool lm, int sweep) {
  return ctl + (lm ? CTL_LM : CTL_REFINE) + (sweep & (RING - 1)) * SLOT_WORDS;
}

// Folds a full ring (RING sweeps of one phase) into the base words; with reset,
// clears the words of the phase that begins (its ring is clear).
__global__ void fold_kernel(int32_t* __restrict__ ctl, int lm, int reset) {
  RingState r{false, false, 0};
  if (!reset) r = ring_state(ctl, lm != 0, RING);
  __syncthreads();
  if (lane() == 0) {
    ctl[CTL_DONE] = r.done ? 1 : 0;
    ctl[CTL_STALLS] = r.stalls & 1;
    ctl[CTL_LAST] = r.last ? 1 : 0;
  }
  if (reset) return;
  for (int at = lane(); at < 8 * RING; at += 64) ctl[(lm ? CTL_LM : CTL_REFINE) + at * MARK_STRIDE] = 0;
}

// The lanes whose key equals the first valid lane's, where enough share it for
// one atomic in their place; 0 where not.  (Every vertex of a community adds to
// the community's words: 130,000 atomics on one word take 1.6 ms.)
__device__ inline uint64_t sharing(bool valid, int32_t key) {
  const uint64_t all = __ballot(valid);
  if (all == 0) return 0;
  const uint64_t same = __ballot(valid && key == __shfl(key, first_lane(all)));
  return __popcll(same) >= 8 ? same : 0;
}
__device__ inline bool in_mask(uint64_t m) { return (m >> lane()) & 1; }

// ----------------------------------------------------------------- CSR build
__global__ void mirror_kernel(const int32_t* __restrict__ src, const int32_t* __restrict__ dst,
                              const float* __restrict__ w, int64_t E, int32_t V, int bits,
                              uint64_t* __restrict__ keys, float* __restrict__ vals) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= E) return;
  const int32_t u = src[i], t = dst[i];
  const float wi = w[i];
  const uint64_t sentinel = (uint64_t)V << bits;
  const bool ok = u >= 0 && u < V && t >= 0 && t < V;  // out-of-range edges are dropped
  keys[2 * i] = ok ? ((uint64_t)u << bits) | (uint64_t)t : sentinel;
  vals[2 * i] = u == t ? 2.0f * wi : wi;
  keys[2 * i + 1] = (ok && u != t) ? ((uint64_t)t << bits) | (uint64_t)u : sentinel;
  vals[2 * i + 1] = wi;
}

__global__ void row_ptr_kernel(const uint64_t* __restrict__ keys, int64_t n, int32_t V, int bits,
                               int32_t* __restrict__ row_ptr) {
  const int32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v > V) return;
  const uint64_t target = (uint64_t)v << bits;
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (keys[mid] < target) lo = mid + 1;
    else hi = mid;
  }
  row_ptr[v] = (int32_t)lo;
}

__global__ void col_kernel(const uint64_t* __restrict__ keys, int64_t n, int bits, int32_t* __restrict__ col) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) col[i] = (int32_t)(keys[i] & (((uint64_t)1 << bits) - 1));
}

__global__ __launch_bounds__(LTHREADS) void degree_kernel(const int32_t* __restrict__ row_ptr,
                                                          const float* __restrict__ wt, int32_t V,
                                                          double* __restrict__ k_v) {
  const int32_t v = blockIdx.x * LWAVES + (threadIdx.x >> 6);
  if (v >= V) return;
  const int32_t a = row_ptr[v], b = row_ptr[v + 1];
  double s = 0.0;
  for (int32_t e = a + lane(); e < b; e += 64) s += (double)wt[e];
  s = wave_sum_f64(s);
  if (lane() == 0) k_v[v] = s;
}

// out[g] = sum of x over graph g's S vertices (one workgroup per graph, fixed
// order: strided per-thread sums with eight loads in flight, then a tree over
// the threads).
constexpr int SUM_THREADS = 1024;

__global__ __launch_bounds__(SUM_THREADS) void graph_sum_kernel(const double* __restrict__ x, int32_t S,
                                                                double* __restrict__ out) {
  __shared__ double part[SUM_THREADS / 64];
  const int32_t g = blockIdx.x;
  const double* row = x + (int64_t)g * S;
  double s = 0.0;
  for (int32_t i0 = threadIdx.x; i0 < S; i0 += 8 * SUM_THREADS) {
    double y[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int32_t i = i0 + u * SUM_THREADS;
      y[u] = i < S ? row[i] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) s += y[u];
  }
  s = wave_sum_f64(s);
  if (lane() == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int i = 0; i < SUM_THREADS / 64; ++i) t += part[i];
    out[g] = t;
  }
}

// ----------------------------------------------------------------- sweeps
__global__ void sigma_zero_kernel(double* __restrict__ sigma, int32_t V) {
  const int32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < V) sigma[v] = 0.0;
}

__global__ void sigma_scatter_kernel(const int32_t* __restrict__ labels, const double* __restrict__ k_v, int32_t V,
                                     double* __restrict__ sigma) {
  const int32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  const int32_t c = v < V ? labels[v] : -1;
  double k = c >= 0 ? k_v[v] : 0.0;
  const bool adds = c >= 0 && k != 0.0;
  const uint64_t same = sharing(adds, c);
  if (same == 0) {
    if (adds) unsafeAtomicAdd(sigma + c, k);
    return;
  }
  const bool mine = in_mask(same);
  if (adds && !mine) unsafeAtomicAdd(sigma + c, k);
  k = wave_sum_f64(mine ? k : 0.0);
  if (lane() == first_lane(same)) unsafeAtomicAdd(sigma + c, k);
}

// Rows are [beg[v], end[v]) of col / wt (of a packed CSR, end = beg + 1; the
// rows of a contracted graph leave room behind their entries).
struct Graph {
  const int32_t* beg;
  const int32_t* end;
  const int32_t* col;
  const float* wt;
  const double* k_v;
  const double* two_m;
  int32_t V;
  int32_t S;
  bool unique;  // no row names another vertex twice
};

// v / S for 0 <= v < 2^31 by a multiplication (a 32-bit division is some 40 issue slots).
struct Divisor {
  uint32_t mul;
  int32_t shift;
  explicit Divisor(int32_t S) : mul(0), shift(0) {
    if (S < 2) return;  // one vertex a graph: v itself
    int bits = 1;
    while (((int64_t)1 << bits) < S) ++bits;
    // mul S - 2^(31 + bits) < S <= 2^bits, so the quotient of every v below 2^31 is exact
    mul = (uint32_t)((((uint64_t)1 << (31 + bits)) + (uint64_t)S - 1) / (uint64_t)S);
    shift = bits - 1;
  }
  __device__ int32_t of(int32_t v) const { return mul == 0 ? v : (int32_t)(__umulhi((uint32_t)v, mul) >> shift); }
};

// A load that stays where it is written (the compiler would move one whose
// value is used late behind the loads it should travel with).
template <class T>
__device__ __forceinline__ T load_now(const T* p) {
  if constexpr (sizeof(T) == 4)
    return __builtin_bit_cast(T, __hip_atomic_load((const uint32_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT));
  else
    return __builtin_bit_cast(T, __hip_atomic_load((const uint64_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT));
}

// Sweeps.  A vertex of at most SMALL_ROW entries (nearly all) is handled by
// half a wave; the longer ones, listed once per level, of up to MID_ROW entries
// by a wave and up to GIANT_MIN by a workgroup.  All hold up to ROW_PER entries
// per thread in registers, so that a vertex costs four rounds of loads whatever
// its row: bounds, degree and label; entries; the neighbours' labels; the
// community totals.  Rows longer than GIANT_MIN have kernels of their own.
//
// What bounds a sweep is the instructions issued per entry and the latency of
// those rounds.  Over the 24 sweeps a phase takes in the six levels of eight
// 32k graphs (262,144 vertices, 19.4 M entries, 29,400 rows of more than 128 at
// first) a local-moving sweep averages 70 us and a refinement sweep 88 + 46 us
// (first level: 120 us, 150 + 75 us).  With a wave per vertex that walked its
// row 64 entries at a time through a 256-slot table, longer rows by one wave
// each in a launch behind it, and kernels that cleared and refilled sigma and
// advanced the control words, it was 205 and 305 us.  Rows of 129-256 entries
// on a workgroup each waited at its barriers: 100 and 118 + 57 us.
//
// Sigma, the communities' total degrees, needs no pass of its own: a sweep
// adds every vertex's degree to its new community in the buffer the next sweep
// reads, and clears the buffer after that (three buffers in turn).  In a
// phase's first sweep every vertex is its own community: sigma is k_v, and
// where no row names a neighbour twice every neighbour is a candidate by
// itself, so no table is built (FIRST).
constexpr int SMALL_ROW = 128;
constexpr int MID_ROW = 256;
constexpr int ROW_PER = 4;
constexpr int HUB_THREADS = 256;
constexpr int SWEEP_BLOCKS = 2048;  // eight a compute unit
constexpr int LONG_BLOCKS = 512;    // a multiple of eight
constexpr int SMALL_SLOTS = 184, HUB_SLOTS = 1472;  // table load at most 70%
constexpr int GROUPS = HUB_THREADS / 32;            // half waves per workgroup
// Both kinds of workgroup use the same LDS (20 KB, eight a compute unit).
static_assert(GROUPS * SMALL_SLOTS == HUB_SLOTS && GROUPS * SMALL_ROW == HUB_THREADS * ROW_PER, "tables and lists");

constexpr int GIANT_MIN = TABLE_CAP;  // rows longer than this take a workgroup of GIANT_THREADS
constexpr int GIANT_SLOTS = 4096;
constexpr int GIANT_THREADS = 1024;
constexpr int GIANT_BLOCKS = 512;  // two 65 KB workgroups per CU
static_assert(SMALL_ROW == 32 * ROW_PER && MID_ROW == 64 * ROW_PER && GIANT_MIN == HUB_THREADS * ROW_PER,
              "rows fit their threads' registers");

constexpr int ROW_COUNTS = 3;

// The rows longer than SMALL_ROW: mids (a wave each) from the front of `rows`,
// hubs (a workgroup each) from its back, giants in a list of their own.
struct RowLists {
  int32_t* rows;
  int32_t* giants;
  int32_t* counts;      // mids, hubs, giants; then a run's level width
  int32_t long_blocks;  // workgroups of a sweep that take mids and hubs
  int32_t first;        // workgroups before those that take the other rows
  __device__ int32_t start(int32_t block) const { return block < long_blocks ? block : 0x7fffffff; }
};

// (Places in the lists are reserved once per workgroup: one atomic per wave and
// list queues thousands of them on a few words.)
constexpr int LIST_THREADS = 1024;

__global__ __launch_bounds__(LIST_THREADS) void row_list_kernel(const int32_t* __restrict__ beg,
                                                                const int32_t* __restrict__ end, int32_t V,
                                                                RowLists l) {
  __shared__ int s_n[3], s_at[3];
  const int32_t v = blockIdx.x * LIST_THREADS + threadIdx.x;
  const int32_t d = v < V ? end[v] - beg[v] : 0;
  const int kind = d > GIANT_MIN ? 2 : (d > MID_ROW ? 1 : (d > SMALL_ROW ? 0 : -1));
  if (threadIdx.x < 3) s_n[threadIdx.x] = 0;
  __syncthreads();
  int at = 0;
  for (int k = 0; k < 3; ++k) {
    const uint64_t m = __ballot(kind == k);
    if (m == 0) continue;
    int base = 0;
    if (lane() == 0) base = atomicAdd(s_n + k, __popcll(m));
    base = __shfl(base, 0);
    if (kind == k) at = base + __popcll(m & ((((uint64_t)1) << lane()) - 1));
  }
  __syncthreads();
  if (threadIdx.x < 3) s_at[threadIdx.x] = s_n[threadIdx.x] ? atomicAdd(l.counts + threadIdx.x, s_n[threadIdx.x]) : 0;
  __syncthreads();
  if (kind < 0) return;
  at += s_at[kind];
  if (kind == 2) l.giants[at] = v;
  else l.rows[kind == 0 ? at : V - 1 - at] = v;
}

// The threads of one vertex, with their part of the workgroup's LDS.
struct SweepShared {
  int32_t tc[HUB_SLOTS];                    // communities, -1 free
  double ts[HUB_SLOTS];                     // weight to them
  uint16_t list[HUB_THREADS * ROW_PER];     // slots in use
  uint64_t best[HUB_THREADS / 64];
  double sum[HUB_THREADS / 64];
  int32_t value, count;
};
// (pairs of mirrored lanes in place of xor 4 and 8: the lanes of a pair's side hold equal values by then)
__device__ __forceinline__ uint64_t half_wave_max(uint64_t x) {
  x = pick_u64<true>(x, dpp_u64<0xB1>(x));
  x = pick_u64<true>(x, dpp_u64<0x4E>(x));
  x = pick_u64<true>(x, dpp_u64<0x141>(x));
  x = pick_u64<true>(x, dpp_u64<0x140>(x));
  return pick_u64<true>(x, xor_u64<16>(x));
}
__device__ __forceinline__ double f64_of(uint64_t x) { return __builtin_bit_cast(double, x); }
__device__ __forceinline__ uint64_t u64_of(double x) { return __builtin_bit_cast(uint64_t, x); }
__device__ __forceinline__ double half_wave_sum(double x) {
  x += f64_of(dpp_u64<0xB1>(u64_of(x)));
  x += f64_of(dpp_u64<0x4E>(u64_of(x)));
  x += f64_of(dpp_u64<0x141>(u64_of(x)));
  x += f64_of(dpp_u64<0x140>(u64_of(x)));
  return x + f64_of(xor_u64<16>(u64_of(x)));
}
__device__ __forceinline__ double full_wave_sum(double x) {
  x = half_wave_sum(x);
  return x + f64_of(xor_u64<32>(u64_of(x)));
}

struct HalfWave {
  static constexpr int N = 32, SLOTS = SMALL_SLOTS;
  int32_t* tc;
  double* ts;
  uint16_t* list;
  __device__ explicit HalfWave(SweepShared& sh)
      : tc(sh.tc + (threadIdx.x >> 5) * SMALL_SLOTS), ts(sh.ts + (threadIdx.x >> 5) * SMALL_SLOTS),
        list(sh.list + (threadIdx.x >> 5) * SMALL_ROW) {}
  __device__ int tid() const { return lane() & 31; }
  __device__ void sync() const { wave_lds_sync(); }
  __device__ uint64_t max(uint64_t x) const { return half_wave_max(x); }
  __device__ double sum(double x) const { return half_wave_sum(x); }
  __device__ uint32_t ballot(bool x) const { return (uint32_t)(__ballot(x) >> (lane() & 32)); }
  // The value of the thread that holds the winning key.
  __device__ int32_t of(uint64_t best, uint64_t mine, int32_t value) const {
    return __shfl(value, (lane() & 32) + __builtin_ctz(ballot(mine == best)));
  }
  __device__ bool any(bool x) const { return ballot(x) != 0; }
  // Lists slot h of the threads that took a free one, behind the n listed before.
  __device__ void start_list() const {}
  __device__ int append(bool taken, int h, int n) const {
    const uint32_t m = ballot(taken);
    if (taken) list[n + __popc(m & ((1u << tid()) - 1))] = (uint16_t)h;
    return n + __popc(m);
  }
  __device__ int listed(int n) const { return n; }
};

struct Wave {
  static constexpr int N = 64, SLOTS = 2 * SMALL_SLOTS;
  int32_t* tc;
  double* ts;
  uint16_t* list;
  __device__ explicit Wave(SweepShared& sh)
      : tc(sh.tc + (threadIdx.x >> 6) * SLOTS), ts(sh.ts + (threadIdx.x >> 6) * SLOTS),
        list(sh.list + (threadIdx.x >> 6) * MID_ROW) {}
  __device__ int tid() const { return lane(); }
  __device__ void sync() const { wave_lds_sync(); }
  __device__ uint64_t max(uint64_t x) const { return wave_max_u64(x); }
  __device__ double sum(double x) const { return full_wave_sum(x); }
  __device__ int32_t of(uint64_t best, uint64_t mine, int32_t value) const {
    return __shfl(value, first_lane(__ballot(mine == best)));
  }
  __device__ bool any(bool x) const { return __ballot(x) != 0; }
  __device__ void start_list() const {}
  __device__ int append(bool taken, int h, int n) const {
    const uint64_t m = __ballot(taken);
    if (taken) list[n + __popcll(m & ((((uint64_t)1) << lane()) - 1))] = (uint16_t)h;
    return n + __popcll(m);
  }
  __device__ int listed(int n) const { return n; }
};

struct Workgroup {
  static constexpr int N = HUB_THREADS, SLOTS = HUB_SLOTS;
  SweepShared* sh;
  int32_t* tc;
  double* ts;
  uint16_t* list;
  __device__ explicit Workgroup(SweepShared& s) : sh(&s), tc(s.tc), ts(s.ts), list(s.list) {}
  __device__ int tid() const { return threadIdx.x; }
  __device__ void sync() const { __syncthreads(); }
  __device__ uint64_t max(uint64_t x) const {
    x = wave_max_u64(x);
    if (lane() == 0) sh->best[threadIdx.x >> 6] = x;
    __syncthreads();
    for (int i = 0; i < HUB_THREADS / 64; ++i) x = pick_u64<true>(x, sh->best[i]);
    __syncthreads();
    return x;
  }
  __device__ double sum(double x) const {
    x = full_wave_sum(x);
    if (lane() == 0) sh->sum[threadIdx.x >> 6] = x;
    __syncthreads();
    double t = 0.0;
    for (int i = 0; i < HUB_THREADS / 64; ++i) t += sh->sum[i];
    __syncthreads();
    return t;
  }
  __device__ int32_t of(uint64_t best, uint64_t mine, int32_t value) const {
    if (mine == best) sh->value = value;  // (equal keys are one candidate)
    __syncthreads();
    const int32_t r = sh->value;
    __syncthreads();
    return r;
  }
  __device__ bool any(bool x) const { return __syncthreads_or(x) != 0; }
  __device__ void start_list() const {
    if (threadIdx.x == 0) sh->count = 0;
  }
  __device__ int append(bool taken, int h, int) const {
    const uint64_t m = __ballot(taken);
    if (m == 0) return 0;
    int at = 0;
    if (lane() == 0) at = atomicAdd(&sh->count, __popcll(m));
    at = __shfl(at, 0);
    if (taken) list[at + __popcll(m & ((((uint64_t)1) << lane()) - 1))] = (uint16_t)h;
    return 0;
  }
  __device__ int listed(int) const { return sh->count; }
};

// One vertex's row in its threads' registers: neighbour, weight and whether
// the entry counts (self loops do not).
struct Row {
  int32_t u[ROW_PER];
  float w[ROW_PER];
  bool ok[ROW_PER];
};
template <class P>
__device__ __forceinline__ void load_row(const P& p, const Graph& gr, int32_t v, int32_t a, int32_t b, Row& r) {
  const int32_t* col = gr.col + a + p.tid();
  const float* wt = gr.wt + a + p.tid();
  const int32_t left = b - a - p.tid();
#pragma unroll
  for (int i = 0; i < ROW_PER; ++i) {
    r.u[i] = v;
    r.w[i] = 0.0f;
    if (i * P::N < left) {
      r.u[i] = col[i * P::N];
      r.w[i] = wt[i * P::N];
    }
  }
#pragma unroll
  for (int i = 0; i < ROW_PER; ++i) r.ok[i] = r.u[i] != v;
}

// Frees the slots of all tables of a workgroup; afterwards each vertex frees
// the ones it used.
__device__ __forceinline__ void clear_tables(SweepShared& sh) {
  for (int j = threadIdx.x; j < HUB_SLOTS; j += HUB_THREADS) {
    sh.tc[j] = -1;
    sh.ts[j] = 0.0;
  }
  __syncthreads();
}

// Sums the weights of the entries that count by community c[i] into the
// group's table and lists the slots in use; returns their number.
template <class P>
__device__ __forceinline__ int fill_table(const P& p, const Row& r, const int32_t* c) {
  p.start_list();
  p.sync();  // (the vertex before has freed its slots)
  int n = 0;
#pragma unroll
  for (int i = 0; i < ROW_PER; ++i) {
    bool taken = false;
    int h = 0;
    if (r.ok[i]) {
      h = (int)(__umul24(((uint32_t)c[i] * 0x9E3779B1u) >> 16, (uint32_t)P::SLOTS) >> 16);
      while (true) {  // (at most 70% of the slots are taken: a free one or the community's is found)
        const int32_t cur = __hip_atomic_load(p.tc + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (cur == c[i]) break;
        if (cur == -1) {
          const int32_t prev = atomicCAS(p.tc + h, -1, c[i]);
          taken = prev == -1;
          if (taken || prev == c[i]) break;
        }
        h = h + 1 == P::SLOTS ? 0 : h + 1;
      }
      unsafeAtomicAdd(p.ts + h, (double)r.w[i]);
    }
    n = p.append(taken, h, n);
  }
  p.sync();
  return p.listed(n);
}

// Calls f(community, weight to it, its total) for the candidates: the entries
// that count where no community has two (FIRST), else the n listed slots.  All
// totals are loaded before any is used.
template <class P, bool FIRST, class F>
__device__ __forceinline__ void each_candidate(const P& p, const Row& r, int n, const double* __restrict__ sigma,
                                               F f) {
  int32_t c[ROW_PER];
  float w[ROW_PER];
  double total[ROW_PER];
  bool ok[ROW_PER];
#pragma unroll
  for (int i = 0; i < ROW_PER; ++i) {
    if constexpr (FIRST) {
      ok[i] = r.ok[i];
      c[i] = r.u[i];
      w[i] = r.w[i];
    } else {
      const int j = p.tid() + P::N * i;
      ok[i] = j < n;
      if (ok[i]) {
        const int h = p.list[j];
        c[i] = p.tc[h];
        w[i] = (float)p.ts[h];
        p.tc[h] = -1;
        p.ts[h] = 0.0;
      }
    }
    if (ok[i]) total[i] = sigma[c[i]];
  }
#pragma unroll
  for (int i = 0; i < ROW_PER; ++i) {
    if (ok[i]) f(c[i], w[i], total[i]);
  }
}

// What a level's sweeps read of a vertex's graph: 1 / m and 1 / (2 m^2).
struct LevelConst {
  const double2* scale;
  const uint32_t* salt;
  Divisor graph_of;
};

// What a sweep reads and writes.
struct MoveSweep {
  const double* sigma;
  double* next;        // totals for the next sweep
  double* clear;       // cleared for the sweep after it
  const int32_t* lin;  // labels (not read in a FIRST sweep)
  int32_t* lout;
  int32_t* ctl;
  int32_t sweep;
  float resolution;
  uint32_t seed;
  LevelConst lc;
};

__device__ inline void finish_move(const MoveSweep& s, int32_t v, int32_t choice, double kv) {
  s.lout[v] = choice;
  s.clear[v] = 0.0;
  if (kv != 0.0) unsafeAtomicAdd(s.next + choice, kv);
}

// What a sweep reads of vertex v before its row: loads that depend on v alone,
// issued together.
struct Vertex {
  int32_t v, a, b, g;
  double kv, tm;
  double2 scale;
  uint32_t salt;
};
__device__ __forceinline__ Vertex load_vertex(const Graph& gr, const LevelConst& lc, int32_t v) {
  Vertex x;
  x.v = v;
  x.g = lc.graph_of.of(v);
  x.a = load_now(gr.beg + v);
  x.b = load_now(gr.end + v);
  x.kv = load_now(gr.k_v + v);
  x.tm = load_now(gr.two_m + x.g);
  x.scale.x = load_now(&lc.scale[x.g].x);
  x.scale.y = load_now(&lc.scale[x.g].y);
  x.salt = load_now(lc.salt + v);
  return x;
}

// Returns whether the vertex moves.
template <class P, bool FIRST>
__device__ __forceinline__ bool move_vertex(const P& p, const Graph& gr, const MoveSweep& s, const MoveState& st,
                                            const Vertex& x, int32_t old) {
  int32_t choice = old;
  if (x.a != x.b && x.tm > 0.0) {
    Row r;
    load_row(p, gr, x.v, x.a, x.b, r);
    const double sig_old_excl = load_now(s.sigma + old) - x.kv;
    float k_old = 0.0f;
    int n = 0;
    if constexpr (FIRST) {
#pragma unroll
      for (int i = 0; i < ROW_PER; ++i) r.ok[i] = r.ok[i] && (r.u[i] > old ? 1 : 0) == st.up;
    } else {
      int32_t c[ROW_PER];
#pragma unroll
      for (int i = 0; i < ROW_PER; ++i) {
        c[i] = old;
        if (r.ok[i]) c[i] = s.lin[r.u[i]];
      }
      double own = 0.0;
#pragma unroll
      for (int i = 0; i < ROW_PER; ++i) {
        own += r.ok[i] && c[i] == old ? (double)r.w[i] : 0.0;
        r.ok[i] = c[i] != old && (c[i] > old ? 1 : 0) == st.up;  // the others are no candidates
      }
      k_old = (float)p.sum(own);
      n = fill_table(p, r, c);
    }
    const double gain = (double)s.resolution * x.kv;
    const float jitter = (rand_uniform(x.salt, 0u, (uint32_t)s.sweep, s.seed) - 0.5f) * 1e-9f;
    uint64_t mine = 0;
    int32_t mine_c = old;
    each_candidate<P, FIRST>(p, r, n, s.sigma, [&](int32_t c, float kn, double sg) {
      const double dq = ((double)kn - (double)k_old) * x.scale.x + gain * (sig_old_excl - sg) * x.scale.y;
      const uint64_t key = pack((float)dq + jitter, cand_pref(c));
      if (key > mine) {
        mine = key;
        mine_c = c;
      }
    });
    const uint64_t best = p.max(mine);
    if (best > pack(0.0f, STAY_PREF)) choice = p.of(best, mine, mine_c);
  }
  if (p.tid() == 0) finish_move(s, x.v, choice, x.kv);
  return choice != old;
}

// A workgroup's vertices: chunks of GROUPS, strided over the workgroups of its
// XCD, each XCD (workgroups run on the eight in turn; the grid is a multiple of
// eight) a contiguous run, so that a graph's labels and totals stay in one L2.
// The half waves go through their chunks without waiting for each other: with
// a workgroup per chunk, the LDS of the waves that were done stayed taken until
// the slowest was (20 of 32 waves a compute unit at work).
//
// Below two chunks a workgroup the long rows take LONG_BLOCKS workgroups of
// their own in the same launch (all sweeps of eight 2k graphs, 2,000 chunks:
// 577 us against 669 with every workgroup taking both); above, all workgroups
// share both (32 8k graphs, whose levels have 32,800 down to 7,100 chunks: all
// sweeps 1,885 us with the line here, 1,964 with it at 16,384 chunks).
struct Share {
  int32_t at, end, step;
};
struct Split {
  unsigned grid;
  int32_t long_blocks;  // workgroups that take long rows: the first ones
  int32_t first;        // workgroups before the first that takes chunks
};
inline Split split_of(int32_t V) {
  const int32_t chunks = (V + GROUPS - 1) / GROUPS;
  if (chunks >= 2 * SWEEP_BLOCKS) return Split{SWEEP_BLOCKS, SWEEP_BLOCKS, 0};
  return Split{(unsigned)(LONG_BLOCKS + (chunks + 7) / 8 * 8), LONG_BLOCKS, LONG_BLOCKS};
}
// A wave's mids: a run of the list (about ascending) for each XCD, as the chunks.
__device__ __forceinline__ Share mid_share(const RowLists& l) {
  if ((int32_t)blockIdx.x >= l.long_blocks) return Share{0, 0, 1};
  const int64_t mids = l.counts[0];
  const int32_t x = blockIdx.x & 7, waves = HUB_THREADS / 64;
  return Share{(int32_t)(mids * x / 8) + (int32_t)(blockIdx.x >> 3) * waves + (int32_t)(threadIdx.x >> 6),
               (int32_t)(mids * (x + 1) / 8), (l.long_blocks >> 3) * waves};
}
__device__ __forceinline__ Share share_of(int32_t V, int32_t first) {
  if ((int32_t)blockIdx.x < first) return Share{0, 0, 1};
  const int64_t chunks = (V + GROUPS - 1) / GROUPS;
  const int32_t b = (int32_t)blockIdx.x - first, x = b & 7;
  return Share{(int32_t)(chunks * x / 8) + (b >> 3), (int32_t)(chunks * (x + 1) / 8), ((int32_t)gridDim.x - first) >> 3};
}

// A sweep after local moving has ended (every vertex stays): what it was given,
// handed on.  Refinement needs nothing handed on: nothing reads the pairs and
// totals of its last sweeps, and the labels are in place.
__device__ __forceinline__ void hand_on(const MoveSweep& s, int32_t V) {
  const int32_t step = (int32_t)(gridDim.x * HUB_THREADS);
  for (int32_t v = (int32_t)(blockIdx.x * HUB_THREADS + threadIdx.x); v < V; v += step) {
    s.lout[v] = s.lin[v];
    s.next[v] = s.sigma[v];
    s.clear[v] = 0.0;
  }
}

template <bool FIRST>
__global__ __launch_bounds__(HUB_THREADS, 8) void local_moving_kernel(Graph gr, MoveSweep s,
                                                                      RowLists l) {
  __shared__ SweepShared sh;  // (FIRST leaves the table out of use; its occupancy is full all the same)
  bool moved = false;
  const MoveState st = move_state(s.ctl, s.sweep);
  if (!FIRST && st.done) {
    hand_on(s, gr.V);
    return;
  }
  if constexpr (!FIRST) clear_tables(sh);
  const int32_t hubs = l.counts[1];
  const Share share = mid_share(l);
  for (int32_t i = l.start(blockIdx.x); i < hubs; i += l.long_blocks) {
    const Vertex x = load_vertex(gr, s.lc, l.rows[gr.V - 1 - i]);
    moved |= move_vertex<Workgroup, FIRST>(Workgroup(sh), gr, s, st, x, FIRST ? x.v : s.lin[x.v]);
    __syncthreads();  // the next vertex takes the table
  }
  for (int32_t i = share.at; i < share.end; i += share.step) {
    const Vertex x = load_vertex(gr, s.lc, l.rows[i]);
    moved |= move_vertex<Wave, FIRST>(Wave(sh), gr, s, st, x, FIRST ? x.v : load_now(s.lin + x.v));
  }
  const Share mine = share_of(gr.V, l.first);
  const HalfWave p(sh);
  for (int32_t c = mine.at; c < mine.end; c += mine.step) {
    const int32_t v = c * GROUPS + (int32_t)(threadIdx.x >> 5);
    if (v >= gr.V) break;
    const Vertex x = load_vertex(gr, s.lc, v);
    const int32_t old = FIRST ? v : load_now(s.lin + v);
    if (x.b - x.a <= SMALL_ROW) moved |= move_vertex<HalfWave, FIRST>(p, gr, s, st, x, old);
  }
  mark_moved(mark_slot(s.ctl, true, s.sweep), moved);
}

// Refinement: a vertex proposes a community inside its parent community (x of
// the label pairs; y is its community), then the proposals' independent set
// commits.  mover[v] holds the parent of a vertex that wants to move, -1 of
// the others: one gather per neighbour tells the commit all it needs.
struct RefineSweep {
  const double* sigma;
  const double* parent_sigma;
  double* next;
  double* clear;
  const int32_t* parent;  // read in a FIRST sweep in place of the pairs
  const int2* lin;
  int2* lout;
  int32_t* labels;        // the communities alone
  int32_t* prop;
  int32_t* mover;
  int32_t* ctl;
  int32_t sweep;
  float resolution;
  float inv_theta;
  int boltzmann;
  uint32_t seed;
  LevelConst lc;
};

template <bool FIRST>
__device__ __forceinline__ int2 refine_self(const RefineSweep& s, int32_t v) {
  if constexpr (FIRST) return int2{load_now(s.parent + v), v};
  return load_now(s.lin + v);
}

// e < x / tm, without the division (some 35 issue slots) unless they are close.
__device__ __forceinline__ bool below_quotient(double e, double x, double tm) {
  const double lhs = e * tm, slack = fabs(x) * 1e-12;
  if (lhs > x + slack) return false;
  if (lhs < x - slack) return true;
  return e < x / tm;
}

template <class P, bool FIRST>
__device__ __forceinline__ void propose_vertex(const P& p, const Graph& gr, const RefineSweep& s, const Vertex& x,
                                               int2 self) {
  const int32_t pv = self.x, old = self.y;
  int32_t choice = old;
  if (x.a != x.b && x.tm > 0.0) {
    Row r;
    load_row(p, gr, x.v, x.a, x.b, r);
    double vol_minus = load_now(s.parent_sigma + pv) - x.kv;
    if (vol_minus < 0.0) vol_minus = 0.0;
    const double sig_old_excl = load_now(s.sigma + old) - x.kv;
    int32_t c[ROW_PER];
    double own = 0.0, e_sum = 0.0;
#pragma unroll
    for (int i = 0; i < ROW_PER; ++i) {
      int2 q{-1, old};
      if (r.ok[i]) {
        if constexpr (FIRST) q = int2{s.parent[r.u[i]], r.u[i]};
        else q = s.lin[r.u[i]];
      }
      r.ok[i] = q.x == pv;  // (parents are vertices, never -1)
      c[i] = q.y;
    }
#pragma unroll
    for (int i = 0; i < ROW_PER; ++i) e_sum += r.ok[i] ? (double)r.w[i] : 0.0;
    e_sum = p.sum(e_sum);
    if (!below_quotient((double)(float)e_sum, (double)s.resolution * x.kv * vol_minus, x.tm)) {
      // {v} is well connected to its parent community
      float k_old = 0.0f;
      int n = 0;
      if constexpr (!FIRST) {
#pragma unroll
        for (int i = 0; i < ROW_PER; ++i) {
          own += r.ok[i] && c[i] == old ? (double)r.w[i] : 0.0;
          r.ok[i] = r.ok[i] && c[i] != old;
        }
        k_old = (float)p.sum(own);
        n = fill_table(p, r, c);
      }
      const double gain = (double)s.resolution * x.kv;
      uint64_t mine = 0;
      int32_t mine_c = old;
      each_candidate<P, FIRST>(p, r, n, s.sigma, [&](int32_t cand, float kn, double sg) {
        const double dq = ((double)kn - (double)k_old) * x.scale.x + gain * (sig_old_excl - sg) * x.scale.y;
        if (dq < 0.0) return;
        const float score = s.boltzmann
            ? (float)(dq * (double)s.inv_theta)
                  + gumbel(rand_uniform_pair(x.salt, (uint32_t)cand, 1u, (uint32_t)s.sweep, s.seed))
            : (float)dq;
        const uint64_t key = pack(score, cand_pref(cand));
        if (key > mine) {
          mine = key;
          mine_c = cand;
        }
      });
      const uint64_t best = p.max(mine);
      const float stay = s.boltzmann
          ? gumbel(rand_uniform_pair(x.salt, (uint32_t)old, 1u, (uint32_t)s.sweep, s.seed))
          : 0.0f;
      if (best > pack(stay, STAY_PREF)) choice = p.of(best, mine, mine_c);
    }
  }
  if (p.tid() == 0) {
    s.prop[x.v] = choice;
    s.mover[x.v] = choice != old ? pv : -1;
  }
}

template <bool FIRST>
__global__ __launch_bounds__(HUB_THREADS, 8) void refine_propose_kernel(Graph gr, RefineSweep s,
                                                                        RowLists l) {
  __shared__ SweepShared sh;
  if (refine_done(s.ctl, s.sweep)) return;
  if constexpr (!FIRST) clear_tables(sh);
  const int32_t hubs = l.counts[1];
  const Share share = mid_share(l);
  for (int32_t i = l.start(blockIdx.x); i < hubs; i += l.long_blocks) {
    const Vertex x = load_vertex(gr, s.lc, l.rows[gr.V - 1 - i]);
    propose_vertex<Workgroup, FIRST>(Workgroup(sh), gr, s, x, refine_self<FIRST>(s, x.v));
    __syncthreads();
  }
  for (int32_t i = share.at; i < share.end; i += share.step) {
    const Vertex x = load_vertex(gr, s.lc, l.rows[i]);
    propose_vertex<Wave, FIRST>(Wave(sh), gr, s, x, refine_self<FIRST>(s, x.v));
  }
  const Share mine = share_of(gr.V, l.first);
  const HalfWave p(sh);
  for (int32_t c = mine.at; c < mine.end; c += mine.step) {
    const int32_t v = c * GROUPS + (int32_t)(threadIdx.x >> 5);
    if (v >= gr.V) break;
    const Vertex x = load_vertex(gr, s.lc, v);
    const int2 self = refine_self<FIRST>(s, v);
    if (x.b - x.a <= SMALL_ROW) propose_vertex<HalfWave, FIRST>(p, gr, s, x, self);
  }
}

// A mover commits unless a moving neighbour in its parent community outranks
// it on (rank, id) (refinement.cu:263-300); the rank is the neighbour's hash,
// computed where it is needed.
struct Commit {
  int32_t v, a, b, to, wants;
  int2 self;
  double kv;
};
template <bool FIRST>
__device__ __forceinline__ Commit load_commit(const Graph& gr, const RefineSweep& s, int32_t v) {
  Commit x;
  x.v = v;
  x.a = load_now(gr.beg + v);
  x.b = load_now(gr.end + v);
  x.wants = load_now(s.mover + v);
  x.to = load_now(s.prop + v);
  x.self = refine_self<FIRST>(s, v);
  x.kv = load_now(gr.k_v + v);
  return x;
}

// Returns whether the vertex moves.
template <class P>
__device__ __forceinline__ bool commit_vertex(const P& p, const Graph& gr, const RefineSweep& s, const Commit& x) {
  const bool wants = x.wants >= 0;
  bool lost = false;
  if (wants) {
    const int32_t g = s.lc.graph_of.of(x.v);
    const uint32_t key = (1u << 16) | (uint32_t)s.sweep, gh = pcg_hash((uint32_t)g);
    const uint32_t rv = mix_salt(pcg_hash(gh ^ (uint32_t)x.v), key, s.seed);
    for (int32_t e0 = x.a; e0 < x.b; e0 += ROW_PER * P::N) {
      int32_t u[ROW_PER], m[ROW_PER];
#pragma unroll
      for (int i = 0; i < ROW_PER; ++i) {
        const int32_t e = e0 + i * P::N + p.tid();
        u[i] = x.v;
        if (e < x.b) u[i] = gr.col[e];
      }
#pragma unroll
      for (int i = 0; i < ROW_PER; ++i) {
        m[i] = -1;
        if (u[i] != x.v) m[i] = s.mover[u[i]];
      }
#pragma unroll
      for (int i = 0; i < ROW_PER; ++i) {
        if (m[i] == x.self.x) {
          const int32_t gu = s.lc.graph_of.of(u[i]);
          const uint32_t ru = mix_salt(pcg_hash((gu == g ? gh : pcg_hash((uint32_t)gu)) ^ (uint32_t)u[i]), key, s.seed);
          lost = lost || ru > rv || (ru == rv && u[i] > x.v);
        }
      }
    }
    lost = p.any(lost);
  }
  const int32_t label = wants && !lost ? x.to : x.self.y;
  if (p.tid() == 0) {
    s.lout[x.v] = int2{x.self.x, label};
    s.labels[x.v] = label;
    s.clear[x.v] = 0.0;
    if (x.kv != 0.0) unsafeAtomicAdd(s.next + label, x.kv);
  }
  return label != x.self.y;
}

template <bool FIRST>
__global__ __launch_bounds__(HUB_THREADS, 8) void refine_commit_kernel(Graph gr, RefineSweep s,
                                                                       RowLists l) {
  __shared__ SweepShared sh;  // (the table stays out of use)
  if (refine_done(s.ctl, s.sweep)) return;
  bool moved = false;
  const int32_t hubs = l.counts[1], long_rows = hubs + l.counts[2];
  const Share share = mid_share(l);
  for (int32_t i = l.start(blockIdx.x); i < long_rows; i += l.long_blocks)
    moved |= commit_vertex(Workgroup(sh), gr, s,
                  load_commit<FIRST>(gr, s, i < hubs ? l.rows[gr.V - 1 - i] : l.giants[i - hubs]));
  for (int32_t i = share.at; i < share.end; i += share.step)
    moved |= commit_vertex(Wave(sh), gr, s, load_commit<FIRST>(gr, s, l.rows[i]));
  const Share mine = share_of(gr.V, l.first);
  const HalfWave p(sh);
  for (int32_t c = mine.at; c < mine.end; c += mine.step) {
    const int32_t v = c * GROUPS + (int32_t)(threadIdx.x >> 5);
    if (v >= gr.V) break;
    const Commit x = load_commit<FIRST>(gr, s, v);
    if (x.b - x.a <= SMALL_ROW) moved |= commit_vertex(p, gr, s, x);
  }
  mark_moved(mark_slot(s.ctl, false, s.sweep), moved);
}

// Test hook: raises the overflow word as a broken local-moving table would.
__global__ void raise_overflow_kernel(int32_t* __restrict__ ctl) {
  if (threadIdx.x == 0) ctl[CTL_OVERFLOW] = 1;
}

// Label pairs of singletons, for graphs whose first refinement sweep reads them.
__global__ void pair_init_kernel(const int32_t* __restrict__ parent, int32_t V, int2* __restrict__ pairs) {
  const int32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < V) pairs[v] = int2{parent[v], v};
}

// Rows longer than GIANT_MIN: one 1024-thread workgroup per vertex.  All
// threads insert the row's neighbour communities into a GIANT_SLOTS-slot LDS
// table (sum of weights in f64, first row position by atomic min); when more
// than TABLE_CAP communities appear, a binary search on the first positions
// keeps exactly the TABLE_CAP that appear first along the row (the rule of
// the per-wave tables).  The row is walked in position order, GIANT_THREADS
// entries at a time, and no community is inserted once TABLE_CAP are held, so
// the table never holds more than 2 x TABLE_CAP - 1.  The candidates are
// scored across the workgroup.  (giant_table reports an overflow only if the
// table bound above were broken; the vertex then stays where it is.)
struct GiantShared {
  int32_t c[GIANT_SLOTS];
  double s[GIANT_SLOTS];
  int32_t first[GIANT_SLOTS];
  uint64_t best[GIANT_THREADS / 64];
  int32_t best_c[GIANT_THREADS / 64];
  double red[GIANT_THREADS / 64];
  int32_t n, overflow, count, k_old_slot;
};

__device__ inline double block_sum_giant(double x, GiantShared& sh) {
  x = wave_sum_f64(x);
  if (lane() == 0) sh.red[threadIdx.x >> 6] = x;
  __syncthreads();
  double t = 0.0;
  for (int i = 0; i < GIANT_THREADS / 64; ++i) t += sh.red[i];
  __syncthreads();
  return t;
}

// Returns false when the table overflowed (caller falls back); on success
// *thr bounds the kept first positions and *e_sum is the admitted weight.
// community_of(u): the neighbour's community, -1 when the entry does not count.
template <class Of>
__device__ bool giant_table(const Graph& gr, Of community_of, int32_t v, int32_t a, int32_t b, GiantShared& sh,
                            int32_t* thr, double* e_sum) {
  const int tid = threadIdx.x;
  for (int j = tid; j < GIANT_SLOTS; j += GIANT_THREADS) {
    sh.c[j] = -1;
    sh.s[j] = 0.0;
    sh.first[j] = 0x7FFFFFFF;
  }
  if (tid == 0) {
    sh.n = 0;
    sh.overflow = 0;
  }
  __syncthreads();
  double e_acc = 0.0;
  bool capped = false;  // TABLE_CAP communities held: later ones cannot be among the first TABLE_CAP
  for (int32_t e0 = a; e0 < b; e0 += GIANT_THREADS) {
    const int32_t e = e0 + tid;
    if (e < b) {
      const int32_t u = gr.col[e];
      const int32_t c = u != v ? community_of(u) : -1;
      if (c >= 0) {
        const float w = gr.wt[e];
        e_acc += (double)w;
        uint32_t h = pcg_hash((uint32_t)c) & (GIANT_SLOTS - 1);
        int probes = 0;
        bool placed = false;
        while (probes++ < GIANT_SLOTS) {
          const int32_t cur = __hip_atomic_load(sh.c + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          if (cur == c) {
            placed = true;
            break;
          }
          if (cur == -1) {
            if (capped) break;  // not held: appears after the first TABLE_CAP communities
            const int32_t prev = atomicCAS(sh.c + h, -1, c);
            if (prev == -1) atomicAdd(&sh.n, 1);
            if (prev == -1 || prev == c) {
              placed = true;
              break;
            }
          }
          h = (h + 1) & (GIANT_SLOTS - 1);
        }
        if (placed) {
          unsafeAtomicAdd(sh.s + h, (double)w);
          atomicMin(sh.first + h, e);
        } else if (!capped) {
          sh.overflow = 1;  // unreachable: at most 2 x TABLE_CAP - 1 entries are ever inserted
        }
      }
    }
    __syncthreads();
    capped = sh.n >= TABLE_CAP;
    __syncthreads();
  }
  __syncthreads();
  *e_sum = block_sum_giant(e_acc, sh);
  if (sh.overflow) return false;
  int32_t t = 0x7FFFFFFF;
  if (sh.n > TABLE_CAP) {  // smallest t with TABLE_CAP first positions below it
    int32_t lo = a, hi = b;
    while (lo < hi) {
      const int32_t mid = lo + (hi - lo) / 2;
      if (tid == 0) sh.count = 0;
      __syncthreads();
      int cnt = 0;
      for (int j = tid; j < GIANT_SLOTS; j += GIANT_THREADS) cnt += sh.first[j] < mid + 1;
      if (cnt) atomicAdd(&sh.count, cnt);
      __syncthreads();
      if (sh.count >= TABLE_CAP) hi = mid;
      else lo = mid + 1;
      __syncthreads();
    }
    t = lo + 1;
  }
  *thr = t;
  return true;
}

// Block-wide max of packed candidates; every thread gets the winner.
__device__ inline int32_t giant_pick(uint64_t mine, int32_t mine_c, uint64_t stay, int32_t old, GiantShared& sh) {
  const uint64_t wbest = wave_max_u64(mine);
  const int32_t wc = __shfl(mine_c, first_lane(__ballot(mine == wbest)));
  if (lane() == 0) {
    sh.best[threadIdx.x >> 6] = wbest;
    sh.best_c[threadIdx.x >> 6] = wc;
  }
  __syncthreads();
  uint64_t best = 0;
  int32_t c = old;
  for (int i = 0; i < GIANT_THREADS / 64; ++i)
    if (sh.best[i] > best) {
      best = sh.best[i];
      c = sh.best_c[i];
    }
  __syncthreads();
  return best > stay ? c : old;
}

__device__ float giant_k_old(GiantShared& sh, int32_t old, int32_t thr) {
  if (threadIdx.x == 0) sh.k_old_slot = -1;
  __syncthreads();
  for (int j = threadIdx.x; j < GIANT_SLOTS; j += GIANT_THREADS)
    if (sh.c[j] == old && sh.first[j] < thr) sh.k_old_slot = j;
  __syncthreads();
  const int32_t slot = sh.k_old_slot;
  return slot >= 0 ? (float)sh.s[slot] : 0.0f;
}

template <bool FIRST>
__global__ __launch_bounds__(GIANT_THREADS) void local_moving_giant_kernel(Graph gr, MoveSweep s,
                                                                           RowLists l) {
  __shared__ GiantShared sh;
  const int32_t count = l.counts[2];
  const MoveState st = move_state(s.ctl, s.sweep);
  if (st.done) return;  // (handed on with the other rows)
  for (int32_t i = blockIdx.x; i < count; i += gridDim.x) {
    const int32_t v = l.giants[i];
    const int32_t old = FIRST ? v : s.lin[v];
    const int32_t g = v / gr.S;
    const double tm = gr.two_m[g];
    const double kv = gr.k_v[v];
    if (!(tm > 0.0)) {
      if (threadIdx.x == 0) finish_move(s, v, old, kv);
      continue;
    }
    const int32_t a = gr.beg[v], b = gr.end[v];
    int32_t thr;
    double e_sum;
    if (!giant_table(gr, [&](int32_t u) { return FIRST ? u : s.lin[u]; }, v, a, b, sh, &thr, &e_sum)) {  // cannot happen
      if (threadIdx.x == 0) {
        finish_move(s, v, old, kv);  // stay, flagged
        s.ctl[CTL_OVERFLOW] = 1;
      }
      __syncthreads();
      continue;
    }
    const float k_old = giant_k_old(sh, old, thr);
    const double m_g = 0.5 * tm;
    const double inv_m = 1.0 / m_g;
    const double inv_2m2 = 1.0 / (2.0 * m_g * m_g);
    const double sig_old_excl = s.sigma[old] - kv;
    const float jitter = (rand_uniform(s.lc.salt[v], 0u, (uint32_t)s.sweep, s.seed) - 0.5f) * 1e-9f;
    uint64_t mine = 0;
    int32_t mine_c = old;
    for (int j = threadIdx.x; j < GIANT_SLOTS; j += GIANT_THREADS) {
      const int32_t c = sh.c[j];
      if (c < 0 || sh.first[j] >= thr || c == old || (c > old ? 1 : 0) != st.up) continue;
      const float kn = (float)sh.s[j];
      const double dq = ((double)kn - (double)k_old) * inv_m
                        + (double)s.resolution * kv * (sig_old_excl - s.sigma[c]) * inv_2m2;
      const float dqf = (float)dq + jitter;
      const uint64_t p = pack(dqf, cand_pref(c));
      if (p > mine) {
        mine = p;
        mine_c = c;
      }
    }
    const int32_t choice = giant_pick(mine, mine_c, pack(0.0f, STAY_PREF), old, sh);
    if (threadIdx.x == 0) finish_move(s, v, choice, kv);
    if (threadIdx.x < 64) mark_moved(mark_slot(s.ctl, true, s.sweep), choice != old);
  }
}

template <bool FIRST>
__global__ __launch_bounds__(GIANT_THREADS) void refine_propose_giant_kernel(Graph gr, RefineSweep s,
                                                                             RowLists l) {
  __shared__ GiantShared sh;
  if (refine_done(s.ctl, s.sweep)) return;
  const int32_t count = l.counts[2];
  for (int32_t i = blockIdx.x; i < count; i += gridDim.x) {
    const int32_t v = l.giants[i];
    const int32_t g = v / gr.S;
    int2 self;
    if constexpr (FIRST) self = int2{s.parent[v], v};
    else self = s.lin[v];
    const int32_t pv = self.x, old = self.y;
    const double tm = gr.two_m[g];
    auto propose = [&](int32_t choice) {
      if (threadIdx.x == 0) {
        s.prop[v] = choice;
        s.mover[v] = choice != old ? pv : -1;
      }
    };
    if (!(tm > 0.0)) {
      propose(old);
      continue;
    }
    const int32_t a = gr.beg[v], b = gr.end[v];
    int32_t thr;
    double e_sum;
    auto community_of = [&](int32_t u) {
      if constexpr (FIRST) {
        return s.parent[u] == pv ? u : -1;
      } else {
        const int2 q = s.lin[u];
        return q.x == pv ? q.y : -1;
      }
    };
    if (!giant_table(gr, community_of, v, a, b, sh, &thr, &e_sum)) {  // cannot happen: stay, flagged
      propose(old);
      if (threadIdx.x == 0) s.ctl[CTL_OVERFLOW] = 1;
      __syncthreads();
      continue;
    }
    const double kv = gr.k_v[v];
    double vol_minus = s.parent_sigma[pv] - kv;
    if (vol_minus < 0.0) vol_minus = 0.0;
    const double bound = (double)s.resolution * kv * vol_minus / tm;
    if ((double)(float)e_sum < bound) {  // {v} is not well connected to its parent community
      propose(old);
      __syncthreads();
      continue;
    }
    const float k_old = giant_k_old(sh, old, thr);
    const double m_g = 0.5 * tm;
    const double inv_m = 1.0 / m_g;
    const double inv_2m2 = 1.0 / (2.0 * m_g * m_g);
    const double sig_old_excl = s.sigma[old] - kv;
    uint64_t mine = 0;
    int32_t mine_c = old;
    for (int j = threadIdx.x; j < GIANT_SLOTS; j += GIANT_THREADS) {
      const int32_t c = sh.c[j];
      if (c < 0 || sh.first[j] >= thr || c == old) continue;
      const float kn = (float)sh.s[j];
      const double dq = ((double)kn - (double)k_old) * inv_m
                        + (double)s.resolution * kv * (sig_old_excl - s.sigma[c]) * inv_2m2;
      if (dq < 0.0) continue;
      const float score = s.boltzmann
          ? (float)(dq * (double)s.inv_theta)
                + gumbel(rand_uniform_pair(s.lc.salt[v], (uint32_t)c, 1u, (uint32_t)s.sweep, s.seed))
          : (float)dq;
      const uint64_t p = pack(score, cand_pref(c));
      if (p > mine) {
        mine = p;
        mine_c = c;
      }
    }
    const float stay = s.boltzmann
        ? gumbel(rand_uniform_pair(s.lc.salt[v], (uint32_t)old, 1u, (uint32_t)s.sweep, s.seed))
        : 0.0f;
    const int32_t choice = giant_pick(mine, mine_c, pack(stay, STAY_PREF), old, sh);
    propose(choice);
  }
}


// q_v = in(v) / 2m - gamma k_v Sigma[c_v] / (4 m^2); Q_g is their sum over
// the graph (helpers.cu:41-78).
__global__ __launch_bounds__(LTHREADS) void modularity_kernel(Graph gr, const int32_t* __restrict__ labels,
                                                              const double* __restrict__ sigma, float resolution,
                                                              double* __restrict__ q_v) {
  const int32_t v = blockIdx.x * LWAVES + (threadIdx.x >> 6);
  if (v >= gr.V) return;
  const int32_t g = v / gr.S;
  const double tm = gr.two_m[g];
  if (!(tm > 0.0)) {
    if (lane() == 0) q_v[v] = 0.0;
    return;
  }
  const int32_t cv = labels[v];
  const int32_t a = gr.beg[v], b = gr.end[v];
  double in_sum = 0.0;
  for (int32_t e = a + lane(); e < b; e += 64)
    if (labels[gr.col[e]] == cv) in_sum += (double)gr.wt[e];
  in_sum = wave_sum_f64(in_sum);
  if (lane() == 0) {
    const double m_g = 0.5 * tm;
    q_v[v] = in_sum / tm - (double)resolution * (gr.k_v[v] * sigma[cv]) / (4.0 * m_g * m_g);
  }
}

// A flagged table overflow turns every graph's modularity into NaN, which the
// host checks: the labels of such a call are not to be trusted.
__global__ void overflow_mark_kernel(const int32_t* __restrict__ ctl, int32_t G, double* __restrict__ modularity) {
  const int32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g < G && ctl[CTL_OVERFLOW] != 0) modularity[g] = __builtin_nan("");
}

__global__ void finish_kernel(const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ result, int32_t V,
                              int32_t* __restrict__ labels) {
  const int32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < V) labels[v] = row_ptr[v] == row_ptr[v + 1] ? -1 : result[v];
}

// ----------------------------------------------------------------- aggregation / densify
__global__ void remap_kernel(const int32_t* __restrict__ src, const int32_t* __restrict__ dst,
                             const float* __restrict__ w, const int32_t* __restrict__ labels, int64_t E,
                             int32_t Vs, int bits, uint64_t* __restrict__ keys, float* __restrict__ vals) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= E) return;
  int32_t s = labels[src[i]], t = labels[dst[i]];
  const int32_t lo = s < t ? s : t, hi = s < t ? t : s;
  const bool ok = lo >= 0 && hi < Vs;
  keys[i] = ok ? ((uint64_t)lo << bits) | (uint64_t)hi : ((uint64_t)Vs << bits);
  vals[i] = ok ? w[i] : 0.0f;
}

__global__ void unpack_kernel(const uint64_t* __restrict__ keys, int64_t E, int bits,
                              const int64_t* __restrict__ count, int32_t* __restrict__ out_src,
                              int32_t* __restrict__ out_dst) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= *count) return;
  const uint64_t k = keys[i];
  out_src[i] = (int32_t)(k >> bits);
  out_dst[i] = (int32_t)(k & (((uint64_t)1 << bits) - 1));
}

// Edges with an endpoint label outside [0, Vs) carry the sentinel key, which
// sorts last: drop that run from the count.
__global__ void count_fix_kernel(const uint64_t* __restrict__ keys, int32_t Vs, int bits, int64_t* __restrict__ count) {
  if (threadIdx.x != 0) return;
  const int64_t n = *count;
  if (n > 0 && (keys[n - 1] >> bits) >= (uint64_t)Vs) *count = n - 1;
}

__global__ void flag_zero_kernel(int32_t* __restrict__ flags, int32_t V) {
  const int32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < V) flags[v] = 0;
}

// Labels below zero stand for the vertex itself; labels outside the vertex's
// graph are ignored (their vertices get rank -1 in the apply step).
__device__ inline int32_t own_label(const int32_t* labels, int32_t v, int32_t S) {
  const int32_t l = labels[v] < 0 ? v : labels[v];
  return (l / S == v / S) ? l : -1;
}

__global__ void flag_mark_kernel(const int32_t* __restrict__ labels, int32_t V, int32_t S,
                                 int32_t* __restrict__ flags) {
  const int32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V) return;
  const int32_t l = own_label(labels, v, S);
  if (l >= 0) flags[l] = 1;
}

__global__ void densify_count_kernel(const int32_t* __restrict__ flags, const int32_t* __restrict__ scan, int32_t G,
                                     int32_t S, int32_t* __restrict__ counts) {
  const int32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g < G) {
    const int32_t last = (g + 1) * S - 1;
    counts[g] = scan[last] + flags[last] - scan[g * S];
  }
}

__global__ void densify_apply_kernel(const int32_t* __restrict__ labels, const int32_t* __restrict__ scan, int32_t V,
                                     int32_t S, int32_t new_S, int32_t* __restrict__ dense) {
  const int32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V) return;
  const int32_t g = v / S;
  const int32_t l = own_label(labels, v, S);
  dense[v] = l < 0 ? -1 : scan[l] - scan[g * S] + g * new_S;
}

// ----------------------------------------------------------------- modularity of a labelled edge list
__device__ inline double block_sum_f64(double x, double* part) {  // 256 threads
  x = wave_sum_f64(x);
  if (lane() == 0) part[threadIdx.x >> 6] = x;
  __syncthreads();
  return part[0] + part[1] + part[2] + part[3];
}

__global__ void mod_zero_kernel(double* __restrict__ k, double* __restrict__ sig, int32_t V,
                                double* __restrict__ acc) {
  const int32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < V) {
    k[v] = 0.0;
    sig[v] = 0.0;
  }
  if (v < 4) acc[v] = 0.0;
}

__global__ __launch_bounds__(256) void mod_edge_kernel(const int32_t* __restrict__ src,
                                                       const int32_t* __restrict__ dst, const float* __restrict__ w,
                                                       int64_t E, const int32_t* __restrict__ labels, int32_t V,
                                                       double* __restrict__ k, double* __restrict__ acc) {
  __shared__ double part[4];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double in = 0.0, xs = 0.0;
  int32_t a = -1;
  if (i < E) {
    const int32_t s0 = src[i], b = dst[i];
    if (s0 >= 0 && s0 < V && b >= 0 && b < V) {
      const double x = (double)w[i];
      a = s0;
      xs = x;
      unsafeAtomicAdd(k + b, x);
      if (labels[s0] == labels[b]) in = x;
    }
  }
  // Source ends: sum runs of equal source within the wave (edge lists come
  // sorted by source, so a hub's edges arrive together), one atomic per run.
  const int ln = lane();
  const int32_t prev_a = __shfl_up(a, 1);
  const int32_t next_a = __shfl_down(a, 1);
  bool h = ln == 0 || prev_a != a;  // a run starts here
  for (int o = 1; o < 64; o <<= 1) {
    const double y = __shfl_up(xs, o);
    const bool hy = __shfl_up(h ? 1 : 0, o) != 0;
    if (ln >= o) {
      if (!h) xs += y;
      h = h || hy;
    }
  }
  if (a >= 0 && (ln == 63 || next_a != a)) unsafeAtomicAdd(k + a, xs);
  in = block_sum_f64(in, part);
  if (threadIdx.x == 0 && in != 0.0) unsafeAtomicAdd(acc, in);
}

__global__ __launch_bounds__(256) void mod_sigma_kernel(const int32_t* __restrict__ labels,
                                                        const double* __restrict__ k, int32_t V,
                                                        double* __restrict__ sig, double* __restrict__ acc) {
  __shared__ double part[4];
  const int32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  double kv = 0.0;
  if (v < V) {
    kv = k[v];
    const int32_t l = labels[v];
    if (l >= 0 && l < V && kv != 0.0) unsafeAtomicAdd(sig + l, kv);
  }
  kv = block_sum_f64(kv, part);
  if (threadIdx.x == 0 && kv != 0.0) unsafeAtomicAdd(acc + 1, kv);
}

__global__ __launch_bounds__(256) void mod_square_kernel(const double* __restrict__ sig, int32_t V,
                                                         double* __restrict__ acc) {
  __shared__ double part[4];
  const int32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  double x = v < V ? sig[v] * sig[v] : 0.0;
  x = block_sum_f64(x, part);
  if (threadIdx.x == 0 && x != 0.0) unsafeAtomicAdd(acc + 2, x);
}

__global__ void mod_final_kernel(const double* __restrict__ acc, float resolution, double* __restrict__ out) {
  if (threadIdx.x != 0) return;
  const double two_m = acc[1];
  *out = two_m > 0.0 ? 2.0 * acc[0] / two_m - (double)resolution * acc[2] / (two_m * two_m) : 0.0;
}

// ----------------------------------------------------------------- CSR of a sorted edge list
// Flags of an edge list: [0] an edge leaves its graph or the vertex range,
// [1] the list is not strictly ascending upper-triangular (src, dst).
__global__ __launch_bounds__(ETHREADS) void edge_check_kernel(const int32_t* __restrict__ src,
                                                              const int32_t* __restrict__ dst, int64_t E, int32_t V,
                                                              int32_t S, int32_t* __restrict__ flags) {
  const int64_t i = (int64_t)blockIdx.x * ETHREADS + threadIdx.x;
  bool bad = false, loose = false;
  if (i < E) {
    const int32_t a = src[i], b = dst[i];
    bad = a < 0 || b < 0 || a >= V || b >= V || a / S != b / S;
    loose = a > b;
    if (i > 0) {
      const int32_t pa = src[i - 1], pb = dst[i - 1];
      loose = loose || pa > a || (pa == a && pb >= b);
    }
  }
  if (__ballot(bad) && lane() == 0) flags[0] = 1;
  if (__ballot(loose) && lane() == 0) flags[1] = 1;
}

// start[k] = first i with key[i] >= k, for k in 0..V (keys ascending, above V
// counted as V), by a workgroup of which thread i holds key i (every thread
// calls).  Key i is the first of the ids behind key i - 1; gaps longer than
// SHORT_GAP ids (a short list over many vertices, graphs without edges) are
// listed and filled by the whole workgroup.  With one thread filling them a run
// over 32 graphs of 32,768 vertices, edges in the last alone, took 81 ms, 2.5 so.
constexpr int SHORT_GAP = 16;

__device__ inline void bounds_at(const uint32_t* __restrict__ keys, int64_t i, int64_t n, uint32_t V,
                                 int32_t* __restrict__ start) {
  __shared__ uint3 gaps[ETHREADS + 1];  // first and last id, value (the last key's thread has two)
  __shared__ int listed;
  if (threadIdx.x == 0) listed = 0;
  __syncthreads();
  auto gap = [&](uint32_t first, uint32_t last, int32_t value) {  // ids first..last, none if last < first
    if (last + 1 <= first + SHORT_GAP) {
      for (uint32_t v = first; v <= last; ++v) start[v] = value;
    } else {
      gaps[atomicAdd(&listed, 1)] = uint3{first, last, (uint32_t)value};
    }
  };
  if (i < n) {
    const uint32_t here = min(keys[i], V);
    gap(i == 0 ? 0u : min(keys[i - 1], V) + 1u, here, (int32_t)i);
    if (i == n - 1) gap(here + 1u, V, (int32_t)n);
  }
  __syncthreads();
  for (int g = 0; g < listed; ++g) {
    const uint3 x = gaps[g];
    for (uint32_t v = x.x + threadIdx.x; v <= x.y; v += ETHREADS) start[v] = (int32_t)x.z;
  }
}

// The list's own order gives every vertex its edges to higher ids; the edges
// to lower ids come from a stable sort by dst (self loops, which have no
// second end, sort behind: key V).
__global__ __launch_bounds__(ETHREADS) void upper_bounds_kernel(const int32_t* __restrict__ src,
                                                                const int32_t* __restrict__ dst, int64_t E, int32_t V,
                                                                int32_t* __restrict__ upper,
                                                                uint32_t* __restrict__ keys,
                                                                uint32_t* __restrict__ vals) {
  const int64_t i = (int64_t)blockIdx.x * ETHREADS + threadIdx.x;
  bounds_at(reinterpret_cast<const uint32_t*>(src), i, E, (uint32_t)V, upper);
  if (i >= E) return;
  keys[i] = src[i] == dst[i] ? (uint32_t)V : (uint32_t)dst[i];
  vals[i] = (uint32_t)i;
}

__global__ __launch_bounds__(ETHREADS) void lower_bounds_kernel(const uint32_t* __restrict__ keys, int64_t E, int32_t V,
                                                                int32_t* __restrict__ lower) {
  const int64_t i = (int64_t)blockIdx.x * ETHREADS + threadIdx.x;
  bounds_at(keys, i, E, (uint32_t)V, lower);
}

// Row v: its lower neighbours, then itself and its upper ones.  row_ptr[v] =
// upper[v] + lower[v], so no scan is needed: edge i lands at i + lower[src + 1],
// sorted edge j of dst v at j + upper[v].
__global__ __launch_bounds__(ETHREADS) void csr_fill_kernel(const int32_t* __restrict__ src,
                                                            const int32_t* __restrict__ dst,
                                                            const float* __restrict__ w, int64_t E, int32_t V,
                                                            const int32_t* __restrict__ upper,
                                                            const int32_t* __restrict__ lower,
                                                            const uint32_t* __restrict__ keys,
                                                            const uint32_t* __restrict__ vals,
                                                            int32_t* __restrict__ row_ptr, int32_t* __restrict__ col,
                                                            float* __restrict__ wt) {
  const int64_t i = (int64_t)blockIdx.x * ETHREADS + threadIdx.x;
  if (i <= V) row_ptr[i] = upper[i] + lower[i];
  if (i >= E) return;
  const int32_t s = src[i], d = dst[i];
  const int64_t at = i + lower[s + 1];
  col[at] = d;
  wt[at] = s == d ? 2.0f * w[i] : w[i];
  const uint32_t v = keys[i];
  if (v < (uint32_t)V) {
    const uint32_t e = vals[i];
    const int64_t to = i + upper[v];
    col[to] = src[e];
    wt[to] = w[e];
  }
}

// ----------------------------------------------------------------- contraction of a CSR
// A level's result contracts the graph: row t of the next level holds, per
// neighbouring super-vertex, the summed weight of the entries between its
// members' rows (the row's own id: both directions of its inner edges, i.e.
// twice their weight, as the CSR stores self loops).  Sums are f64, rounded
// once.  Rows stay in the order the table leaves them in: only rows longer
// than GIANT_MIN are walked in neighbour order, and those are summed in dense
// windows, which leave them sorted.
constexpr int AGG_WAVES = 4;
constexpr int AGG_SLOTS = 512;           // LDS table of one wave: 6 KB
constexpr int AGG_SHORT = 448;           // entries of the members' rows that one wave takes (table load 7/8)
constexpr int AGG_FLIGHT = 4;            // entries a thread has in flight
constexpr int AGG_THREADS = 256;         // longer: one workgroup
constexpr int AGG_LONG_SLOTS = 2048;
constexpr int AGG_LONG_MOST = 960;       // neighbours after which a row leaves for the dense windows
static_assert(AGG_LONG_MOST + AGG_FLIGHT * AGG_THREADS < AGG_LONG_SLOTS, "every insert between two checks finds a place");
static_assert(AGG_LONG_MOST <= GIANT_MIN, "rows walked in neighbour order come sorted");
constexpr int AGG_LONG_BLOCKS = 1280;
constexpr int AGG_DENSE_THREADS = 1024;
constexpr int AGG_WINDOW = 16384;        // ids per dense window: 128 KB of f64 sums
constexpr int AGG_DENSE_BLOCKS = 256;

enum { AGG_N_LONG = 0, AGG_N_DENSE = 1, AGG_TICKET = 2, AGG_WORDS = 4 };

// One u64 per super-vertex: members above, entries of their rows below (their
// totals stay below 2^31).
__global__ __launch_bounds__(ETHREADS) void agg_zero_kernel(uint64_t* __restrict__ hist, int32_t n,
                                                            int32_t* __restrict__ lists) {
  const int32_t i = blockIdx.x * ETHREADS + threadIdx.x;
  if (i < n) hist[i] = 0;
  if (i < AGG_WORDS) lists[i] = 0;
}

__global__ __launch_bounds__(ETHREADS) void agg_hist_kernel(const int32_t* __restrict__ dense,
                                                            const int32_t* __restrict__ beg,
                                                            const int32_t* __restrict__ end, int32_t V,
                                                            uint64_t* __restrict__ hist) {
  const int32_t v = blockIdx.x * ETHREADS + threadIdx.x;
  const int32_t s = v < V ? dense[v] : -1;
  int32_t entries = s >= 0 ? end[v] - beg[v] : 0;
  auto add = [&](int members) {
    atomicAdd(reinterpret_cast<unsigned long long*>(hist + s),
              ((unsigned long long)members << 32) | (unsigned long long)(uint32_t)entries);
  };
  const uint64_t same = sharing(s >= 0, s);
  const bool mine = in_mask(same);
  if (s >= 0 && !mine) add(1);
  if (same == 0) return;
  entries = mine ? entries : 0;
  for (int o = 32; o >= 1; o >>= 1) entries += __shfl_xor(entries, o);
  if (lane() == first_lane(same)) add(__popcll(same));
}

__global__ __launch_bounds__(ETHREADS) void agg_fill_kernel(const int32_t* __restrict__ dense, int32_t V,
                                                            const uint64_t* __restrict__ first,
                                                            uint64_t* __restrict__ hist,
                                                            int32_t* __restrict__ members) {
  const int32_t v = blockIdx.x * ETHREADS + threadIdx.x;
  const int32_t s = v < V ? dense[v] : -1;
  // (the members left count down to 1; a super-vertex's lanes that share take theirs in one step)
  auto take = [&](unsigned long long members) {
    return (uint32_t)(atomicAdd(reinterpret_cast<unsigned long long*>(hist + s), ~(members << 32) + 1ull) >> 32);
  };
  const uint64_t same = sharing(s >= 0, s);
  const bool mine = in_mask(same);
  uint32_t left = 0;
  if (s >= 0 && !mine) left = take(1);
  if (same != 0) {
    const int leader = first_lane(same);
    uint32_t first_left = 0;
    if (lane() == leader) first_left = take((unsigned long long)__popcll(same));
    first_left = (uint32_t)__shfl((int)first_left, leader);
    if (mine) left = first_left - (uint32_t)__popcll(same & ((((uint64_t)1) << lane()) - 1));
  }
  if (s >= 0) members[(uint32_t)(first[s] >> 32) + left - 1u] = v;
}

// Row starts of the next level, and the list of rows for a whole workgroup.
__global__ __launch_bounds__(LIST_THREADS) void agg_list_kernel(const uint64_t* __restrict__ first, int32_t Vs,
                                                                int32_t* __restrict__ beg, int32_t* __restrict__ end,
                                                                int32_t* __restrict__ list,
                                                                int32_t* __restrict__ lists) {
  __shared__ int s_n, s_at;
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();
  const int32_t s = blockIdx.x * LIST_THREADS + threadIdx.x;
  uint32_t a = 0, n = 0;
  if (s < Vs) {
    a = (uint32_t)first[s];
    n = (uint32_t)first[s + 1] - a;
    beg[s] = (int32_t)a;
    end[s] = (int32_t)a;  // an empty row; the others store their end when they are summed
  }
  const bool is_long = n > (uint32_t)AGG_SHORT;
  const uint64_t m = __ballot(is_long);
  int b = 0;
  if (lane() == 0 && m) b = atomicAdd(&s_n, __popcll(m));
  b = __shfl(b, 0);
  __syncthreads();
  if (threadIdx.x == 0) s_at = s_n ? atomicAdd(lists + AGG_N_LONG, s_n) : 0;
  __syncthreads();
  if (is_long) list[s_at + b + __popcll(m & ((((uint64_t)1) << lane()) - 1))] = s;
}

struct Contract {
  const int32_t* beg;      // rows of the level that is contracted
  const int32_t* end;
  const int32_t* col;
  const float* wt;
  const int32_t* dense;    // super-vertex of each of its vertices
  const int32_t* members;  // vertices by super-vertex
  const uint64_t* first;   // (first member, first entry) of each super-vertex
  int32_t S;               // super-vertices per graph
  int32_t* out_end;
  int32_t* out_col;
  float* out_wt;
  double* out_k;           // row sums
};

// Calls add(super neighbour, weight) for every entry of the members
// [m0, m1)'s rows, NT threads at a time; pause() after every AGG_FLIGHT x NT
// entries (a true return ends the walk).  Up to NT members are laid end to end
// (s_pre: entries before each, s_beg: its row), so short rows fill the threads.
template <int NT, class Sync, class Scan, class Add, class Pause>
__device__ __forceinline__ void walk_members(const Contract& c, int32_t m0, int32_t m1, int tid, int32_t* s_pre,
                                             int32_t* s_beg, Sync sync, Scan scan, Add add, Pause pause) {
  for (int32_t base = m0; base < m1; base += NT) {
    const int n = min(NT, m1 - base);
    int32_t a = 0, len = 0;
    if (tid < n) {
      const int32_t v = c.members[base + tid];
      a = c.beg[v];
      len = c.end[v] - a;
    }
    int total;
    const int before = scan(len, total);
    s_pre[tid] = before;
    s_beg[tid] = a;
    sync();
    int top = 1;
    while (top < n) top <<= 1;
    bool stop = false;
    for (int q0 = 0; q0 < total && !stop; q0 += AGG_FLIGHT * NT) {
      int32_t e[AGG_FLIGHT], t[AGG_FLIGHT];
      float w[AGG_FLIGHT];
#pragma unroll
      for (int f = 0; f < AGG_FLIGHT; ++f) {
        const int q = min(q0 + f * NT + tid, total - 1);
        int i = 0;  // the last member with s_pre[i] <= q
        for (int h = top >> 1; h >= 1; h >>= 1) {
          if (i + h < n && s_pre[i + h] <= q) i += h;
        }
        e[f] = s_beg[i] + q - s_pre[i];
      }
#pragma unroll
      for (int f = 0; f < AGG_FLIGHT; ++f) {
        t[f] = c.col[e[f]];
        w[f] = c.wt[e[f]];
      }
#pragma unroll
      for (int f = 0; f < AGG_FLIGHT; ++f) t[f] = c.dense[t[f]];
#pragma unroll
      for (int f = 0; f < AGG_FLIGHT; ++f) {
        if (q0 + f * NT + tid < total && t[f] >= 0) add((uint32_t)t[f], w[f]);
      }
      stop = pause();
    }
    sync();  // the next members take the arrays
    if (stop) return;
  }
}

__device__ inline int wave_exclusive_scan(int x, int& total) {
  int inc = x;
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(inc, o);
    if (lane() >= o) inc += y;
  }
  total = __shfl(inc, 63);
  return inc - x;
}

__global__ __launch_bounds__(64 * AGG_WAVES) void agg_short_kernel(Contract c, int32_t Vs) {
  __shared__ uint32_t tab_k[AGG_WAVES][AGG_SLOTS];
  __shared__ double tab_s[AGG_WAVES][AGG_SLOTS];
  __shared__ int32_t pre[AGG_WAVES][64], row[AGG_WAVES][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane();
  const int32_t s = blockIdx.x * AGG_WAVES + wave;
  if (s >= Vs) return;
  const uint64_t f0 = c.first[s], f1 = c.first[s + 1];
  const uint32_t n = (uint32_t)f1 - (uint32_t)f0;
  if (n == 0 || n > (uint32_t)AGG_SHORT) {
    if (n == 0 && ln == 0) c.out_k[s] = 0.0;
    return;
  }
  uint32_t* tk = tab_k[wave];
  double* ts = tab_s[wave];
  const uint32_t size = table_size(min(n, (uint32_t)c.S), AGG_SLOTS);
  for (uint32_t j = ln; j < size; j += 64) {
    tk[j] = EMPTY;
    ts[j] = 0.0;
  }
  wave_lds_sync();
  walk_members<64>(
      c, (int32_t)(f0 >> 32), (int32_t)(f1 >> 32), ln, pre[wave], row[wave], [] { wave_lds_sync(); },
      [](int x, int& total) { return wave_exclusive_scan(x, total); },
      [&](uint32_t t, float w) { insert(tk, ts, size, t, w, nullptr); }, [] { return false; });
  const uint32_t out = (uint32_t)f0;
  int m = 0;
  double k = 0.0;
  for (uint32_t j0 = 0; j0 < size; j0 += 64) {
    const uint32_t id = tk[j0 + ln];
    const uint64_t used = __ballot(id != EMPTY);
    if (id != EMPTY) {
      const int64_t at = (int64_t)out + m + __popcll(used & ((((uint64_t)1) << ln) - 1));
      const float w = (float)ts[j0 + ln];
      c.out_col[at] = (int32_t)id;
      c.out_wt[at] = w;
      k += (double)w;
    }
    m += __popcll(used);
  }
  k = wave_sum_f64(k);
  if (ln == 0) {
    c.out_end[s] = (int32_t)(out + m);
    c.out_k[s] = k;
  }
}

// Block-wide exclusive scan of one int per thread (NW waves).
template <int NW>
__device__ inline int block_exclusive_scan(int x, int& total, int* s_wave) {
  int wave_total;
  int before = wave_exclusive_scan(x, wave_total);
  if (lane() == 63) s_wave[threadIdx.x >> 6] = wave_total;
  __syncthreads();
  total = 0;
  for (int i = 0; i < NW; ++i) {
    if (i < (int)(threadIdx.x >> 6)) before += s_wave[i];
    total += s_wave[i];
  }
  __syncthreads();
  return before;
}

__global__ __launch_bounds__(AGG_THREADS) void agg_long_kernel(Contract c, const int32_t* __restrict__ list,
                                                               int32_t* __restrict__ dense_list, int32_t* lists) {
  constexpr int NW = AGG_THREADS / 64;
  __shared__ uint32_t tk[AGG_LONG_SLOTS];
  __shared__ double ts[AGG_LONG_SLOTS];
  __shared__ int32_t pre[AGG_THREADS], row[AGG_THREADS];
  __shared__ double red[NW];
  __shared__ int s_wave[NW], s_added, s_ticket;
  const int tid = threadIdx.x;
  const int32_t listed = lists[AGG_N_LONG];
  while (true) {
    if (tid == 0) {
      s_ticket = atomicAdd(lists + AGG_TICKET, 1);
      s_added = 0;
    }
    __syncthreads();
    const int32_t it = s_ticket;
    if (it >= listed) return;
    const int32_t s = list[it];
    const uint64_t f0 = c.first[s], f1 = c.first[s + 1];
    const uint32_t n = (uint32_t)f1 - (uint32_t)f0;
    const uint32_t size = table_size(min(n, (uint32_t)c.S), AGG_LONG_SLOTS);
    for (uint32_t j = tid; j < size; j += AGG_THREADS) {
      tk[j] = EMPTY;
      ts[j] = 0.0;
    }
    __syncthreads();
    walk_members<AGG_THREADS>(
        c, (int32_t)(f0 >> 32), (int32_t)(f1 >> 32), tid, pre, row, [] { __syncthreads(); },
        [&](int x, int& total) { return block_exclusive_scan<NW>(x, total, s_wave); },
        [&](uint32_t t, float w) { insert(tk, ts, size, t, w, &s_added); },
        [&] {
          if (size < AGG_LONG_SLOTS) return false;  // room for every id
          __syncthreads();
          const bool full = s_added > AGG_LONG_MOST;
          __syncthreads();
          return full;
        });
    __syncthreads();
    if (s_added > AGG_LONG_MOST) {
      if (tid == 0) dense_list[atomicAdd(lists + AGG_N_DENSE, 1)] = s;
      __syncthreads();
      continue;
    }
    constexpr int PER = AGG_LONG_SLOTS / AGG_THREADS;
    uint32_t id[PER];
    int own = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const uint32_t j = tid + AGG_THREADS * i;
      id[i] = j < size ? tk[j] : EMPTY;
      own += id[i] != EMPTY ? 1 : 0;
    }
    int m;
    int64_t at = (int64_t)(uint32_t)f0 + block_exclusive_scan<NW>(own, m, s_wave);
    double k = 0.0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (id[i] != EMPTY) {
        const float w = (float)ts[tid + AGG_THREADS * i];
        c.out_col[at] = (int32_t)id[i];
        c.out_wt[at] = w;
        k += (double)w;
        ++at;
      }
    }
    k = wave_sum_f64(k);
    if (lane() == 0) red[tid >> 6] = k;
    __syncthreads();
    if (tid == 0) {
      c.out_end[s] = (int32_t)((uint32_t)f0 + m);
      c.out_k[s] = red[0] + red[1] + red[2] + red[3];
    }
    __syncthreads();
  }
}

constexpr size_t agg_dense_lds() { return AGG_WINDOW * 8 + AGG_WINDOW / 8; }

__global__ __launch_bounds__(AGG_DENSE_THREADS) void agg_dense_kernel(Contract c,
                                                                      const int32_t* __restrict__ dense_list,
                                                                      const int32_t* __restrict__ lists) {
  constexpr int NW = AGG_DENSE_THREADS / 64, PER = AGG_WINDOW / AGG_DENSE_THREADS;
  static_assert(PER == 16, "a thread owns half a mark word");
  extern __shared__ double sum_s[];
  uint32_t* mark = reinterpret_cast<uint32_t*>(sum_s + AGG_WINDOW);
  __shared__ int32_t pre[AGG_DENSE_THREADS], row[AGG_DENSE_THREADS];
  __shared__ double red[NW];
  __shared__ int s_wave[NW];
  const int tid = threadIdx.x;
  const int32_t listed = lists[AGG_N_DENSE];
  for (int32_t it = blockIdx.x; it < listed; it += gridDim.x) {
    const int32_t s = dense_list[it];
    const uint64_t f0 = c.first[s], f1 = c.first[s + 1];
    const int32_t g0 = s / c.S * c.S;
    int done = 0;
    double k = 0.0;
    for (int32_t lo = g0; lo < g0 + c.S; lo += AGG_WINDOW) {
      for (int j = tid; j < AGG_WINDOW; j += AGG_DENSE_THREADS) sum_s[j] = 0.0;
      for (int j = tid; j < AGG_WINDOW / 32; j += AGG_DENSE_THREADS) mark[j] = 0u;
      __syncthreads();
      walk_members<AGG_DENSE_THREADS>(
          c, (int32_t)(f0 >> 32), (int32_t)(f1 >> 32), tid, pre, row, [] { __syncthreads(); },
          [&](int x, int& total) { return block_exclusive_scan<NW>(x, total, s_wave); },
          [&](uint32_t t, float w) {
            const int32_t d = (int32_t)t - lo;
            if (d >= 0 && d < AGG_WINDOW) {
              unsafeAtomicAdd(sum_s + d, (double)w);
              atomicOr(mark + (d >> 5), 1u << (d & 31));
            }
          },
          [] { return false; });
      __syncthreads();
      const uint32_t bits = (mark[tid >> 1] >> (16 * (tid & 1))) & 0xffffu;
      int m;
      int64_t at = (int64_t)(uint32_t)f0 + done + block_exclusive_scan<NW>(__popc(bits), m, s_wave);
      for (int i = 0; i < PER; ++i) {
        if ((bits >> i) & 1u) {
          const int d = tid * PER + i;
          const float w = (float)sum_s[d];
          c.out_col[at] = lo + d;
          c.out_wt[at] = w;
          k += (double)w;
          ++at;
        }
      }
      done += m;
      __syncthreads();
    }
    k = wave_sum_f64(k);
    if (lane() == 0) red[tid >> 6] = k;
    __syncthreads();
    if (tid == 0) {
      double t = 0.0;
      for (int i = 0; i < NW; ++i) t += red[i];
      c.out_end[s] = (int32_t)((uint32_t)f0 + done);
      c.out_k[s] = t;
    }
    __syncthreads();
  }
}

// ----------------------------------------------------------------- the run's own small kernels
// Start of a level: identity labels, the first sweep's cleared totals, cleared
// lists and control words (the overflow word stays raised after the first
// level), and what the sweeps would compute of every vertex or graph again and again.
__global__ __launch_bounds__(ETHREADS) void level_init_kernel(int32_t V, int32_t* __restrict__ labels,
                                                              int32_t* __restrict__ moves, double* __restrict__ total,
                                                              int32_t* __restrict__ ctl,
                                                              int32_t* __restrict__ counts,
                                                              const double* __restrict__ two_m,
                                                              double2* __restrict__ scale,
                                                              uint32_t* __restrict__ salt, Divisor graph_of,
                                                              int32_t G, int first) {
  const int32_t v = blockIdx.x * ETHREADS + threadIdx.x;
  if (v < G) {
    const double m = 0.5 * two_m[v];  // (a graph without weight is not asked for these)
    scale[v] = double2{1.0 / m, 1.0 / (2.0 * m * m)};
  }
  if (v < V) {
    salt[v] = salt_of((uint32_t)graph_of.of(v), (uint32_t)v);
    labels[v] = v;
    moves[v] = v;
    total[v] = 0.0;
  }
  for (int32_t i = v; i < CTL_WORDS; i += gridDim.x * ETHREADS) {
    if (i != CTL_OVERFLOW || first) ctl[i] = 0;
  }
  if (v <= ROW_COUNTS) counts[v] = 0;
}

// width = the largest number of distinct labels of a graph.
__global__ __launch_bounds__(256) void width_kernel(const int32_t* __restrict__ flags, const int32_t* __restrict__ scan,
                                                    int32_t G, int32_t S, int32_t* __restrict__ width) {
  __shared__ int s_max;
  if (threadIdx.x == 0) s_max = 0;
  __syncthreads();
  for (int32_t g = threadIdx.x; g < G; g += 256) {
    const int32_t last = (g + 1) * S - 1;
    atomicMax(&s_max, scan[last] + flags[last] - scan[g * S]);
  }
  __syncthreads();
  if (threadIdx.x == 0) *width = s_max;
}

// Ranks of a level's labels among its graph's labels in use, and *width, the
// largest number of them in a graph:
// one workgroup per graph marks them in a bitmap in LDS and counts the bits
// below.  It takes the place of five launches over all vertices (clear, mark,
// scan in two, width), 25 us and 14 us a level at eight 32k and 2k graphs.
constexpr int RANK_THREADS = 1024;
constexpr int RANK_MOST = 1 << 18;  // vertices of a graph: two words per 32 in 64 KB of LDS

__global__ __launch_bounds__(RANK_THREADS) void rank_kernel(const int32_t* __restrict__ labels, int32_t S,
                                                            int32_t* __restrict__ rank,
                                                            int32_t* __restrict__ width) {
  extern __shared__ uint32_t rank_lds[];
  __shared__ int32_t s_wave[RANK_THREADS / 64];
  constexpr int U = 8;  // loads of a thread in flight
  const int words = (S + 31) / 32;
  uint32_t* bits = rank_lds;
  uint32_t* below = rank_lds + words;  // bits set in the words before
  const int32_t g0 = blockIdx.x * S;
  for (int i = threadIdx.x; i < words; i += RANK_THREADS) bits[i] = 0;
  __syncthreads();
  for (int i0 = threadIdx.x; i0 < S; i0 += U * RANK_THREADS) {
    int32_t l[U];
#pragma unroll
    for (int u = 0; u < U; ++u) l[u] = labels[g0 + min(i0 + u * RANK_THREADS, S - 1)] - g0;  // (the last one again)
#pragma unroll
    for (int u = 0; u < U; ++u) atomicOr(bits + (l[u] >> 5), 1u << (l[u] & 31));
  }
  __syncthreads();
  const int per = (words + RANK_THREADS - 1) / RANK_THREADS;
  const int w0 = threadIdx.x * per, w1 = min(words, w0 + per);
  int32_t mine = 0;
  for (int w = w0; w < w1; ++w) mine += __popc(bits[w]);
  int32_t upto = mine;
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t before = __shfl_up(upto, o);
    if (lane() >= o) upto += before;
  }
  if (lane() == 63) s_wave[threadIdx.x >> 6] = upto;
  __syncthreads();
  int32_t at = upto - mine, all = 0;
  for (int i = 0; i < RANK_THREADS / 64; ++i) {
    if (i < (int)(threadIdx.x >> 6)) at += s_wave[i];
    all += s_wave[i];
  }
  for (int w = w0; w < w1; ++w) {
    below[w] = (uint32_t)at;
    at += __popc(bits[w]);
  }
  if (threadIdx.x == 0) atomicMax(width, all);  // (cleared by level_init_kernel)
  __syncthreads();
  for (int i0 = threadIdx.x; i0 < S; i0 += U * RANK_THREADS) {
    int32_t l[U];
#pragma unroll
    for (int u = 0; u < U; ++u) l[u] = labels[g0 + min(i0 + u * RANK_THREADS, S - 1)] - g0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * RANK_THREADS;
      if (i < S)
        rank[g0 + i] = (int32_t)below[l[u] >> 5] + __popc(bits[l[u] >> 5] & ((1u << (l[u] & 31)) - 1));
    }
  }
}

// The level's dense ids (ranks behind the graph's width), the community of
// every first-level vertex in them, and the contraction's cleared counters.
__global__ __launch_bounds__(ETHREADS) void dense_chain_kernel(const int32_t* __restrict__ rank, int32_t V,
                                                               Divisor graph_of, int32_t width, int32_t V0, int first,
                                                               int32_t* __restrict__ dense,
                                                               int32_t* __restrict__ chain,
                                                               uint64_t* __restrict__ hist, int32_t n,
                                                               int32_t* __restrict__ lists) {
  const int32_t v = blockIdx.x * ETHREADS + threadIdx.x;
  if (v < V) dense[v] = rank[v] + graph_of.of(v) * width;
  if (v < V0) {
    const int32_t c = first ? v : chain[v];
    chain[v] = rank[c] + graph_of.of(c) * width;
  }
  if (v < n) hist[v] = 0;
  if (v < AGG_WORDS) lists[v] = 0;
}

// chain: the community of every original vertex so far, in the level's own ids.
__global__ __launch_bounds__(ETHREADS) void chain_kernel(const int32_t* __restrict__ dense, int32_t V0, int first,
                                                         int32_t* __restrict__ chain) {
  const int32_t v = blockIdx.x * ETHREADS + threadIdx.x;
  if (v < V0) chain[v] = dense[first ? v : chain[v]];
}

// Per vertex of the first level: weight of its row inside its community, and
// its degree times the community's total (helpers.cu:41-78).
__global__ __launch_bounds__(LTHREADS) void inside_kernel(Graph gr, const int32_t* __restrict__ labels,
                                                          const double* __restrict__ sigma,
                                                          double* __restrict__ inside, double* __restrict__ square) {
  const int32_t v = blockIdx.x * LWAVES + (threadIdx.x >> 6);
  if (v >= gr.V) return;
  const int32_t cv = labels[v];
  const int32_t a = gr.beg[v], b = gr.end[v];
  double in_sum = 0.0;
  for (int32_t e = a + lane(); e < b; e += 64)
    if (labels[gr.col[e]] == cv) in_sum += (double)gr.wt[e];
  in_sum = wave_sum_f64(in_sum);
  if (lane() == 0) {
    inside[v] = in_sum;
    square[v] = gr.k_v[v] * sigma[cv];
  }
}

// Modularity of the disjoint union: out[0]; out[1] != 0 when a table overflowed.
__global__ void union_modularity_kernel(const double* __restrict__ two_m, const double* __restrict__ inside,
                                        const double* __restrict__ square, int32_t G, float resolution,
                                        const int32_t* __restrict__ ctl, double* __restrict__ out) {
  if (threadIdx.x != 0) return;
  double m = 0.0, in_sum = 0.0, sq = 0.0;
  for (int32_t g = 0; g < G; ++g) {
    m += two_m[g];
    in_sum += inside[g];
    sq += square[g];
  }
  out[0] = m > 0.0 ? in_sum / m - (double)resolution * sq / (m * m) : 0.0;
  out[1] = ctl[CTL_OVERFLOW] != 0 ? 1.0 : 0.0;
}

__global__ __launch_bounds__(ETHREADS) void isolated_kernel(const int32_t* __restrict__ row_ptr, int32_t V,
                                                            int32_t* __restrict__ labels) {
  const int32_t v = blockIdx.x * ETHREADS + threadIdx.x;
  if (v < V && row_ptr[v] == row_ptr[v + 1]) labels[v] = -1;
}

// ----------------------------------------------------------------- dense community ids
// Words of graph g: [0, W) the labels in use, [W, W + S) the vertices without
// one; an exclusive scan over them numbers the labels by rank and then those
// vertices by position (partition.py:269-286).
__global__ __launch_bounds__(ETHREADS) void community_mark_kernel(const int32_t* __restrict__ labels, int32_t G,
                                                                  int32_t S, int32_t W, int32_t* __restrict__ words) {
  const int32_t v = blockIdx.x * ETHREADS + threadIdx.x;
  if (v >= G * S) return;
  const int32_t g = v / S;
  const int64_t base = (int64_t)g * (W + S);
  const int32_t l = labels[v];
  words[base + W + (v - g * S)] = l < 0 ? 1 : 0;
  if (l >= 0) words[base + (l - g * W)] = 1;
}

__global__ __launch_bounds__(ETHREADS) void community_zero_kernel(int32_t G, int32_t S, int32_t W,
                                                                  int32_t* __restrict__ words) {
  const int32_t i = blockIdx.x * ETHREADS + threadIdx.x;
  if (i < G * W) words[(int64_t)(i / W) * (W + S) + i % W] = 0;
}

__global__ __launch_bounds__(ETHREADS) void community_apply_kernel(const int32_t* __restrict__ labels, int32_t G,
                                                                   int32_t S, int32_t W,
                                                                   const int32_t* __restrict__ words,
                                                                   const int32_t* __restrict__ scan,
                                                                   int32_t* __restrict__ ids,
                                                                   int32_t* __restrict__ counts) {
  const int32_t v = blockIdx.x * ETHREADS + threadIdx.x;
  if (v >= G * S) return;
  const int32_t g = v / S;
  const int64_t base = (int64_t)g * (W + S);
  const int32_t l = labels[v];
  ids[v] = scan[base + (l < 0 ? W + (v - g * S) : l - g * W)] - scan[base];
  if (v == g * S) {
    const int64_t last = base + W + S - 1;
    counts[g] = scan[last] + words[last] - scan[base];
  }
}

// ----------------------------------------------------------------- host side
inline unsigned blocks(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

int launch_check() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : ckv_internal::set_error(CKV_E_LAUNCH, hipGetErrorString(e));
}

struct LeidenLayout {
  size_t keys_a, keys_b, vals_a, vals_b, temp, temp_bytes, row_ptr, col, k_v, two_m, totals[4], lab, moves[2], pairs[2],
      prop, mover, ctl, rows, giants, counts, scale, salt, total;
};

LeidenLayout leiden_layout(int64_t E, int32_t G, int32_t S) {
  LeidenLayout L{};
  const int64_t n = 2 * E;
  const int64_t V = (int64_t)G * S;
  size_t temp_bytes = 0;
  if (n > 0)
    (void)hipcub::DeviceRadixSort::SortPairs(nullptr, temp_bytes, (uint64_t*)nullptr, (uint64_t*)nullptr,
                                       (float*)nullptr, (float*)nullptr, (int)n, 0, 64, (hipStream_t)0);
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off += align256(bytes);
    return at;
  };
  L.keys_a = take(n * 8);
  L.keys_b = take(n * 8);
  L.vals_a = take(n * 4);
  L.vals_b = take(n * 4);
  L.temp_bytes = temp_bytes;
  L.temp = take(temp_bytes);
  L.row_ptr = take((V + 1) * 4);
  L.col = take(n * 4);
  L.k_v = take(V * 8);
  L.two_m = take(G * 8);
  for (size_t& at : L.totals) at = take(V * 8);
  L.lab = take(V * 4);
  for (int i = 0; i < 2; ++i) {
    L.moves[i] = take(V * 4);
    L.pairs[i] = take(V * 8);
  }
  L.prop = take(V * 4);
  L.mover = take(V * 4);
  L.salt = take(V * 4);
  L.scale = take(G * 16);
  L.ctl = take(CTL_WORDS * 4);
  L.rows = take(V * 4);
  L.giants = take(V * 4);
  L.counts = take((ROW_COUNTS + 1) * 4);
  L.total = off;
  return L;
}

struct AggLayout {
  size_t keys_a, keys_b, vals_a, uniq, temp, temp_bytes, total;
};

AggLayout agg_layout(int64_t E) {
  AggLayout L{};
  size_t sort_bytes = 0, red_bytes = 0;
  if (E > 0) {
    (void)hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, (uint64_t*)nullptr, (uint64_t*)nullptr, (float*)nullptr,
                                       (float*)nullptr, (int)E, 0, 64, (hipStream_t)0);
    (void)hipcub::DeviceReduce::ReduceByKey(nullptr, red_bytes, (uint64_t*)nullptr, (uint64_t*)nullptr, (float*)nullptr,
                                      (float*)nullptr, (int64_t*)nullptr, hipcub::Sum(), (int)E, (hipStream_t)0);
  }
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off += align256(bytes);
    return at;
  };
  L.keys_a = take(E * 8);
  L.keys_b = take(E * 8);
  L.vals_a = take(E * 4 * 2);  // values in, sorted values
  L.uniq = take(E * 8);
  L.temp_bytes = sort_bytes > red_bytes ? sort_bytes : red_bytes;
  L.temp = take(L.temp_bytes);
  L.total = off;
  return L;
}

size_t densify_temp_bytes(int64_t V) {
  size_t bytes = 0;
  (void)hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, (int32_t*)nullptr, (int32_t*)nullptr, (int)V, (hipStream_t)0);
  return bytes;
}

// Sort the (key, weight) pairs in keys_a / vals_a of an AggLayout, sum equal
// keys, drop the sentinel run and unpack (src, dst).
int coalesce(const AggLayout& L, char* ws, int64_t n, int32_t vertices, int bits, int end_bit, int32_t* out_src,
             int32_t* out_dst, float* out_weight, int64_t* out_count, hipStream_t st) {
  uint64_t* keys_a = (uint64_t*)(ws + L.keys_a);
  uint64_t* keys_b = (uint64_t*)(ws + L.keys_b);
  float* vals_in = (float*)(ws + L.vals_a);
  float* vals_sorted = vals_in + n;
  uint64_t* uniq = (uint64_t*)(ws + L.uniq);
  size_t temp_bytes = L.temp_bytes;
  if (hipcub::DeviceRadixSort::SortPairs(ws + L.temp, temp_bytes, keys_a, keys_b, vals_in, vals_sorted, (int)n, 0,
                                         end_bit, st) != hipSuccess)
    return ckv_internal::set_error(CKV_E_LAUNCH, "edge sort failed");
  temp_bytes = L.temp_bytes;
  if (hipcub::DeviceReduce::ReduceByKey(ws + L.temp, temp_bytes, keys_b, uniq, vals_sorted, out_weight, out_count,
                                        hipcub::Sum(), (int)n, st) != hipSuccess)
    return ckv_internal::set_error(CKV_E_LAUNCH, "edge reduce failed");
  count_fix_kernel<<<1, 64, 0, st>>>(uniq, vertices, bits, out_count);
  unpack_kernel<<<blocks(n, ETHREADS), ETHREADS, 0, st>>>(uniq, n, bits, out_count, out_src, out_dst);
  return launch_check();
}

}  // namespace
}  // namespace ckv

using namespace ckv;

static bool g_test_raise_overflow = false;

namespace ckv {
namespace {

// The arrays of one level's sweeps.
struct SweepBuffers {
  double* total[4];    // communities' total degrees, in turn
  int32_t* labels;     // the result; identity on entry
  int32_t* moves[2];   // local moving's labels; moves[0] is the identity on entry
  int2* pairs[2];      // refinement's (parent, label)
  int32_t* prop;
  int32_t* mover;
  int32_t* ctl;
  RowLists lists;
  double2* scale;
  uint32_t* salt;
};

// Queues a level: cleared state, lists of long rows, local moving and
// refinement.  The communities end in b.labels.
void run_sweeps(const Graph& gr, const SweepBuffers& b, float resolution, float theta, int32_t max_inner_iter,
                int32_t seed, int32_t use_boltzmann, bool first_level, hipStream_t st) {
  const int32_t V = gr.V;
  const Divisor graph_of(gr.S);
  const LevelConst lc{b.scale, b.salt, graph_of};
  level_init_kernel<<<blocks(V, ETHREADS), ETHREADS, 0, st>>>(V, b.labels, b.moves[0], b.total[0], b.ctl,
                                                              b.lists.counts, gr.two_m, b.scale, b.salt, graph_of,
                                                              V / gr.S, first_level);
  row_list_kernel<<<blocks(V, LIST_THREADS), LIST_THREADS, 0, st>>>(gr.beg, gr.end, V, b.lists);
  const Split split = split_of(V);
  const unsigned grid = split.grid;
  RowLists lists = b.lists;
  lists.long_blocks = split.long_blocks;
  lists.first = split.first;
  // (a row of different neighbours, its self loop twice, is at most one longer than its graph)
  const bool giants = !gr.unique || gr.S >= GIANT_MIN;
  double* const* t = b.total;
  for (int32_t i = 0; i < max_inner_iter; ++i) {
    if (i > 0 && i % RING == 0) fold_kernel<<<1, 64, 0, st>>>(b.ctl, 1, 0);
    const MoveSweep s{i == 0 ? gr.k_v : t[(i - 1) % 3], t[i % 3], t[(i + 1) % 3], b.moves[i & 1], b.moves[(i & 1) ^ 1],
                      b.ctl, i, resolution, (uint32_t)seed, lc};
    if (i == 0 && gr.unique) {
      local_moving_kernel<true><<<grid, HUB_THREADS, 0, st>>>(gr, s, lists);
      if (giants) local_moving_giant_kernel<true><<<GIANT_BLOCKS, GIANT_THREADS, 0, st>>>(gr, s, lists);
    } else {
      local_moving_kernel<false><<<grid, HUB_THREADS, 0, st>>>(gr, s, lists);
      if (giants)
        local_moving_giant_kernel<false><<<GIANT_BLOCKS, GIANT_THREADS, 0, st>>>(gr, s, lists);
    }
  }
  if (g_test_raise_overflow) raise_overflow_kernel<<<1, 64, 0, st>>>(b.ctl);
  // refinement from singletons inside the local-moving communities
  const int32_t* parent = b.moves[max_inner_iter & 1];
  const double* parent_total = max_inner_iter == 0 ? gr.k_v : t[(max_inner_iter - 1) % 3];
  double* r[3] = {t[max_inner_iter % 3], t[(max_inner_iter + 1) % 3], t[3]};  // r[0] was cleared by the last sweep
  const float temperature = theta > 0.0f ? theta : 1.0e-3f;
  const float inv_theta = 1.0f / temperature;
  if (max_inner_iter > RING) fold_kernel<<<1, 64, 0, st>>>(b.ctl, 1, 1);
  if (!gr.unique) pair_init_kernel<<<blocks(V, ETHREADS), ETHREADS, 0, st>>>(parent, V, b.pairs[0]);
  for (int32_t i = 0; i < max_inner_iter; ++i) {
    if (i > 0 && i % RING == 0) fold_kernel<<<1, 64, 0, st>>>(b.ctl, 0, 0);
    const RefineSweep s{i == 0 ? gr.k_v : r[(i - 1) % 3], parent_total, r[i % 3], r[(i + 1) % 3], parent,
                        b.pairs[i & 1], b.pairs[(i & 1) ^ 1], b.labels, b.prop, b.mover, b.ctl, i, resolution,
                        inv_theta, use_boltzmann ? 1 : 0, (uint32_t)seed, lc};
    if (i == 0 && gr.unique) {
      refine_propose_kernel<true><<<grid, HUB_THREADS, 0, st>>>(gr, s, lists);
      if (giants)
        refine_propose_giant_kernel<true><<<GIANT_BLOCKS, GIANT_THREADS, 0, st>>>(gr, s, lists);
      refine_commit_kernel<true><<<grid, HUB_THREADS, 0, st>>>(gr, s, lists);
    } else {
      refine_propose_kernel<false><<<grid, HUB_THREADS, 0, st>>>(gr, s, lists);
      if (giants)
        refine_propose_giant_kernel<false><<<GIANT_BLOCKS, GIANT_THREADS, 0, st>>>(gr, s, lists);
      refine_commit_kernel<false><<<grid, HUB_THREADS, 0, st>>>(gr, s, lists);
    }
  }
}

}  // namespace
}  // namespace ckv

extern "C" void ckv_leiden_test_raise_overflow(int32_t enable) { g_test_raise_overflow = enable != 0; }

extern "C" size_t ckv_leiden_workspace_bytes(int64_t edges, int32_t graphs, int32_t seq_len) {
  if (edges < 0 || graphs <= 0 || seq_len <= 0) return 0;
  return leiden_layout(edges, graphs, seq_len).total;
}

extern "C" int ckv_batched_leiden(const int32_t* edge_src, const int32_t* edge_dst, const float* edge_weight,
                                  int64_t edges, int32_t graphs, int32_t seq_len, float resolution, float theta,
                                  int32_t max_inner_iter, int32_t seed, int32_t use_boltzmann, int32_t* labels,
                                  double* modularity, void* workspace, void* stream) {
  if (graphs <= 0 || seq_len <= 0) return ckv_internal::set_error(CKV_E_INVALID, "graphs and seq_len must be positive");
  if (!labels || !modularity) return ckv_internal::set_error(CKV_E_INVALID, "null Leiden output");
  if (edges < 0 || (edges > 0 && (!edge_src || !edge_dst || !edge_weight || !workspace)))
    return ckv_internal::set_error(CKV_E_INVALID, "Leiden edges need src, dst, weight and a workspace");
  const int64_t V64 = (int64_t)graphs * seq_len;
  if (V64 >= (int64_t)1 << 30 || 2 * edges >= ((int64_t)1 << 31) - 1)
    return ckv_internal::set_error(CKV_E_LIMIT, "Leiden graph too large (vertices < 2^30, 2 * edges < 2^31)");
  if (max_inner_iter < 0) return ckv_internal::set_error(CKV_E_INVALID, "max_inner_iter must be nonnegative");
  hipStream_t st = (hipStream_t)stream;
  const int32_t V = (int32_t)V64;
  if (edges == 0) {
    // leiden.cu:68-76: every vertex isolated, modularity 0
    if (hipMemsetAsync(labels, 0xFF, (size_t)V * 4, st) != hipSuccess ||
        hipMemsetAsync(modularity, 0, (size_t)graphs * 8, st) != hipSuccess)
      return launch_check();
    return 0;
  }
  const LeidenLayout L = leiden_layout(edges, graphs, seq_len);
  char* ws = (char*)workspace;
  uint64_t* keys_a = (uint64_t*)(ws + L.keys_a);
  uint64_t* keys_b = (uint64_t*)(ws + L.keys_b);
  float* vals_a = (float*)(ws + L.vals_a);
  float* vals_b = (float*)(ws + L.vals_b);
  int32_t* row_ptr = (int32_t*)(ws + L.row_ptr);
  int32_t* col = (int32_t*)(ws + L.col);
  double* k_v = (double*)(ws + L.k_v);
  double* two_m = (double*)(ws + L.two_m);
  double* sigma = (double*)(ws + L.totals[0]);
  int32_t* lab = (int32_t*)(ws + L.lab);
  int32_t* ctl = (int32_t*)(ws + L.ctl);

  const int bits = bits_for((uint64_t)V - 1);
  const int end_bit = bits + bits_for((uint64_t)V);
  const int64_t n = 2 * edges;
  mirror_kernel<<<blocks(edges, ETHREADS), ETHREADS, 0, st>>>(edge_src, edge_dst, edge_weight, edges, V, bits, keys_a,
                                                             vals_a);
  size_t temp_bytes = L.temp_bytes;
  if (hipcub::DeviceRadixSort::SortPairs(ws + L.temp, temp_bytes, keys_a, keys_b, vals_a, vals_b, (int)n, 0, end_bit,
                                         st) != hipSuccess)
    return ckv_internal::set_error(CKV_E_LAUNCH, "Leiden CSR sort failed");
  row_ptr_kernel<<<blocks(V + 1, ETHREADS), ETHREADS, 0, st>>>(keys_b, n, V, bits, row_ptr);
  col_kernel<<<blocks(n, ETHREADS), ETHREADS, 0, st>>>(keys_b, n, bits, col);
  const unsigned vgrid = blocks(V, LWAVES), egrid = blocks(V, ETHREADS);
  degree_kernel<<<vgrid, LTHREADS, 0, st>>>(row_ptr, vals_b, V, k_v);
  graph_sum_kernel<<<graphs, SUM_THREADS, 0, st>>>(k_v, seq_len, two_m);
  const Graph gr{row_ptr, row_ptr + 1, col, vals_b, k_v, two_m, V, seq_len, false};
  const SweepBuffers buf{{(double*)(ws + L.totals[0]), (double*)(ws + L.totals[1]), (double*)(ws + L.totals[2]),
                          (double*)(ws + L.totals[3])},
                         lab,
                         {(int32_t*)(ws + L.moves[0]), (int32_t*)(ws + L.moves[1])},
                         {(int2*)(ws + L.pairs[0]), (int2*)(ws + L.pairs[1])},
                         (int32_t*)(ws + L.prop), (int32_t*)(ws + L.mover), ctl,
                         {(int32_t*)(ws + L.rows), (int32_t*)(ws + L.giants), (int32_t*)(ws + L.counts), 0, 0},
                         (double2*)(ws + L.scale), (uint32_t*)(ws + L.salt)};
  run_sweeps(gr, buf, resolution, theta, max_inner_iter, seed, use_boltzmann, true, st);
  sigma_zero_kernel<<<egrid, ETHREADS, 0, st>>>(sigma, V);
  sigma_scatter_kernel<<<egrid, ETHREADS, 0, st>>>(lab, k_v, V, sigma);
  double* share = (double*)(ws + L.totals[1]);
  modularity_kernel<<<vgrid, LTHREADS, 0, st>>>(gr, lab, sigma, resolution, share);
  graph_sum_kernel<<<graphs, SUM_THREADS, 0, st>>>(share, seq_len, modularity);
  overflow_mark_kernel<<<blocks(graphs, ETHREADS), ETHREADS, 0, st>>>(ctl, graphs, modularity);
  finish_kernel<<<egrid, ETHREADS, 0, st>>>(row_ptr, lab, V, labels);
  return launch_check();
}

extern "C" size_t ckv_aggregate_coo_workspace_bytes(int64_t edges) {
  return edges <= 0 ? 0 : agg_layout(edges).total;
}

extern "C" int ckv_aggregate_coo(const int32_t* edge_src, const int32_t* edge_dst, const float* edge_weight,
                                 int64_t edges, const int32_t* labels, int32_t super_vertices, int32_t* out_src,
                                 int32_t* out_dst, float* out_weight, int64_t* out_count, void* workspace,
                                 void* stream) {
  if (edges < 0 || super_vertices <= 0 || !out_count)
    return ckv_internal::set_error(CKV_E_INVALID, "bad aggregation sizes");
  hipStream_t st = (hipStream_t)stream;
  if (edges == 0) {
    if (hipMemsetAsync(out_count, 0, 8, st) != hipSuccess) return launch_check();
    return 0;
  }
  if (!edge_src || !edge_dst || !edge_weight || !labels || !out_src || !out_dst || !out_weight || !workspace)
    return ckv_internal::set_error(CKV_E_INVALID, "null aggregation pointer");
  if (edges >= ((int64_t)1 << 31) - 1 || super_vertices >= (1 << 30))
    return ckv_internal::set_error(CKV_E_LIMIT, "aggregation too large");
  const AggLayout L = agg_layout(edges);
  char* ws = (char*)workspace;
  uint64_t* keys_a = (uint64_t*)(ws + L.keys_a);
  float* vals_in = (float*)(ws + L.vals_a);
  const int bits = bits_for((uint64_t)super_vertices - 1);
  const int end_bit = bits + bits_for((uint64_t)super_vertices);
  remap_kernel<<<blocks(edges, ETHREADS), ETHREADS, 0, st>>>(edge_src, edge_dst, edge_weight, labels, edges,
                                                             super_vertices, bits, keys_a, vals_in);
  return coalesce(L, ws, edges, super_vertices, bits, end_bit, out_src, out_dst, out_weight, out_count, st);
}

extern "C" size_t ckv_densify_workspace_bytes(int32_t graphs, int32_t seq_len) {
  if (graphs <= 0 || seq_len <= 0) return 0;
  const int64_t V = (int64_t)graphs * seq_len;
  return 2 * align256((size_t)V * 4) + align256(densify_temp_bytes(V));
}

extern "C" int ckv_densify_count(const int32_t* labels, int32_t graphs, int32_t seq_len, int32_t* counts,
                                 void* workspace, void* stream) {
  if (!labels || !counts || !workspace || graphs <= 0 || seq_len <= 0)
    return ckv_internal::set_error(CKV_E_INVALID, "bad densify arguments");
  const int64_t V64 = (int64_t)graphs * seq_len;
  if (V64 >= (int64_t)1 << 30) return ckv_internal::set_error(CKV_E_LIMIT, "densify: too many vertices");
  const int32_t V = (int32_t)V64;
  hipStream_t st = (hipStream_t)stream;
  int32_t* flags = (int32_t*)workspace;
  int32_t* scan = (int32_t*)((char*)workspace + align256((size_t)V * 4));
  void* temp = (char*)workspace + 2 * align256((size_t)V * 4);
  size_t temp_bytes = densify_temp_bytes(V);
  flag_zero_kernel<<<blocks(V, ETHREADS), ETHREADS, 0, st>>>(flags, V);
  flag_mark_kernel<<<blocks(V, ETHREADS), ETHREADS, 0, st>>>(labels, V, seq_len, flags);
  if (hipcub::DeviceScan::ExclusiveSum(temp, temp_bytes, flags, scan, V, st) != hipSuccess)
    return ckv_internal::set_error(CKV_E_LAUNCH, "densify scan failed");
  densify_count_kernel<<<blocks(graphs, ETHREADS), ETHREADS, 0, st>>>(flags, scan, graphs, seq_len, counts);
  return launch_check();
}

extern "C" int ckv_densify_apply(const int32_t* labels, int32_t graphs, int32_t seq_len, int32_t new_seq_len,
                                 int32_t* dense, const void* workspace, void* stream) {
  if (!labels || !dense || !workspace || graphs <= 0 || seq_len <= 0 || new_seq_len <= 0)
    return ckv_internal::set_error(CKV_E_INVALID, "bad densify arguments");
  const int64_t V64 = (int64_t)graphs * seq_len;
  if (V64 >= (int64_t)1 << 30 || (int64_t)graphs * new_seq_len >= (int64_t)1 << 30)
    return ckv_internal::set_error(CKV_E_LIMIT, "densify: too many vertices");
  const int32_t V = (int32_t)V64;
  const int32_t* scan = (const int32_t*)((const char*)workspace + align256((size_t)V * 4));
  densify_apply_kernel<<<blocks(V, ETHREADS), ETHREADS, 0, (hipStream_t)stream>>>(labels, scan, V, seq_len,
                                                                                   new_seq_len, dense);
  return launch_check();
}

extern "C" size_t ckv_partition_modularity_workspace_bytes(int32_t vertices) {
  return vertices <= 0 ? 0 : 2 * align256((size_t)vertices * 8) + 256;
}

extern "C" int ckv_partition_modularity(const int32_t* edge_src, const int32_t* edge_dst, const float* edge_weight,
                                        int64_t edges, const int32_t* labels, int32_t vertices, float resolution,
                                        double* modularity, void* workspace, void* stream) {
  if (vertices <= 0 || edges < 0 || !labels || !modularity || !workspace ||
      (edges > 0 && (!edge_src || !edge_dst || !edge_weight)))
    return ckv_internal::set_error(CKV_E_INVALID, "bad modularity arguments");
  hipStream_t st = (hipStream_t)stream;
  double* k = (double*)workspace;
  double* sig = (double*)((char*)workspace + align256((size_t)vertices * 8));
  double* acc = (double*)((char*)workspace + 2 * align256((size_t)vertices * 8));
  mod_zero_kernel<<<blocks(vertices, ETHREADS), ETHREADS, 0, st>>>(k, sig, vertices, acc);
  if (edges > 0)
    mod_edge_kernel<<<blocks(edges, 256), 256, 0, st>>>(edge_src, edge_dst, edge_weight, edges, labels, vertices, k,
                                                        acc);
  mod_sigma_kernel<<<blocks(vertices, 256), 256, 0, st>>>(labels, k, vertices, sig, acc);
  mod_square_kernel<<<blocks(vertices, 256), 256, 0, st>>>(sig, vertices, acc);
  mod_final_kernel<<<1, 64, 0, st>>>(acc, resolution, modularity);
  return launch_check();
}

// ----------------------------------------------------------------- the whole multi-level run
namespace ckv {
namespace {

struct RunLayout {
  size_t row_ptr, col0, wt0, col[2], wt[2], beg[2], end[2], k[2], two_m, two_m0, totals[4], lab, moves[2], pairs[2], prop,
      mover, salt, scale, ctl, hubs, giants, counts, flags, scan, dense, hist, first, members, dense_list,
      lists, words, temp, temp_bytes, sort, total;
};

// Sorting scratch and the rows of the contracted levels share their place (the
// sorts end before the first contraction).
RunLayout run_layout(int64_t E, int32_t G, int32_t S) {
  RunLayout L{};
  const int64_t n = 2 * E, V = (int64_t)G * S;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off += align256(bytes);
    return at;
  };
  L.row_ptr = take((V + 1) * 4);
  L.col0 = take(n * 4);
  L.wt0 = take(n * 4);
  for (int i = 0; i < 2; ++i) {
    L.beg[i] = take(V * 4);
    L.end[i] = take(V * 4);
    L.k[i] = take(V * 8);
    L.moves[i] = take(V * 4);
    L.pairs[i] = take(V * 8);
  }
  L.two_m = take(G * 8);
  L.two_m0 = take(G * 8);
  for (size_t& at : L.totals) at = take(V * 8);
  L.lab = take(V * 4);
  L.prop = take(V * 4);
  L.mover = take(V * 4);
  L.salt = take(V * 4);
  L.scale = take(G * 16);
  L.ctl = take(CTL_WORDS * 4);
  L.hubs = take(V * 4);
  L.giants = take(V * 4);
  L.counts = take(256);
  L.flags = take(V * 4);
  L.scan = take(V * 4);
  L.dense = take(V * 4);
  L.hist = take((V + 1) * 8);
  L.first = take((V + 1) * 8);
  L.members = take(V * 4);
  L.dense_list = take(V * 4);
  L.lists = take(AGG_WORDS * 4);
  L.words = take(64);
  size_t scan64 = 0, sort64 = 0;
  (void)rocprim::exclusive_scan(nullptr, scan64, (const uint64_t*)nullptr, (uint64_t*)nullptr, (uint64_t)0,
                                (size_t)V + 1, rocprim::plus<uint64_t>(), (hipStream_t)0);
  (void)hipcub::DeviceRadixSort::SortPairs(nullptr, sort64, (uint64_t*)nullptr, (uint64_t*)nullptr, (float*)nullptr,
                                           (float*)nullptr, (int)n, 0, 64, (hipStream_t)0);
  const size_t scan32 = scan_bytes((size_t)V), sort32 = sort_pairs_bytes((size_t)E);
  L.temp_bytes = scan64 > scan32 ? scan64 : scan32;
  L.temp_bytes = L.temp_bytes > sort64 ? L.temp_bytes : sort64;
  L.temp_bytes = L.temp_bytes > sort32 ? L.temp_bytes : sort32;
  L.temp = take(L.temp_bytes);
  L.sort = off;
  for (int i = 0; i < 2; ++i) {
    L.col[i] = take(n * 4);
    L.wt[i] = take(n * 4);
  }
  const size_t unsorted = L.sort + 2 * align256(n * 8) + align256(n * 4);
  L.total = off > unsorted ? off : unsorted;
  return L;
}

// Reads `bytes` device bytes at `from` after everything queued on st.
int read_back(void* to, const void* from, size_t bytes, hipStream_t st) {
  if (hipMemcpyAsync(to, from, bytes, hipMemcpyDeviceToHost, st) != hipSuccess || hipStreamSynchronize(st) != hipSuccess)
    return launch_check() ? CKV_E_LAUNCH : ckv_internal::set_error(CKV_E_LAUNCH, "reading back a Leiden count failed");
  return 0;
}

}  // namespace
}  // namespace ckv

extern "C" size_t ckv_leiden_run_workspace_bytes(int64_t edges, int32_t graphs, int32_t seq_len) {
  if (edges <= 0 || graphs <= 0 || seq_len <= 0 || (int64_t)graphs * seq_len >= (int64_t)1 << 30 ||
      2 * edges >= ((int64_t)1 << 31) - 1)
    return 0;
  return run_layout(edges, graphs, seq_len).total;
}

extern "C" int ckv_leiden_run(const int32_t* edge_src, const int32_t* edge_dst, const float* edge_weight, int64_t edges,
                              int32_t graphs, int32_t seq_len, int32_t max_level, float resolution, float theta,
                              int32_t max_inner_iter, int32_t seed, int32_t use_boltzmann, int32_t* labels,
                              double* degree, int32_t* width, double* result, void* workspace, void* stream) {
  if (graphs <= 0 || seq_len <= 0) return ckv_internal::set_error(CKV_E_INVALID, "graphs and seq_len must be positive");
  if (!labels || !degree || !width || !result) return ckv_internal::set_error(CKV_E_INVALID, "null Leiden output");
  if (edges <= 0 || !edge_src || !edge_dst || !edge_weight || !workspace)
    return ckv_internal::set_error(CKV_E_INVALID, "a Leiden run needs edges (src, dst, weight) and a workspace");
  const int64_t V64 = (int64_t)graphs * seq_len;
  if (V64 >= (int64_t)1 << 30 || 2 * edges >= ((int64_t)1 << 31) - 1)
    return ckv_internal::set_error(CKV_E_LIMIT, "Leiden graph too large (vertices < 2^30, 2 * edges < 2^31)");
  if (max_inner_iter < 0) return ckv_internal::set_error(CKV_E_INVALID, "max_inner_iter must be nonnegative");
  hipStream_t st = (hipStream_t)stream;
  const int32_t V0 = (int32_t)V64;
  const int64_t n = 2 * edges;
  const RunLayout L = run_layout(edges, graphs, seq_len);
  char* ws = (char*)workspace;
  auto i32 = [&](size_t at) { return (int32_t*)(ws + at); };
  auto f64 = [&](size_t at) { return (double*)(ws + at); };
  int32_t* row_ptr = i32(L.row_ptr);
  int32_t* col0 = i32(L.col0);
  float* wt0 = (float*)(ws + L.wt0);
  int32_t* ctl = i32(L.ctl);
  int32_t* words = i32(L.words);  // edge flags, then the level's width
  int32_t* lists = i32(L.lists);
  uint64_t* hist = (uint64_t*)(ws + L.hist);
  uint64_t* first = (uint64_t*)(ws + L.first);

  // ---- the edges: inside their graphs? in order?
  agg_zero_kernel<<<1, ETHREADS, 0, st>>>((uint64_t*)words, 1, lists);
  edge_check_kernel<<<blocks(edges, ETHREADS), ETHREADS, 0, st>>>(edge_src, edge_dst, edges, V0, seq_len, words);
  int32_t host[2];
  if (int rc = read_back(host, words, 8, st)) return rc;
  if (host[0]) return ckv_internal::set_error(CKV_E_INVALID, "edges must join two vertices of the same graph");
  if (!host[1]) {
    // ascending (src, dst), as build_adjacency leaves them: 32-bit keys of one end of each edge
    uint32_t* keys_in = (uint32_t*)(ws + L.sort);
    uint32_t* vals_in = keys_in + align256(edges * 4) / 4;
    uint32_t* keys = vals_in + align256(edges * 4) / 4;
    uint32_t* vals = keys + align256(edges * 4) / 4;
    int32_t* upper = i32(L.hist);
    int32_t* lower = i32(L.first);
    upper_bounds_kernel<<<blocks(edges, ETHREADS), ETHREADS, 0, st>>>(edge_src, edge_dst, edges, V0, upper, keys_in,
                                                                      vals_in);
    if (sort_pairs(ws + L.temp, L.temp_bytes, keys_in, keys, vals_in, vals, (size_t)edges, bits_for((uint64_t)V0),
                   st) != hipSuccess)
      return ckv_internal::set_error(CKV_E_LAUNCH, "Leiden CSR sort failed");
    lower_bounds_kernel<<<blocks(edges, ETHREADS), ETHREADS, 0, st>>>(keys, edges, V0, lower);
    csr_fill_kernel<<<blocks(edges > V0 ? edges : V0 + 1, ETHREADS), ETHREADS, 0, st>>>(
        edge_src, edge_dst, edge_weight, edges, V0, upper, lower, keys, vals, row_ptr, col0, wt0);
  } else {
    uint64_t* keys_a = (uint64_t*)(ws + L.sort);
    uint64_t* keys_b = keys_a + align256(n * 8) / 8;
    float* vals_a = (float*)(keys_b + align256(n * 8) / 8);
    const int bits = bits_for((uint64_t)V0 - 1), end_bit = bits + bits_for((uint64_t)V0);
    mirror_kernel<<<blocks(edges, ETHREADS), ETHREADS, 0, st>>>(edge_src, edge_dst, edge_weight, edges, V0, bits,
                                                               keys_a, vals_a);
    size_t temp_bytes = L.temp_bytes;
    if (hipcub::DeviceRadixSort::SortPairs(ws + L.temp, temp_bytes, keys_a, keys_b, vals_a, wt0, (int)n, 0, end_bit,
                                           st) != hipSuccess)
      return ckv_internal::set_error(CKV_E_LAUNCH, "Leiden CSR sort failed");
    row_ptr_kernel<<<blocks(V0 + 1, ETHREADS), ETHREADS, 0, st>>>(keys_b, n, V0, bits, row_ptr);
    col_kernel<<<blocks(n, ETHREADS), ETHREADS, 0, st>>>(keys_b, n, bits, col0);
  }
  degree_kernel<<<blocks(V0, LWAVES), LTHREADS, 0, st>>>(row_ptr, wt0, V0, degree);
  graph_sum_kernel<<<graphs, SUM_THREADS, 0, st>>>(degree, seq_len, f64(L.two_m0));

  // ---- levels
  const Graph gr0{row_ptr, row_ptr + 1, col0, wt0, degree, f64(L.two_m0), V0, seq_len, host[1] == 0};
  Graph gr = gr0;
  for (int32_t level = 0;; ++level) {
    const unsigned egrid = blocks(gr.V, ETHREADS);
    const SweepBuffers buf{{f64(L.totals[0]), f64(L.totals[1]), f64(L.totals[2]), f64(L.totals[3])},
                           i32(L.lab),
                           {i32(L.moves[0]), i32(L.moves[1])},
                           {(int2*)(ws + L.pairs[0]), (int2*)(ws + L.pairs[1])},
                           i32(L.prop), i32(L.mover), ctl, {i32(L.hubs), i32(L.giants), i32(L.counts), 0, 0},
                           (double2*)(ws + L.scale), (uint32_t*)(ws + L.salt)};
    run_sweeps(gr, buf, resolution, theta, max_inner_iter, seed + level, use_boltzmann, level == 0, st);
    // ranks of the labels in use, per graph
    const int32_t* lab = i32(L.lab);
    int32_t* flags = i32(L.flags);
    int32_t* scan = i32(L.scan);
    int32_t* dense = i32(L.dense);
    const bool ranked = gr.S <= RANK_MOST;
    if (ranked) {
      const size_t lds = (size_t)(gr.S + 31) / 32 * 8;
      int32_t* widest = i32(L.counts) + ROW_COUNTS;
      rank_kernel<<<graphs, RANK_THREADS, lds, st>>>(lab, gr.S, scan, widest);
      if (int rc = read_back(width, widest, 4, st)) return rc;
      const int32_t n = graphs * *width + 1;
      dense_chain_kernel<<<blocks(n > V0 ? n : V0, ETHREADS), ETHREADS, 0, st>>>(
          scan, gr.V, Divisor(gr.S), *width, V0, level == 0, dense, labels, hist, n, lists);
    } else {
      flag_zero_kernel<<<egrid, ETHREADS, 0, st>>>(flags, gr.V);
      flag_mark_kernel<<<egrid, ETHREADS, 0, st>>>(lab, gr.V, gr.S, flags);
      if (exclusive_scan_i32(ws + L.temp, L.temp_bytes, flags, scan, (size_t)gr.V, st) != hipSuccess)
        return ckv_internal::set_error(CKV_E_LAUNCH, "densify scan failed");
      width_kernel<<<1, 256, 0, st>>>(flags, scan, graphs, gr.S, words);
      if (int rc = read_back(width, words, 4, st)) return rc;
      densify_apply_kernel<<<egrid, ETHREADS, 0, st>>>(lab, scan, gr.V, gr.S, *width, dense);
      chain_kernel<<<blocks(V0, ETHREADS), ETHREADS, 0, st>>>(dense, V0, level == 0, labels);
    }
    if (level + 1 >= max_level || *width >= gr.S) break;
    // contract
    const int32_t Vs = graphs * *width;
    const int to = level & 1;
    const Contract c{gr.beg, gr.end, gr.col, gr.wt, dense, i32(L.members), first, *width, i32(L.end[to]),
                     i32(L.col[to]), (float*)(ws + L.wt[to]), f64(L.k[to])};
    if (!ranked) agg_zero_kernel<<<blocks(Vs + 1, ETHREADS), ETHREADS, 0, st>>>(hist, Vs + 1, lists);
    agg_hist_kernel<<<egrid, ETHREADS, 0, st>>>(dense, gr.beg, gr.end, gr.V, hist);
    size_t temp_bytes = L.temp_bytes;
    if (rocprim::exclusive_scan(ws + L.temp, temp_bytes, (const uint64_t*)hist, first, (uint64_t)0, (size_t)Vs + 1,
                                rocprim::plus<uint64_t>(), st) != hipSuccess)
      return ckv_internal::set_error(CKV_E_LAUNCH, "contraction scan failed");
    agg_fill_kernel<<<egrid, ETHREADS, 0, st>>>(dense, gr.V, first, hist, i32(L.members));
    agg_list_kernel<<<blocks(Vs, LIST_THREADS), LIST_THREADS, 0, st>>>(first, Vs, i32(L.beg[to]), i32(L.end[to]),
                                                                      i32(L.hubs), lists);
    agg_short_kernel<<<blocks(Vs, AGG_WAVES), 64 * AGG_WAVES, 0, st>>>(c, Vs);
    agg_long_kernel<<<AGG_LONG_BLOCKS, AGG_THREADS, 0, st>>>(c, i32(L.hubs), i32(L.dense_list), lists);
    if (*width > AGG_LONG_MOST) {  // (a row has at most as many neighbours as its graph has super-vertices)
      if (hipFuncSetAttribute(reinterpret_cast<const void*>(agg_dense_kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)agg_dense_lds()) != hipSuccess)
        return launch_check();
      agg_dense_kernel<<<AGG_DENSE_BLOCKS, AGG_DENSE_THREADS, agg_dense_lds(), st>>>(c, i32(L.dense_list), lists);
    }
    gr = Graph{i32(L.beg[to]), i32(L.end[to]), i32(L.col[to]), (float*)(ws + L.wt[to]), f64(L.k[to]), f64(L.two_m), Vs,
               *width, true};
    graph_sum_kernel<<<graphs, SUM_THREADS, 0, st>>>(gr.k_v, gr.S, f64(L.two_m));
  }

  // ---- modularity of the result on the first level's graph
  const unsigned egrid = blocks(V0, ETHREADS);
  sigma_zero_kernel<<<egrid, ETHREADS, 0, st>>>(f64(L.totals[0]), V0);
  sigma_scatter_kernel<<<egrid, ETHREADS, 0, st>>>(labels, degree, V0, f64(L.totals[0]));
  inside_kernel<<<blocks(V0, LWAVES), LTHREADS, 0, st>>>(gr0, labels, f64(L.totals[0]), f64(L.totals[1]),
                                                         f64(L.totals[2]));
  double* sums = f64(L.k[0]);  // per graph: inside, square; then the result
  double* squares = f64(L.k[1]);
  graph_sum_kernel<<<graphs, SUM_THREADS, 0, st>>>(f64(L.totals[1]), seq_len, sums);
  graph_sum_kernel<<<graphs, SUM_THREADS, 0, st>>>(f64(L.totals[2]), seq_len, squares);
  union_modularity_kernel<<<1, 64, 0, st>>>(f64(L.two_m0), sums, squares, graphs, resolution, ctl, f64(L.hist));
  isolated_kernel<<<egrid, ETHREADS, 0, st>>>(row_ptr, V0, labels);
  if (int rc = launch_check()) return rc;
  double out[2];
  if (int rc = read_back(out, ws + L.hist, 16, st)) return rc;
  *result = out[0];
  if (out[1] != 0.0)
    return ckv_internal::set_error(CKV_E_LIMIT, "a neighbour-community table overflowed; the labels are not valid");
  return 0;
}

extern "C" size_t ckv_dense_communities_workspace_bytes(int32_t graphs, int32_t seq_len, int32_t width) {
  if (graphs <= 0 || seq_len <= 0 || width < 0) return 0;
  const int64_t n = (int64_t)graphs * ((int64_t)seq_len + width);
  return 2 * align256((size_t)n * 4) + align256(scan_bytes((size_t)n));
}

extern "C" int ckv_dense_communities(const int32_t* labels, int32_t graphs, int32_t seq_len, int32_t width,
                                     int32_t* community_ids, int32_t* community_counts, void* workspace, void* stream) {
  if (!labels || !community_ids || !community_counts || !workspace || graphs <= 0 || seq_len <= 0 || width < 0)
    return ckv_internal::set_error(CKV_E_INVALID, "bad community arguments");
  const int64_t n = (int64_t)graphs * ((int64_t)seq_len + width);
  if ((int64_t)graphs * seq_len >= (int64_t)1 << 30 || (int64_t)graphs * width >= (int64_t)1 << 30)
    return ckv_internal::set_error(CKV_E_LIMIT, "too many vertices or labels (each below 2^30, as a run's are)");
  hipStream_t st = (hipStream_t)stream;
  int32_t* words = (int32_t*)workspace;
  int32_t* scan = (int32_t*)((char*)workspace + align256((size_t)n * 4));
  void* temp = (char*)workspace + 2 * align256((size_t)n * 4);
  const unsigned grid = blocks((int64_t)graphs * seq_len, ETHREADS);
  if (width > 0)
    community_zero_kernel<<<blocks((int64_t)graphs * width, ETHREADS), ETHREADS, 0, st>>>(graphs, seq_len, width, words);
  community_mark_kernel<<<grid, ETHREADS, 0, st>>>(labels, graphs, seq_len, width, words);
  if (exclusive_scan_i32(temp, scan_bytes((size_t)n), words, scan, (size_t)n, st) != hipSuccess)
    return ckv_internal::set_error(CKV_E_LAUNCH, "community scan failed");
  community_apply_kernel<<<grid, ETHREADS, 0, st>>>(labels, graphs, seq_len, width, words, scan, community_ids,
                                                    community_counts);
  return launch_check();
}
