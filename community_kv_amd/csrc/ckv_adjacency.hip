// The coalesced token graph of the prefill's top-k edges (reference:
// graph/partition.py:168-249): per row of graph g at position p with columns
// c_i of score s_i, the direct edges (p, c_i) of weight s_i * lam / 2 and, when
// lam < 1, the co-occurrence edges (c_i, c_j), i <= j, of weight
// s_i * s_j * (1 - lam); equal (min, max) pairs summed, pairs in order.
//
// A row of 8 columns stands for 44 entries, 46.9 M for a 32k layer of 32 query
// heads, so the entries are never written: a vertex's edges to higher ids are
// gathered from the rows that name it.
//
//   posting_kernel    one (vertex, entry) pair per column, and one per row
//                     whose position lies below one of its columns
//   radix sort        pairs by vertex, stable: a vertex's postings are a run in row order
//   list_kernel       the runs, in two lists by length
//   gather_kernel     one wave per short run: each posting's row is read, the neighbours
//                     above the vertex gather in an LDS hash table (f64 sums) and leave
//                     ordered by id
//   gather_big_kernel the same by one workgroup per long run
//                     (the longest in parts, each added to a sum per id in memory)
//   gather_dense_kernel  the sums of the longest in a row; vertices with more
//                     neighbours than that table holds, summed in LDS by rank
//   scan + emit_kernel   edges to their places in the output
//
// Rows of few entries (those without co-occurrence edges, lam = 1, and of one
// column) are written out and sorted by pair all the same: there a posting,
// which looks at all columns of its row, stands for one entry or two.
//
//   expand_kernel     the entries, 64-bit keys (min, max)
//   radix sort, reduce_by_key, unpack_kernel
//
// 32 x 32,751 rows without co-occurrence edges, 8 and 16 columns: 1,080 and
// 3,850 us by postings, 730 and 1,280 so; 32 x 4,023 rows of 64: 2,030 and 630;
// 32 x 32,758 of one column with them 500 and 345; of two: 500 by postings, 530
// sorted.  By postings they also took scratch for kappa + 1 edges a posting.
//
// The sums are f64 sums of the f32 entry weights, rounded once, on both ways.
//
// Measured on 32 x 32,751 rows of 8 (9.8 M edges out): 2.9 ms for the expansion, the
// 64-bit radix sort of its 46.9 M entries and their reduction before,
// 1.2 ms so.  What bounds it now: the random reads of the rows (32 bytes
// of columns and of scores per posting, from L2 and the Infinity Cache) and
// the LDS inserts.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <type_traits>

#include "ckv_amd.h"
#include "ckv_error.h"
#include "ckv_sort.h"
#include "ckv_table.h"

namespace ckv {
namespace {

constexpr int THREADS = 256;
constexpr int WAVE_SLOTS = 512;        // LDS table of one wave: 6 KB
constexpr int WAVE_CANDIDATES = 448;   // candidates of a short run at most (table load 7/8)
constexpr int WAVES = 4;               // waves per workgroup: a run's length decides how long its wave holds the
                                       // workgroup's LDS, so workgroups are small (24 KB, six fill a compute unit)
constexpr int WAVE_BLOCKS = 1536;
constexpr int FLIGHT = 4;              // candidates a thread has in flight: postings, then their rows, then the inserts
constexpr int BIG_THREADS = 256;
constexpr int BIG_SLOTS = 2048;        // 24 KB
constexpr int BIG_MOST = 960;          // neighbours after which a vertex leaves for the dense list
static_assert(BIG_MOST + FLIGHT * BIG_THREADS < BIG_SLOTS, "every insert between two checks finds a place");
constexpr int BIG_BLOCKS = 1280;       // (four a compute unit at once: 24 KB + the id bitmap of 32k vertices)
constexpr int MAP_WORDS = 4096;        // id bitmap of a graph: up to 131,072 vertices
constexpr int DENSE_THREADS = 1024;
constexpr int DENSE_IDS = 32 * MAP_WORDS;  // ids per bitmap
constexpr int DENSE_SUMS = 14336;      // f64 sums per pass: 112 KB beside the bitmap's 32 KB
constexpr int DENSE_BLOCKS = 256;
constexpr int SPLIT_MIN = 4096;        // postings from which a run is taken by several workgroups
constexpr int PART = 1024;             // postings of a part, at most PARTS_MOST of a run
constexpr int PARTS_MOST = 1024;
static_assert(SPLIT_MIN >= 4 * PART, "parts are full but for the last");

struct TopkGraph {
  const int32_t* idx;    // [G * R][K]
  const float* sc;       // [G * R][K]
  const int64_t* pos;    // [G * R]
  int32_t G, R, K, S;
  int shift;             // bits of a posting below its row
  float half_lam, co_lam;
};

// Postings [first, last) of one vertex.
struct Run {
  uint32_t first, last;
};

// Postings [first, last) of the run that starts at posting `run`.
struct Part {
  uint32_t run, first, last;
};

enum { LIST_SHORT = 0, LIST_LONG = 1, LIST_SPLIT = 2, LIST_PARTS = 3, LIST_DENSE = 4, LIST_TICKET = 5,
       LIST_DENSE_TICKET = 6, LIST_WORDS = 8 };

// A posting names (row << shift) | i: column i of the row, or (i == K) its
// position.  A position is a posting only if one of the row's columns lies
// above it: then that direct edge starts at the position (a causal prefill has
// none).  The pair of (i, row) stands at i * rows + row, so the stores of
// consecutive rows are consecutive.
template <int KT>
__global__ __launch_bounds__(THREADS) void posting_kernel(TopkGraph t, uint32_t* __restrict__ keys,
                                                          uint32_t* __restrict__ vals, int32_t* __restrict__ lists) {
  const int K = KT ? KT : t.K;
  const int64_t rows = (int64_t)t.G * t.R;
  const int64_t row = (int64_t)blockIdx.x * THREADS + threadIdx.x;
  if (row < LIST_WORDS) lists[row] = 0;  // no run listed yet
  if (row >= rows) return;
  const int32_t base = (int32_t)(row / t.R) * t.S;
  const uint32_t none = (uint32_t)(t.G * t.S);  // sorts last
  const int64_t p = t.pos[row];
  bool above = false;
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const int32_t c = t.idx[row * K + i];
    const bool ok = c >= 0 && c < t.S;
    above = above || (ok && c > p);
    keys[i * rows + row] = ok ? (uint32_t)(base + c) : none;
    vals[i * rows + row] = ((uint32_t)row << t.shift) | (uint32_t)i;
  }
  keys[K * rows + row] = (above && p >= 0 && p < t.S) ? (uint32_t)(base + (int32_t)p) : none;
  vals[K * rows + row] = ((uint32_t)row << t.shift) | (uint32_t)K;
}

// A candidate edge of vertex v: column j of a posting's row.
struct Candidate {
  uint32_t u;    // the neighbour (> v) when ok
  bool ok;
  float w;
  double self;   // weight it adds to the pair (v, v)
  bool has_self;
};

// What a candidate needs from memory.
struct Loaded {
  int32_t c;
  float s, si;   // scores of column j and of the posting's own column
  int64_t p;     // the row's position (lane j == i only)
};

template <int KT, bool SCORES = true>
__device__ __forceinline__ Loaded load_candidate(const TopkGraph& t, uint32_t posting, int j) {
  const int K = KT ? KT : t.K;
  const uint32_t row = posting >> t.shift;
  const int i = (int)(posting & ((1u << t.shift) - 1u));
  const int64_t at = (int64_t)row * K;
  Loaded l;
  l.c = t.idx[at + j];
  l.s = SCORES ? t.sc[at + j] : 0.0f;
  l.si = SCORES ? t.sc[at + (i < K ? i : j)] : 0.0f;
  l.p = (j == i) ? t.pos[row] : -1;
  return l;
}

// The lane of the posting's own column carries the column's pair with itself
// and the row's direct edge.
template <int KT>
__device__ __forceinline__ Candidate candidate(const TopkGraph& t, uint32_t posting, int j, const Loaded& l,
                                               int32_t v, int32_t base) {
  const int K = KT ? KT : t.K;
  const int i = (int)(posting & ((1u << t.shift) - 1u));
  Candidate r{0u, false, 0.0f, 0.0, false};
  if (i == K) {  // the vertex is the row's position: direct edges to the columns above it
    r.u = (uint32_t)(base + l.c);
    r.ok = l.c < t.S && base + l.c > v;
    r.w = l.s * t.half_lam;
  } else if (j == i) {
    const bool direct = l.p >= 0 && l.p < t.S && base + l.p >= v;
    const float w = l.s * t.half_lam;
    r.u = (uint32_t)(base + (int32_t)l.p);
    r.ok = direct && base + l.p > v;
    r.w = w;
    r.has_self = true;
    r.self += (double)((l.s * l.s) * t.co_lam);
    if (direct && !r.ok) r.self += (double)w;
  } else if (l.c >= 0 && l.c < t.S && base + l.c >= v) {
    const float w = (l.si * l.s) * t.co_lam;
    r.u = (uint32_t)(base + l.c);
    r.ok = base + l.c > v;
    r.w = w;
    r.has_self = !r.ok && j > i;  // the column again: one entry of the pair (i, j), i < j
    if (r.has_self) r.self = (double)w;
  }
  return r;
}

// Walks the candidates q = first, first + step, ... of the run that starts at
// posting a, FLIGHT at a time; add(candidate) for each, pause() after each FLIGHT
// (a true return ends the walk).  Without SCORES the weights are not read.
template <int KT, bool SCORES = true, class N, class Add, class Pause>
__device__ __forceinline__ void walk(const TopkGraph& t, const uint32_t* __restrict__ postings, uint32_t a, N n,
                                     uint32_t first, uint32_t step, int32_t v, int32_t base, Add add, Pause pause) {
  const uint32_t K = KT ? KT : (uint32_t)t.K;
  for (N q0 = 0; q0 < n; q0 += (N)FLIGHT * step) {
    uint32_t post[FLIGHT], j[FLIGHT];
    Loaded l[FLIGHT];
#pragma unroll
    for (int f = 0; f < FLIGHT; ++f) {
      const N q = q0 + (N)f * step + first;
      const N qc = q < n ? q : n - 1;  // (past the end: the last one again, not added)
      const N p = KT ? qc / (N)KT : qc / K;
      j[f] = (uint32_t)(qc - p * K);
      post[f] = postings[a + p];
    }
#pragma unroll
    for (int f = 0; f < FLIGHT; ++f) l[f] = load_candidate<KT, SCORES>(t, post[f], (int)j[f]);
#pragma unroll
    for (int f = 0; f < FLIGHT; ++f) {
      if (q0 + (N)f * step + first < n) add(candidate<KT>(t, post[f], (int)j[f], l[f], v, base));
    }
    if (pause()) break;
  }
}

// The edges of one run [a, b) of vertex v by one wave.
template <int KT>
__device__ __forceinline__ void gather_run(const TopkGraph& t, const uint32_t* __restrict__ postings, uint32_t a,
                                           uint32_t b, int32_t v, uint32_t* tk, double* ts,
                                           int32_t* __restrict__ count, uint32_t* __restrict__ tmp_id,
                                           float* __restrict__ tmp_w) {
  const int ln = lane();
  const int32_t base = v / t.S * t.S;
  const uint32_t n = (b - a) * (uint32_t)t.K;
  const uint32_t size = table_size(min(n, (uint32_t)(base + t.S - v)), WAVE_SLOTS);
  for (uint32_t j = ln; j < size; j += 64) {
    tk[j] = EMPTY;
    ts[j] = 0.0;
  }
  wave_lds_sync();
  double self = 0.0;
  bool any_self = false;
  walk<KT>(t, postings, a, n, (uint32_t)ln, 64u, v, base,
           [&](const Candidate& c) {
             any_self = any_self || c.has_self;
             self += c.self;
             if (c.ok) insert(tk, ts, size, c.u, c.w, nullptr);  // (never more ids than the table holds)
           },
           [] { return false; });
  wave_lds_sync();
  self = wave_sum_f64(self);
  const int lead = __ballot(any_self) != 0 ? 1 : 0;
  // Compact the occupied slots to the front (every lane has read its slots
  // before any is overwritten), then order them by counting smaller ids.
  constexpr int PER = WAVE_SLOTS / 64;
  uint32_t k[PER];
  float w[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (64u * i >= size) break;  // (a multiple of 64; most runs have a table of 64 or 128)
    const uint32_t j = ln + 64 * i;
    k[i] = tk[j];
    w[i] = k[i] != EMPTY ? (float)ts[j] : 0.0f;
  }
  wave_lds_sync();
  float* tw = reinterpret_cast<float*>(ts);
  int m = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (64u * i >= size) break;
    const uint64_t used = __ballot(k[i] != EMPTY);
    if (k[i] != EMPTY) {
      const int at = m + __popcll(used & ((((uint64_t)1) << ln) - 1));
      tk[at] = k[i];
      tw[at] = w[i];
    }
    m += __popcll(used);
  }
  if (ln < 4 && m + ln < WAVE_SLOTS) tk[m + ln] = EMPTY;  // fills the last group of four
  wave_lds_sync();
  const int64_t out = (int64_t)a * (t.K + 1);
  if (lead && ln == 0) {
    tmp_id[out] = (uint32_t)v;
    tmp_w[out] = (float)self;
  }
  for (int i = ln; i < m; i += 64) {
    const uint32_t mine = tk[i];
    int rank = 0;
    for (int j = 0; j < m; j += 4) {
      const uint4 o = *reinterpret_cast<const uint4*>(tk + j);
      rank += (o.x < mine) + (o.y < mine) + (o.z < mine) + (o.w < mine);
    }
    tmp_id[out + lead + rank] = mine;
    tmp_w[out + lead + rank] = tw[i];
  }
  if (ln == 0) count[a] = lead + m;
  wave_lds_sync();  // the wave's next run clears the table
}

// End of the run of v that starts before `end` and goes on there: the first
// posting of another vertex in [end, n], found by probing 64 places at a time
// (the interval narrows 63-fold per round).
__device__ inline uint32_t run_end(const uint32_t* __restrict__ keys, uint32_t end, uint32_t n, uint32_t v) {
  uint32_t lo = end, hi = n, step = 1;
  while (lo < hi) {
    const uint32_t at = lo + (uint32_t)lane() * step;
    const uint64_t other = __ballot(at >= hi || keys[at < hi ? at : hi - 1] != v);
    const uint32_t f = other ? (uint32_t)__builtin_ctzll(other) : 64u;  // probes below f are of v, probe f is not
    if (f < 64) hi = min(lo + f * step, hi);
    if (f > 0) lo = min(lo + (f - 1) * step + 1, hi);
    step = max(1u, (hi - lo + 62) / 63);
  }
  return lo;
}

// Lists the runs by their length.  A workgroup takes LIST_GROUPS x 1,024
// postings and reserves its places in a list at once: with one reservation per
// wave, 294,000 atomics on two words took 870 us.
constexpr int LIST_THREADS = 1024;
constexpr int LIST_GROUPS = 4;

__global__ __launch_bounds__(LIST_THREADS) void list_kernel(const uint32_t* __restrict__ keys, uint32_t n, uint32_t V,
                                                            uint32_t short_most, uint32_t split_min,
                                                            int32_t* __restrict__ count, Run* __restrict__ short_runs,
                                                            Run* __restrict__ long_runs, Run* __restrict__ split_runs,
                                                            Part* __restrict__ parts, int32_t* __restrict__ lists) {
  __shared__ int s_n[2], s_at[2];
  const int ln = lane();
  const uint64_t below = (((uint64_t)1) << ln) - 1;
  if (threadIdx.x < 2) s_n[threadIdx.x] = 0;
  __syncthreads();
  uint32_t stop[LIST_GROUPS];
  int place[LIST_GROUPS];  // in the workgroup's part of list `kind`
  int kind[LIST_GROUPS];
  constexpr int NONE = -1;
#pragma unroll
  for (int g = 0; g < LIST_GROUPS; ++g) {
    const uint32_t here = (blockIdx.x * LIST_GROUPS + g) * LIST_THREADS + threadIdx.x;
    const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)here);
    const bool in = here < n;
    const uint32_t key = in ? keys[here] : EMPTY;
    const bool start = in && (here == 0 || keys[here - 1] != key);
    const uint64_t starts = __ballot(start);
    if (in) count[here] = 0;  // runs that have edges store their number later
    const bool mine = start && key < V;
    const uint64_t real = __ballot(mine);
    uint32_t end = first + 64 < n ? first + 64 : n;
    if (real != 0 && end < n) {
      const int last = 63 - __builtin_clzll(starts);
      if ((real >> last) & 1) end = run_end(keys, end, n, (uint32_t)__builtin_amdgcn_readlane((int)key, last));
    }
    const uint64_t later = ln == 63 ? 0ull : starts >> (ln + 1);
    stop[g] = later ? here + 1 + (uint32_t)__builtin_ctzll(later) : end;
    const uint32_t length = stop[g] - here;
    kind[g] = !mine ? NONE : length <= short_most ? LIST_SHORT : length < split_min ? LIST_LONG : LIST_SPLIT;
    const uint64_t ms = __ballot(kind[g] == LIST_SHORT), ml = __ballot(kind[g] == LIST_LONG);
    int bs = 0, bl = 0;
    if (ln == 0) {
      if (ms) bs = atomicAdd(s_n, __popcll(ms));
      if (ml) bl = atomicAdd(s_n + 1, __popcll(ml));
    }
    bs = __builtin_amdgcn_readfirstlane(bs);
    bl = __builtin_amdgcn_readfirstlane(bl);
    place[g] = kind[g] == LIST_SHORT ? bs + __popcll(ms & below) : bl + __popcll(ml & below);
  }
  __syncthreads();
  if (threadIdx.x < 2) s_at[threadIdx.x] = s_n[threadIdx.x] ? atomicAdd(lists + threadIdx.x, s_n[threadIdx.x]) : 0;
  __syncthreads();
#pragma unroll
  for (int g = 0; g < LIST_GROUPS; ++g) {
    const uint32_t here = (blockIdx.x * LIST_GROUPS + g) * LIST_THREADS + threadIdx.x;
    if (kind[g] == LIST_SHORT) short_runs[s_at[0] + place[g]] = Run{here, stop[g]};
    if (kind[g] == LIST_LONG) long_runs[s_at[1] + place[g]] = Run{here, stop[g]};
    if (kind[g] == LIST_SPLIT) {  // (few: n / split_min at most)
      const uint32_t length = stop[g] - here;
      const uint32_t size = max((uint32_t)PART, (length + PARTS_MOST - 1) / PARTS_MOST);
      const uint32_t many = (length + size - 1) / size;
      split_runs[atomicAdd(lists + LIST_SPLIT, 1)] = Run{here, stop[g]};
      Part* to = parts + atomicAdd(lists + LIST_PARTS, (int)many);
      for (uint32_t i = 0; i < many; ++i) to[i] = Part{here, here + i * size, min(here + (i + 1) * size, stop[g])};
    }
  }
}

// The edges of the run that starts at posting a wait in tmp at a * (K + 1): a
// posting brings at most K neighbours, the run one pair with itself; count[a]
// holds their number (0 at postings that start no run).
//
// A split run's edges first stand as a sum per id from its vertex on, in the
// ids' part of that place (a split run is long enough for them: split_length).
// A sum that nothing was added to is -0.0: what is added is no -0.0, so no sum
// becomes it.
__host__ __device__ inline uint32_t split_length(int32_t S, int32_t K) {
  const uint32_t fits = (uint32_t)((2 * (int64_t)S + 2 + K) / (K + 1));
  return fits > (uint32_t)SPLIT_MIN ? fits : (uint32_t)SPLIT_MIN;
}
template <int KT>
__device__ __forceinline__ double* split_sums(const TopkGraph& t, uint32_t a, uint32_t* tmp_id) {
  const int64_t out = (int64_t)a * ((KT ? KT : t.K) + 1);
  return reinterpret_cast<double*>(tmp_id + ((out + 1) & ~(int64_t)1));
}
constexpr double NOTHING = -0.0;
__device__ inline bool is_nothing(double x) { return __builtin_bit_cast(uint64_t, x) == 0x8000000000000000ull; }
constexpr int CHUNK = 4096;  // ids of a split run that a workgroup clears or copies at a time

template <int KT>
__global__ __launch_bounds__(64 * WAVES) void gather_kernel(TopkGraph t, const uint32_t* __restrict__ keys,
                                                            const uint32_t* __restrict__ postings,
                                                            const Run* __restrict__ runs,
                                                            const Run* __restrict__ split_runs,
                                                            const int32_t* __restrict__ lists,
                                                            int32_t* __restrict__ count, uint32_t* __restrict__ tmp_id,
                                                            float* __restrict__ tmp_w) {
  __shared__ __align__(16) uint32_t tab_k[WAVES][WAVE_SLOTS];
  __shared__ double tab_s[WAVES][WAVE_SLOTS];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int32_t chunks = (t.S + CHUNK - 1) / CHUNK;
  const int64_t clear = (int64_t)lists[LIST_SPLIT] * chunks;
  for (int64_t it = blockIdx.x; it < clear; it += gridDim.x) {
    const uint32_t a = split_runs[it / chunks].first;
    const int32_t v = (int32_t)keys[a], ids = t.S - v % t.S, at = (int32_t)(it % chunks) * CHUNK;
    double* sums = split_sums<KT>(t, a, tmp_id);
    for (int i = at + threadIdx.x; i < min(ids, at + CHUNK); i += 64 * WAVES) sums[i] = NOTHING;
  }
  const int32_t listed = lists[LIST_SHORT];
  for (int32_t it = blockIdx.x * WAVES + wave; it < listed; it += gridDim.x * WAVES) {
    const Run r = runs[it];
    gather_run<KT>(t, postings, r.first, r.last, (int32_t)keys[r.first], tab_k[wave], tab_s[wave], count, tmp_id,
                   tmp_w);
  }
}

// A workgroup's first item is its own number, the next ones are taken in turn
// (all threads call).  With a ticket for the first one too, 1,280 workgroups
// queued 15 us for one word, in calls with nothing to do for them as well.
__device__ inline int32_t next_ticket(int32_t* word, int* s_ticket) {
  __syncthreads();
  if (threadIdx.x == 0) *s_ticket = (int32_t)gridDim.x + atomicAdd(word, 1);
  __syncthreads();
  return *s_ticket;
}

// One workgroup per part of a split run and per long run (taken in turn by a
// ticket: their lengths differ by a hundredfold).  A part's neighbours gather
// in the LDS table as far as BIG_MOST of them go (the ones that many rows name
// come early) and are added to the run's sums at its end; the others are added
// there at once.
//
// A long run's neighbours: up to BIG_MOST in the table; a vertex that has more
// goes to the dense list.  They are ordered by a bitmap of the graph's vertices
// (words of it dynamic LDS, with a running count per word): the set bits below
// an id are its rank.  Counting smaller ids instead, as the waves do for their
// few, grows with the square (and orders graphs of more vertices than the
// bitmap has).
template <int KT>
__global__ __launch_bounds__(BIG_THREADS) void gather_big_kernel(
    TopkGraph t, const uint32_t* __restrict__ keys, const uint32_t* __restrict__ postings,
    const Run* __restrict__ runs, const Part* __restrict__ parts, Run* __restrict__ dense, int32_t* lists,
    int32_t* __restrict__ count, uint32_t* __restrict__ tmp_id, float* __restrict__ tmp_w) {
  __shared__ __align__(16) uint32_t tk[BIG_SLOTS];
  __shared__ double ts[BIG_SLOTS];
  extern __shared__ uint32_t map_s[];  // [words] bits, [words] set bits before the word
  __shared__ double red[BIG_THREADS / 64];
  __shared__ int wave_n[BIG_THREADS / 64];
  __shared__ int s_added, s_self, s_ticket;
  const int tid = threadIdx.x, wv = tid >> 6, ln = lane();
  const int32_t split = lists[LIST_PARTS], listed = split + lists[LIST_LONG];
  const int words = t.S <= 32 * MAP_WORDS ? (t.S + 31) >> 5 : 0;
  uint32_t* before_s = map_s + words;
  for (int32_t it = (int32_t)blockIdx.x; it < listed; it = next_ticket(lists + LIST_TICKET, &s_ticket)) {
    if (it < split) {
      const Part part = parts[it];
      const int32_t v = (int32_t)keys[part.run];
      const int32_t base = v / t.S * t.S;
      double* sums = split_sums<KT>(t, part.run, tmp_id);
      for (uint32_t j = tid; j < BIG_SLOTS; j += BIG_THREADS) {
        tk[j] = EMPTY;
        ts[j] = 0.0;
      }
      if (tid == 0) s_added = 0;
      __syncthreads();
      double self = 0.0;
      bool any_self = false;
      walk<KT>(t, postings, part.first, (uint64_t)(part.last - part.first) * (uint32_t)t.K, (uint32_t)tid, BIG_THREADS,
               v, base,
               [&](const Candidate& c) {
                 any_self = any_self || c.has_self;
                 self += c.self;
                 if (c.ok && !insert_few(tk, ts, BIG_SLOTS, c.u, c.w, &s_added, BIG_MOST))
                   unsafeAtomicAdd(sums + (c.u - (uint32_t)v), (double)c.w + 0.0);  // (no -0.0)
               },
               [] { return false; });
      self = wave_sum_f64(self);
      if (__ballot(any_self) != 0 && ln == 0) unsafeAtomicAdd(sums, self + 0.0);
      __syncthreads();
      for (uint32_t j = tid; j < BIG_SLOTS; j += BIG_THREADS) {
        if (tk[j] != EMPTY) unsafeAtomicAdd(sums + (tk[j] - (uint32_t)v), ts[j] + 0.0);
      }
      __syncthreads();
      continue;
    }
    const uint32_t a = runs[it - split].first, b = runs[it - split].last;
    const int32_t v = (int32_t)keys[a];
    const int32_t base = v / t.S * t.S;
    const uint64_t n = (uint64_t)(b - a) * (uint32_t)t.K;
    const uint64_t room = (uint64_t)(base + t.S - v);
    const uint32_t size = table_size(n < room ? n : room, BIG_SLOTS);
    for (uint32_t j = tid; j < size; j += BIG_THREADS) {
      tk[j] = EMPTY;
      ts[j] = 0.0;
    }
    for (int j = tid; j < words; j += BIG_THREADS) map_s[j] = 0u;
    if (tid == 0) s_added = s_self = 0;
    __syncthreads();
    double self = 0.0;
    bool any_self = false;
    walk<KT>(t, postings, a, n, (uint32_t)tid, BIG_THREADS, v, base,
             [&](const Candidate& c) {
               any_self = any_self || c.has_self;
               self += c.self;
               if (c.ok) insert(tk, ts, size, c.u, c.w, &s_added);
             },
             [&] {
               if (size < BIG_SLOTS) return false;  // room for every candidate
               __syncthreads();
               const bool full = s_added > BIG_MOST;
               __syncthreads();
               return full;
             });
    self = wave_sum_f64(self);
    if (ln == 0) red[wv] = self;
    if (any_self) s_self = 1;
    __syncthreads();
    if (s_added > BIG_MOST) {
      if (tid == 0) dense[atomicAdd(lists + LIST_DENSE, 1)] = Run{a, b};
      __syncthreads();
      continue;
    }
    const int lead = s_self;
    double total = 0.0;
    for (int i = 0; i < BIG_THREADS / 64; ++i) total += red[i];
    const int64_t out = (int64_t)a * (t.K + 1);
    if (lead && tid == 0) {
      tmp_id[out] = (uint32_t)v;
      tmp_w[out] = (float)total;
    }
    // Thread t holds the slots t, t + 256, ...
    constexpr int PER = BIG_SLOTS / BIG_THREADS;
    uint32_t k[PER];
    float w[PER];
    int own = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const uint32_t j = tid + BIG_THREADS * i;
      k[i] = j < size ? tk[j] : EMPTY;
      w[i] = k[i] != EMPTY ? (float)ts[j] : 0.0f;
      own += k[i] != EMPTY ? 1 : 0;
      if (words > 0 && k[i] != EMPTY) {
        const uint32_t d = k[i] - (uint32_t)base;
        atomicOr(map_s + (d >> 5), 1u << (d & 31));
      }
    }
    __syncthreads();
    const int per = (words + BIG_THREADS - 1) / BIG_THREADS;  // consecutive map words of a thread
    int mine = own;
    if (words > 0) {
      mine = 0;
      for (int i = 0; i < per; ++i) {
        const int j = tid * per + i;
        if (j < words) mine += __popc(map_s[j]);
      }
    }
    int incl = mine;
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(incl, o);
      if (ln >= o) incl += y;
    }
    if (ln == 63) wave_n[wv] = incl;
    __syncthreads();
    int at = incl - mine, m = 0;
    for (int i = 0; i < BIG_THREADS / 64; ++i) {
      if (i < wv) at += wave_n[i];
      m += wave_n[i];
    }
    if (words > 0) {
      for (int i = 0; i < per; ++i) {
        const int j = tid * per + i;
        if (j < words) {
          before_s[j] = (uint32_t)at;
          at += __popc(map_s[j]);
        }
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        if (k[i] != EMPTY) {
          const uint32_t d = k[i] - (uint32_t)base;
          const int rank = (int)before_s[d >> 5] + __popc(map_s[d >> 5] & ((1u << (d & 31)) - 1u));
          tmp_id[out + lead + rank] = k[i];
          tmp_w[out + lead + rank] = w[i];
        }
      }
    } else {
      float* tw = reinterpret_cast<float*>(ts);
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        if (k[i] != EMPTY) {
          tk[at] = k[i];
          tw[at] = w[i];
          ++at;
        }
      }
      if (tid < 4) tk[m + tid] = EMPTY;  // (m <= BIG_MOST: never a compacted place)
      __syncthreads();
      for (int i = tid; i < m; i += BIG_THREADS) {
        int rank = 0;
        for (int j = 0; j < m; j += 4) {
          const uint4 o = *reinterpret_cast<const uint4*>(tk + j);
          rank += (o.x < tk[i]) + (o.y < tk[i]) + (o.z < tk[i]) + (o.w < tk[i]);
        }
        tmp_id[out + lead + rank] = tk[i];
        tmp_w[out + lead + rank] = tw[i];
      }
    }
    if (tid == 0) count[a] = lead + m;
    __syncthreads();
  }
}

// The runs that one LDS table does not hold.
//
// Split runs: a workgroup puts the sums that something was added to in a row.
// Ids take the place of the sums: those of a round are read before they are
// overwritten, and an id is half as long as a sum, so no later one is.
//
// Vertices of one workgroup with more than BIG_MOST neighbours: their rows are
// read once for a bitmap of the neighbours, whose set bits below an id are its
// rank, and once for every DENSE_SUMS ranks, whose sums lie in LDS in order
// (graphs of more than DENSE_IDS vertices: bitmap by bitmap).  A pass per
// window of 16,384 consecutive ids instead read the rows of a vertex with a few
// thousand neighbours eight times at 131,072 positions.
//
// The whole graph of 32 heads in 8 graphs at 131,072 positions, columns drawn by
// a power law: 9.2 ms; planted columns and one that all rows name 5.6, with all
// heads in one graph 8.1; at 32,768 positions 1.4 and 1.3.  (Every run on one
// workgroup: 26.4 ms, 30.9, 207; 3.5, 16.1.  The sort of all entries that the
// gathering replaced: 11.5, 11.4, 9.7; 2.7, 2.2.)
constexpr size_t dense_lds_bytes() { return DENSE_SUMS * 8 + MAP_WORDS * 8; }

// Block-wide exclusive scan of one int per thread; the total in *sum.
__device__ __forceinline__ int dense_scan(int x, int* wave_n, int* sum) {
  const int wv = threadIdx.x >> 6;
  int incl = x;
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(incl, o);
    if (lane() >= o) incl += y;
  }
  if (lane() == 63) wave_n[wv] = incl;
  __syncthreads();
  int at = incl - x, all = 0;
  for (int i = 0; i < DENSE_THREADS / 64; ++i) {
    if (i < wv) at += wave_n[i];
    all += wave_n[i];
  }
  __syncthreads();
  *sum = all;
  return at;
}

template <int KT>
__global__ __launch_bounds__(DENSE_THREADS) void gather_dense_kernel(
    TopkGraph t, const uint32_t* __restrict__ keys, const uint32_t* __restrict__ postings,
    const Run* __restrict__ split_runs, const Run* __restrict__ dense, int32_t* lists, int32_t* __restrict__ count,
    uint32_t* tmp_id, float* __restrict__ tmp_w) {
  extern __shared__ double dense_s[];
  uint32_t* map = reinterpret_cast<uint32_t*>(dense_s + DENSE_SUMS);
  uint32_t* below = map + MAP_WORDS;  // neighbours in the words before
  __shared__ double red[DENSE_THREADS / 64];
  __shared__ int wave_n[DENSE_THREADS / 64], s_ticket;
  constexpr int OWN = MAP_WORDS / DENSE_THREADS;  // consecutive words of a thread
  const int tid = threadIdx.x, wv = tid >> 6;
  const int32_t split = lists[LIST_SPLIT], listed = split + lists[LIST_DENSE];
  for (int32_t it = (int32_t)blockIdx.x; it < listed; it = next_ticket(lists + LIST_DENSE_TICKET, &s_ticket)) {
    if (it < split) {
      constexpr int U = 4;
      const uint32_t a = split_runs[it].first;
      const int32_t v = (int32_t)keys[a], ids = t.S - v % t.S;
      const int64_t out = (int64_t)a * (t.K + 1);
      const double* sums = split_sums<KT>(t, a, tmp_id);
      int done = 0;
      for (int i0 = 0; i0 < ids; i0 += U * DENSE_THREADS) {
        double x[U];
        int own = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int i = i0 + U * tid + u;
          x[u] = i < ids ? sums[i] : NOTHING;
          own += is_nothing(x[u]) ? 0 : 1;
        }
        int m;
        int64_t at = out + done + dense_scan(own, wave_n, &m);  // (its barriers: all sums of the round are read)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (!is_nothing(x[u])) {
            tmp_id[at] = (uint32_t)(v + i0 + U * tid + u);
            tmp_w[at] = (float)x[u];
            ++at;
          }
        }
        done += m;
        __syncthreads();
      }
      if (tid == 0) count[a] = done;
      continue;
    }
    const uint32_t a = dense[it - split].first, b = dense[it - split].last;
    const int32_t v = (int32_t)keys[a];
    const int32_t base = v / t.S * t.S;
    const uint64_t n = (uint64_t)(b - a) * (uint32_t)t.K;
    const int64_t out = (int64_t)a * (t.K + 1);
    int done = 0;
    for (int32_t lo = v; lo < base + t.S; lo += DENSE_IDS) {
      for (int j = tid; j < MAP_WORDS; j += DENSE_THREADS) map[j] = 0u;
      __syncthreads();
      bool any_self = false;
      walk<KT, false>(t, postings, a, n, (uint32_t)tid, DENSE_THREADS, v, base,
                      [&](const Candidate& c) {
                        any_self = any_self || c.has_self;
                        const uint32_t d = c.u - (uint32_t)lo;  // (below lo: beyond the bitmap)
                        if (c.ok && d < (uint32_t)DENSE_IDS) atomicOr(map + (d >> 5), 1u << (d & 31));
                      },
                      [] { return false; });
      const int lead = __syncthreads_or(any_self ? 1 : 0) != 0 && lo == v ? 1 : 0;
      int mine = 0, m;
#pragma unroll
      for (int i = 0; i < OWN; ++i) mine += __popc(map[OWN * tid + i]);
      int at = dense_scan(mine, wave_n, &m);
      done += lead;
      for (int i = 0; i < OWN; ++i) {
        uint32_t bits = map[OWN * tid + i];
        below[OWN * tid + i] = (uint32_t)at;
        for (; bits != 0; bits &= bits - 1, ++at)
          tmp_id[out + done + at] = (uint32_t)lo + 32u * (uint32_t)(OWN * tid + i) + (uint32_t)__builtin_ctz(bits);
      }
      for (int r0 = 0; r0 == 0 || r0 < m; r0 += DENSE_SUMS) {
        const int ranks = min(m - r0, DENSE_SUMS);
        for (int j = tid; j < ranks; j += DENSE_THREADS) dense_s[j] = 0.0;
        __syncthreads();
        double self = 0.0;
        walk<KT>(t, postings, a, n, (uint32_t)tid, DENSE_THREADS, v, base,
                 [&](const Candidate& c) {
                   self += c.self;
                   const uint32_t d = c.u - (uint32_t)lo;
                   if (c.ok && d < (uint32_t)DENSE_IDS) {
                     const int r = (int)below[d >> 5] + __popc(map[d >> 5] & ((1u << (d & 31)) - 1u)) - r0;
                     if (r >= 0 && r < ranks) unsafeAtomicAdd(dense_s + r, (double)c.w);
                   }
                 },
                 [] { return false; });
        if (lead != 0 && r0 == 0) {
          self = wave_sum_f64(self);
          if (lane() == 0) red[wv] = self;
        }
        __syncthreads();
        if (lead != 0 && r0 == 0 && tid == 0) {
          double total = 0.0;
          for (int i = 0; i < DENSE_THREADS / 64; ++i) total += red[i];
          tmp_id[out] = (uint32_t)v;
          tmp_w[out] = (float)total;
        }
        for (int j = tid; j < ranks; j += DENSE_THREADS) tmp_w[out + done + r0 + j] = (float)dense_s[j];
        __syncthreads();
      }
      done += m;
    }
    if (tid == 0) count[a] = done;
  }
}

// Copies the runs' edges to their places, a wave per run; a workgroup per dense
// run and per CHUNK of a split one.  The last posting's place ends the output.
__global__ __launch_bounds__(64 * WAVES) void emit_kernel(const uint32_t* __restrict__ keys,
                                                          const int32_t* __restrict__ count,
                                                          const int32_t* __restrict__ place,
                                                          const Run* __restrict__ short_runs,
                                                          const Run* __restrict__ long_runs,
                                                          const Run* __restrict__ split_runs,
                                                          const Run* __restrict__ dense_runs,
                                                          const int32_t* __restrict__ lists, uint32_t n, int32_t K,
                                                          int32_t S, const uint32_t* __restrict__ tmp_id,
                                                          const float* __restrict__ tmp_w, int32_t* __restrict__ out_src,
                                                          int32_t* __restrict__ out_dst, float* __restrict__ out_w,
                                                          int64_t* __restrict__ out_count) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int32_t chunks = (S + CHUNK - 1) / CHUNK;
  const int64_t pieces = (int64_t)lists[LIST_SPLIT] * chunks, items = pieces + lists[LIST_DENSE];
  for (int64_t it = blockIdx.x; it < items; it += gridDim.x) {
    const bool piece = it < pieces;
    const uint32_t a = (piece ? split_runs[it / chunks] : dense_runs[it - pieces]).first;
    const int i0 = piece ? (int)(it % chunks) * CHUNK : 0;
    const int m = piece ? min(count[a], i0 + CHUNK) : count[a], at = place[a], v = (int)keys[a];
    const int64_t from = (int64_t)a * (K + 1);
#pragma unroll 4
    for (int i = i0 + (int)threadIdx.x; i < m; i += 64 * WAVES) {
      out_src[at + i] = v;
      out_dst[at + i] = (int32_t)tmp_id[from + i];
      out_w[at + i] = tmp_w[from + i];
    }
  }
  const int32_t shorts = lists[LIST_SHORT], listed = shorts + lists[LIST_LONG];
  for (int32_t it = blockIdx.x * WAVES + wave; it < listed; it += gridDim.x * WAVES) {
    const uint32_t a = (it < shorts ? short_runs[it] : long_runs[it - shorts]).first;
    const int m = count[a], at = place[a], v = (int)keys[a];
    if (m > BIG_MOST + 1) continue;  // a dense run: copied above
    const int64_t from = (int64_t)a * (K + 1);
    for (int i = lane(); i < m; i += 64) {
      out_src[at + i] = v;
      out_dst[at + i] = (int32_t)tmp_id[from + i];
      out_w[at + i] = tmp_w[from + i];
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) *out_count = (int64_t)place[n - 1] + count[n - 1];
}

// ----------------------------------------------------------------- entries sorted by pair
// Entry i of a row: the direct edges, then the co-occurrence pairs of the upper
// triangle, row-major.  Entries with a column or position outside the sequence
// carry the sentinel key, which sorts last.
__global__ __launch_bounds__(THREADS) void expand_kernel(TopkGraph t, int per_row, int bits,
                                                         uint64_t* __restrict__ keys, float* __restrict__ vals) {
  const int64_t i = (int64_t)blockIdx.x * THREADS + threadIdx.x;
  if (i >= (int64_t)t.G * t.R * per_row) return;
  const int64_t row = i / per_row, at = row * t.K, base = row / t.R * t.S;
  int e = (int)(i - row * per_row);
  int64_t a, b;  // the ends' positions
  float w;
  if (e < t.K) {
    a = t.pos[row];
    b = t.idx[at + e];
    w = t.sc[at + e] * t.half_lam;
  } else {
    int r = 0;
    for (e -= t.K; e >= t.K - r; ++r) e -= t.K - r;
    a = t.idx[at + r];
    b = t.idx[at + r + e];
    w = (t.sc[at + r] * t.sc[at + r + e]) * t.co_lam;
  }
  const bool ok = a >= 0 && a < t.S && b >= 0 && b < t.S;
  const uint64_t lo = (uint64_t)(base + (a < b ? a : b)), hi = (uint64_t)(base + (a < b ? b : a));
  keys[i] = ok ? (lo << bits) | hi : (uint64_t)((int64_t)t.G * t.S) << bits;
  vals[i] = ok ? w : 0.0f;
}

// Ends of the pairs; a sentinel among them is the last and no edge.
__global__ __launch_bounds__(THREADS) void unpack_kernel(const uint64_t* __restrict__ pairs,
                                                         const int64_t* __restrict__ count, int bits, uint64_t V,
                                                         int32_t* __restrict__ out_src, int32_t* __restrict__ out_dst,
                                                         int64_t* __restrict__ out_count) {
  const int64_t n = *count, i = (int64_t)blockIdx.x * THREADS + threadIdx.x;
  if (i == 0) *out_count = (pairs[n - 1] >> bits) >= V ? n - 1 : n;
  if (i >= n) return;
  const uint64_t k = pairs[i];
  out_src[i] = (int32_t)(k >> bits);
  out_dst[i] = (int32_t)(k & (((uint64_t)1 << bits) - 1));
}

struct AsDouble {
  __host__ __device__ double operator()(float x) const { return (double)x; }
};
using DoubleOf = rocprim::transform_iterator<const float*, AsDouble, double>;

hipError_t sort_entries(void* temp, size_t& bytes, const uint64_t* keys_in, uint64_t* keys, const float* vals_in,
                        float* vals, size_t n, int end_bit, hipStream_t st) {
  return rocprim::radix_sort_pairs(temp, bytes, keys_in, keys, vals_in, vals, n, 0, (unsigned)end_bit, st);
}
hipError_t sum_entries(void* temp, size_t& bytes, const uint64_t* keys, const float* vals, size_t n, uint64_t* pairs,
                       float* sums, int64_t* count, hipStream_t st) {
  return rocprim::reduce_by_key(temp, bytes, keys, DoubleOf(vals, AsDouble()), n, pairs, sums, count,
                                rocprim::plus<double>(), rocprim::equal_to<uint64_t>(), st);
}

// pairs takes the place of keys_in (free once they are sorted).
struct SortLayout {
  size_t keys_in, keys, vals_in, vals, count, temp, temp_bytes, total;
};

SortLayout sort_layout(int64_t n) {
  SortLayout L{};
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off += align256(bytes);
    return at;
  };
  size_t sort = 0, sum = 0;
  (void)sort_entries(nullptr, sort, nullptr, nullptr, nullptr, nullptr, (size_t)n, 64, (hipStream_t)0);
  (void)sum_entries(nullptr, sum, nullptr, nullptr, (size_t)n, nullptr, nullptr, nullptr, (hipStream_t)0);
  L.keys_in = take((size_t)n * 8);
  L.keys = take((size_t)n * 8);
  L.vals_in = take((size_t)n * 4);
  L.vals = take((size_t)n * 4);
  L.count = take(8);
  L.temp_bytes = sort > sum ? sort : sum;
  L.temp = take(L.temp_bytes);
  L.total = off;
  return L;
}

// Rows of at most two entries, or without co-occurrence edges.
inline bool by_entries(int32_t kappa, float lam) { return !(lam < 1.0f) || kappa == 1; }

// ----------------------------------------------------------------- host side
struct AdjLayout {
  size_t keys_in, vals_in, keys, vals, temp, temp_bytes, count, place, short_runs, long_runs, split_runs, parts, dense,
      lists, tmp_id, tmp_w, total;
};

// n: postings (rows x (kappa + 1)).  A long run has more than WAVE_CANDIDATES / kappa of them.
AdjLayout adj_layout(int64_t n, int32_t kappa) {
  AdjLayout L{};
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off += align256(bytes);
    return at;
  };
  const size_t sort = sort_pairs_bytes((size_t)n), scan = scan_bytes((size_t)n);
  const size_t runs = (size_t)n / (size_t)(WAVE_CANDIDATES / kappa + 1) + 1;
  L.keys_in = take((size_t)n * 4);
  L.vals_in = take((size_t)n * 4);
  L.keys = take((size_t)n * 4);
  L.vals = take((size_t)n * 4);
  L.count = take((size_t)n * 4);
  L.place = take((size_t)n * 4);
  L.short_runs = take((size_t)n * sizeof(Run));
  L.long_runs = take(runs * sizeof(Run));
  L.dense = take(runs * sizeof(Run));
  L.split_runs = take(((size_t)n / SPLIT_MIN + 1) * sizeof(Run));
  L.parts = take(((size_t)n / PART + (size_t)n / SPLIT_MIN + 1) * sizeof(Part));
  L.lists = take(LIST_WORDS * 4);
  L.temp_bytes = sort > scan ? sort : scan;
  L.temp = take(L.temp_bytes);
  L.tmp_id = take((size_t)n * (size_t)(kappa + 1) * 4);
  L.tmp_w = take((size_t)n * (size_t)(kappa + 1) * 4);
  L.total = off;
  return L;
}

inline unsigned blocks_for(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

inline int64_t adjacency_entries(int32_t graphs, int32_t rows, int32_t kappa, float lam) {
  const int per_row = kappa + (lam < 1.0f ? kappa * (kappa + 1) / 2 : 0);
  return (int64_t)graphs * rows * per_row;
}
inline int64_t adjacency_postings(int32_t graphs, int32_t rows, int32_t kappa) {
  return (int64_t)graphs * rows * (kappa + 1);
}

int launch_check() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : ckv_internal::set_error(CKV_E_LAUNCH, hipGetErrorString(e));
}

}  // namespace
}  // namespace ckv

using namespace ckv;

extern "C" size_t ckv_adjacency_workspace_bytes(int32_t graphs, int32_t rows, int32_t kappa, float lam) {
  if (graphs <= 0 || rows <= 0 || kappa <= 0) return 0;
  if (by_entries(kappa, lam)) return sort_layout(adjacency_entries(graphs, rows, kappa, lam)).total;
  return adj_layout(adjacency_postings(graphs, rows, kappa), kappa).total;
}

extern "C" int64_t ckv_adjacency_capacity(int32_t graphs, int32_t rows, int32_t kappa, float lam) {
  if (graphs <= 0 || rows < 0 || kappa <= 0) return 0;
  return adjacency_entries(graphs, rows, kappa, lam);
}

extern "C" int ckv_build_adjacency(const int32_t* topk_indices, const float* topk_scores,
                                   const int64_t* query_positions, int32_t graphs, int32_t rows, int32_t kappa,
                                   int32_t seq_len, float lam, int32_t* out_src, int32_t* out_dst, float* out_weight,
                                   int64_t* out_count, void* workspace, void* stream) {
  if (graphs <= 0 || rows < 0 || kappa <= 0 || kappa > 64 || seq_len <= 0 || !out_count || !(lam >= 0.0f && lam <= 1.0f))
    return ckv_internal::set_error(CKV_E_INVALID, "bad adjacency sizes (kappa <= 64, lam in [0, 1])");
  hipStream_t st = (hipStream_t)stream;
  if (rows == 0) {
    if (hipMemsetAsync(out_count, 0, 8, st) != hipSuccess) return launch_check();
    return 0;
  }
  if (!topk_indices || !topk_scores || !query_positions || !out_src || !out_dst || !out_weight || !workspace)
    return ckv_internal::set_error(CKV_E_INVALID, "null adjacency pointer");
  const int64_t V = (int64_t)graphs * seq_len;
  const int64_t n = adjacency_postings(graphs, rows, kappa);
  if (adjacency_entries(graphs, rows, kappa, lam) >= ((int64_t)1 << 31) - 1 || V >= (int64_t)1 << 30)
    return ckv_internal::set_error(CKV_E_LIMIT, "adjacency too large");
  const TopkGraph t{topk_indices, topk_scores, query_positions, graphs, rows, kappa, seq_len,
                    bits_for((uint64_t)kappa), lam / 2.0f, 1.0f - lam};
  char* ws = (char*)workspace;
  if (by_entries(kappa, lam)) {
    const int64_t entries = adjacency_entries(graphs, rows, kappa, lam);
    const SortLayout L = sort_layout(entries);
    uint64_t* keys_in = (uint64_t*)(ws + L.keys_in);
    uint64_t* sorted = (uint64_t*)(ws + L.keys);
    float* vals_in = (float*)(ws + L.vals_in);
    float* vals = (float*)(ws + L.vals);
    int64_t* pairs = (int64_t*)(ws + L.count);
    const int bits = bits_for((uint64_t)V - 1);
    expand_kernel<<<blocks_for(entries, THREADS), THREADS, 0, st>>>(t, (int)(entries / ((int64_t)graphs * rows)), bits,
                                                                   keys_in, vals_in);
    size_t temp = L.temp_bytes;
    if (sort_entries(ws + L.temp, temp, keys_in, sorted, vals_in, vals, (size_t)entries, bits + bits_for((uint64_t)V),
                     st) != hipSuccess)
      return ckv_internal::set_error(CKV_E_LAUNCH, "entry sort failed");
    temp = L.temp_bytes;
    if (sum_entries(ws + L.temp, temp, sorted, vals, (size_t)entries, keys_in, out_weight, pairs, st) != hipSuccess)
      return ckv_internal::set_error(CKV_E_LAUNCH, "entry sum failed");
    unpack_kernel<<<blocks_for(entries, THREADS), THREADS, 0, st>>>(keys_in, pairs, bits, (uint64_t)V, out_src, out_dst,
                                                                   out_count);
    return launch_check();
  }
  const AdjLayout L = adj_layout(n, kappa);
  uint32_t* keys_in = (uint32_t*)(ws + L.keys_in);
  uint32_t* vals_in = (uint32_t*)(ws + L.vals_in);
  uint32_t* keys = (uint32_t*)(ws + L.keys);
  uint32_t* vals = (uint32_t*)(ws + L.vals);
  int32_t* count = (int32_t*)(ws + L.count);
  int32_t* place = (int32_t*)(ws + L.place);
  Run* short_runs = (Run*)(ws + L.short_runs);
  Run* long_runs = (Run*)(ws + L.long_runs);
  Run* dense = (Run*)(ws + L.dense);
  Run* split_runs = (Run*)(ws + L.split_runs);
  Part* parts = (Part*)(ws + L.parts);
  int32_t* lists = (int32_t*)(ws + L.lists);
  uint32_t* tmp_id = (uint32_t*)(ws + L.tmp_id);
  float* tmp_w = (float*)(ws + L.tmp_w);
  // A vertex has fewer neighbours than its graph has vertices; in a graph small
  // enough for every table runs are split, and that launch paid for (5 us of
  // some 200), where it has rows enough to make one workgroup long.
  const bool heavy = seq_len > BIG_MOST || (int64_t)rows * (kappa + 1) >= 16 * SPLIT_MIN;
  const uint32_t split_min = heavy ? split_length(seq_len, kappa) : UINT32_MAX;
  auto gather = [&](auto width) -> int {
    constexpr int KT = decltype(width)::value;
    posting_kernel<KT><<<blocks_for((int64_t)graphs * rows, THREADS), THREADS, 0, st>>>(t, keys_in, vals_in, lists);
    if (sort_pairs(ws + L.temp, L.temp_bytes, keys_in, keys, vals_in, vals, (size_t)n, bits_for((uint64_t)V), st) !=
        hipSuccess)
      return ckv_internal::set_error(CKV_E_LAUNCH, "posting sort failed");
    list_kernel<<<blocks_for(n, LIST_GROUPS * LIST_THREADS), LIST_THREADS, 0, st>>>(
        keys, (uint32_t)n, (uint32_t)V, (uint32_t)(WAVE_CANDIDATES / kappa), split_min, count,
        short_runs, long_runs, split_runs, parts, lists);
    gather_kernel<KT><<<WAVE_BLOCKS, 64 * WAVES, 0, st>>>(t, keys, vals, short_runs, split_runs, lists, count, tmp_id,
                                                         tmp_w);
    const size_t map_bytes = seq_len <= 32 * MAP_WORDS ? (size_t)((seq_len + 31) / 32) * 8 : 0;
    gather_big_kernel<KT><<<BIG_BLOCKS, BIG_THREADS, map_bytes, st>>>(t, keys, vals, long_runs, parts, dense, lists,
                                                                      count, tmp_id, tmp_w);
    if (heavy) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gather_dense_kernel<KT>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)dense_lds_bytes());
      if (e != hipSuccess) {
        (void)hipGetLastError();
        return ckv_internal::set_error(CKV_E_LAUNCH, hipGetErrorString(e));
      }
      gather_dense_kernel<KT><<<DENSE_BLOCKS, DENSE_THREADS, dense_lds_bytes(), st>>>(
          t, keys, vals, split_runs, dense, lists, count, tmp_id, tmp_w);
    }
    return 0;
  };
  // the reference's edge width has its own code (divisions become shifts)
  const int rc = kappa == 8 ? gather(std::integral_constant<int, 8>{})
                            : kappa == 16 ? gather(std::integral_constant<int, 16>{})
                                          : gather(std::integral_constant<int, 0>{});
  if (rc != 0) return rc;
  if (exclusive_scan_i32(ws + L.temp, L.temp_bytes, count, place, (size_t)n, st) != hipSuccess)
    return ckv_internal::set_error(CKV_E_LAUNCH, "edge scan failed");
  emit_kernel<<<2048, 64 * WAVES, 0, st>>>(keys, count, place, short_runs, long_runs, split_runs, dense, lists,
                                           (uint32_t)n, kappa, seq_len, tmp_id, tmp_w, out_src, out_dst, out_weight,
                                           out_count);
  return launch_check();
}
