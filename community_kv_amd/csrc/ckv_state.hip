// Prefill graph state assembled on the GPU from dense community labels: the
// recency-descending membership CSR, FP8 (or f32) centroid tables with their
// community sizes, the modularity weights of the prefill edges and the
// per-token community table.  Restates the reference's state build after
// Leiden (graph/partition.py:382-535, called from build_partitioned_layer
// 538-618).
//
// Every integer output is exact, and the centroid sums follow one fixed order
// (a community's members in ascending position order, in blocks of 64: each
// block summed in order by one wave, lane = two dims, then the block sums
// added in order), so they are reproducible bit for bit; blocks spread a large
// community over many waves.  The modularity weights add edge weights with
// float atomics, like the reference's scatter_add_; their summation order is
// not fixed.
//
// Launch sequence of ckv_build_layer_state (one stream):
//   state_prep_kernel     per (graph, position chunk): community histogram; in further
//                         workgroups labels -> token_communities (-1 past the prompt)
//                         and the modularity weights cleared
//   chunk_scan_kernel     per (graph, community): its members in newer chunks, its total
//   csr_scan_kernel       per graph: CSR offsets and the table of 64-member blocks
//   csr_scatter_kernel    per (graph, chunk): member positions, newest first
//   block_sum_kernel      per (retrieval head, block): in-order key sum of 64 members; the
//                         centroid of a community of one block
//   centroid_kernel       per (retrieval head, community of several blocks or none): block
//                         sums in order, mean -> clamp -> E4M3 / f32
//   edge_weight_kernel    modularity weights from an edge list, or
//   topk_weight_kernel    the same weights from the prefill top-k edges
#include <hip/hip_runtime.h>

#include <algorithm>

#include <stdint.h>

#include "ckv_device.h"
#include "ckv_error.h"

namespace ckv {
namespace {

constexpr int MAX_CHUNKS = 64;           // position chunks per graph (histogram / scatter)
constexpr int MIN_CHUNK = 512;
constexpr int SUM_BLOCK = 64;            // members per centroid partial sum
constexpr int COUNT_THREADS = 1024;
constexpr int SCAN_THREADS = 1024;
constexpr int HIST_THREADS = 256;
constexpr int STATE_LDS_COMMUNITIES = 16384;  // per-community LDS counters of one kernel (64 KB)
constexpr int CENTROID_WAVES = 4;        // community rows per centroid workgroup
constexpr int EDGE_THREADS = 256;

// Positions per chunk: at least MIN_CHUNK, at most MAX_CHUNKS chunks, a multiple of 64.
inline int state_chunk(int seq_len, int num_sink) {
  const int n = seq_len - num_sink;
  int c = (n + MAX_CHUNKS - 1) / MAX_CHUNKS;
  c = (c + 63) / 64 * 64;
  return c < MIN_CHUNK ? MIN_CHUNK : c;
}
inline int state_chunks(int seq_len, int num_sink) {
  const int n = seq_len - num_sink;
  return n <= 0 ? 0 : (n + state_chunk(seq_len, num_sink) - 1) / state_chunk(seq_len, num_sink);
}
// Upper bound of the 64-member blocks of one graph.
inline int64_t state_max_blocks(int seq_len, int num_sink, int maxc) {
  return (int64_t)(seq_len - num_sink + SUM_BLOCK - 1) / SUM_BLOCK + maxc;
}

// Workspace carve-up (int32 units): histograms, block starts, block communities, f32 partial sums.
struct StateWorkspace {
  int32_t* hist;       // [graphs][chunks][maxc]
  int32_t* blk_first;  // [graphs][maxc + 1]
  int32_t* blk_comm;   // [graphs][max_blocks]
  float* partial;      // [retrieval_heads][max_blocks][128]
};

inline size_t state_ws_words(int graphs, int heads, int seq_len, int num_sink, int maxc, StateWorkspace* w,
                             int32_t* base) {
  const int64_t chunks = state_chunks(seq_len, num_sink);
  const int64_t mb = state_max_blocks(seq_len, num_sink, maxc);
  size_t off = 0;
  auto take = [&](int64_t words) {
    const size_t at = off;
    off += (size_t)((words + 63) / 64 * 64);  // 256-byte aligned pieces
    return at;
  };
  const size_t h = take((int64_t)graphs * chunks * maxc);
  const size_t bf = take((int64_t)graphs * (maxc + 1));
  const size_t bc = take((int64_t)graphs * mb);
  const size_t pt = take((int64_t)heads * mb * D);
  if (w && base) {
    w->hist = base + h;
    w->blk_first = base + bf;
    w->blk_comm = base + bc;
    w->partial = reinterpret_cast<float*>(base + pt);
  }
  return off;
}

// community_counts[g] = 1 + the largest label of a non-sink position, 0 when
// there is none, -1 when a non-sink label is negative.  One workgroup per
// graph, bound by load latency: eight loads of a thread are in flight together
// (32,768 positions: 10.8 us with one, 4.4 us with eight).
__global__ __launch_bounds__(COUNT_THREADS) void label_count_kernel(const int32_t* __restrict__ labels, int seq_len,
                                                                    int num_sink, int32_t* __restrict__ counts) {
  constexpr int U = 8;
  const int g = blockIdx.x;
  const int32_t* row = labels + (int64_t)g * seq_len;
  int mx = -1, mn = 0;
  for (int p0 = num_sink + threadIdx.x; p0 < seq_len; p0 += U * COUNT_THREADS) {
    int v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = gload_i32(row + min(p0 + u * COUNT_THREADS, seq_len - 1));  // (the last label again)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      mx = max(mx, v[u]);
      mn = min(mn, v[u]);
    }
  }
  __shared__ int s_max[COUNT_THREADS / 64], s_min[COUNT_THREADS / 64];
  mx = wave_max_i32(mx);
  mn = -wave_max_i32(-mn);
  if ((threadIdx.x & 63) == 0) {
    s_max[threadIdx.x >> 6] = mx;
    s_min[threadIdx.x >> 6] = mn;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 0; w < COUNT_THREADS / 64; ++w) {
      mx = max(mx, s_max[w]);
      mn = min(mn, s_min[w]);
    }
    counts[g] = mn < 0 ? -1 : mx + 1;
  }
}

// Everything that needs the labels alone, in one launch.  Workgroups below
// graphs * chunks: hist[g][chunk][c] = members of community c among the
// chunk's positions (communities below lds_n are counted in LDS, the others in
// the output row).  The others fill the token table and clear the weights.
__global__ __launch_bounds__(HIST_THREADS) void state_prep_kernel(
    const int32_t* __restrict__ labels, int seq_len, int num_sink, int maxc, int lds_n, int chunk_len, int chunks,
    int graphs, int32_t* __restrict__ hist, int token_capacity, int32_t* __restrict__ tokens,
    float* __restrict__ weight, int64_t weights, float* __restrict__ total) {
  extern __shared__ int h_s[];
  if ((int)blockIdx.x >= graphs * chunks) {
    const int64_t i0 = (int64_t)(blockIdx.x - graphs * chunks) * HIST_THREADS + threadIdx.x;
    const int64_t step = (int64_t)(gridDim.x - graphs * chunks) * HIST_THREADS;
    const int64_t all = (int64_t)graphs * token_capacity;
    for (int64_t i = i0; i < all; i += step) {
      const int g = (int)(i / token_capacity);
      const int t = (int)(i - (int64_t)g * token_capacity);
      tokens[i] = t < seq_len ? labels[(int64_t)g * seq_len + t] : -1;
    }
    if (weight != nullptr) {
      for (int64_t i = i0; i < weights; i += step) weight[i] = 0.0f;
      for (int64_t i = i0; i < graphs; i += step) total[i] = 0.0f;
    }
    return;
  }
  const int chunk = blockIdx.x % chunks, g = blockIdx.x / chunks;
  int32_t* out = hist + ((int64_t)g * chunks + chunk) * maxc;
  for (int c = threadIdx.x; c < lds_n; c += HIST_THREADS) h_s[c] = 0;
  for (int c = lds_n + threadIdx.x; c < maxc; c += HIST_THREADS) out[c] = 0;
  wait_vm();  // the zeroed row is in place before any workgroup thread adds to it
  __syncthreads();
  const int32_t* row = labels + (int64_t)g * seq_len;
  const int p0 = num_sink + chunk * chunk_len;
  const int p1 = min(p0 + chunk_len, seq_len);
  for (int p = p0 + threadIdx.x; p < p1; p += HIST_THREADS) {
    const int c = row[p];
    if (c >= 0 && c < lds_n) atomicAdd(h_s + c, 1);
    else if (c >= lds_n && c < maxc) atomicAdd(out + c, 1);
  }
  __syncthreads();
  for (int c = threadIdx.x; c < lds_n; c += HIST_THREADS) out[c] = h_s[c];
}

// Per (graph, community): hist[chunk][c] becomes the members of c in later
// chunks (the CSR is recency descending), offsets[c] the community's total.
// Spread over all compute units: with one workgroup per graph walking every
// community's chunks, 13,000 communities took 146 us.
__global__ __launch_bounds__(HIST_THREADS) void chunk_scan_kernel(int maxc, int chunks, int32_t* __restrict__ hist,
                                                                  int32_t* __restrict__ offsets) {
  const int g = blockIdx.y;
  const int c = blockIdx.x * HIST_THREADS + threadIdx.x;
  if (c >= maxc) return;
  int32_t* h = hist + (int64_t)g * chunks * maxc + c;
  int run = 0;
  for (int i0 = chunks - 1; i0 >= 0; i0 -= 16) {  // sixteen loads in flight, then their stores
    int n[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) n[u] = gload_i32(h + (int64_t)max(i0 - u, 0) * maxc);
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      if (i0 - u >= 0) {
        h[(int64_t)(i0 - u) * maxc] = run;
        run += n[u];
      }
    }
  }
  offsets[(int64_t)g * (maxc + 1) + c] = run;
}

// Per graph: the communities' totals (in offsets) become CSR offsets and block
// starts, in place; each thread scans a run of consecutive communities, so the
// workgroup scans once.
__global__ __launch_bounds__(SCAN_THREADS) void csr_scan_kernel(int maxc, int64_t max_blocks,
                                                                int32_t* __restrict__ offsets,
                                                                int32_t* __restrict__ blk_first,
                                                                int32_t* __restrict__ blk_comm) {
  const int g = blockIdx.x;
  const int tid = threadIdx.x;
  int32_t* off = offsets + (int64_t)g * (maxc + 1);
  int32_t* bf = blk_first + (int64_t)g * (maxc + 1);
  int32_t* bc = blk_comm + (int64_t)g * max_blocks;
  __shared__ int s_wave[SCAN_THREADS / 64], s_wblk[SCAN_THREADS / 64];
  const int per = (maxc + SCAN_THREADS - 1) / SCAN_THREADS;
  const int c0 = min(tid * per, maxc), c1 = min(c0 + per, maxc);
  int t = 0, nb = 0;
#pragma unroll 4
  for (int c = c0; c < c1; ++c) {
    const int n = off[c];
    t += n;
    nb += (n + SUM_BLOCK - 1) / SUM_BLOCK;
  }
  const int inc = wave_inclusive_scan(t);
  const int incb = wave_inclusive_scan(nb);
  if ((tid & 63) == 63) {
    s_wave[tid >> 6] = inc;
    s_wblk[tid >> 6] = incb;
  }
  __syncthreads();
  int base = inc - t, bbase = incb - nb;
  for (int wv = 0; wv < (tid >> 6); ++wv) {
    base += s_wave[wv];
    bbase += s_wblk[wv];
  }
#pragma unroll 4
  for (int c = c0; c < c1; ++c) {
    const int n = off[c];
    const int b = (n + SUM_BLOCK - 1) / SUM_BLOCK;
    off[c] = base;
    bf[c] = bbase;
    for (int j = 0; j < b; ++j) bc[bbase + j] = c;
    base += n;
    bbase += b;
  }
  if (tid == SCAN_THREADS - 1) {
    off[maxc] = base;
    bf[maxc] = bbase;
  }
}

// One wave per (graph, chunk): walks the chunk's positions from the newest
// down, 64 at a time (lane l takes the l-th newest).  Lanes with equal labels
// find each other bit by bit (one ballot per label bit: at most 17 rounds
// against one per distinct label, 122 us at 512 communities and 8 x 32,768
// positions before, 8.2 us now), the lanes before a lane in its set
// rank it, and the set's first lane advances the community's cursor.
// Cursors of communities below lds_n live in LDS (members of the chunk placed
// so far; the community's first slot is prefetched for SCATTER_GROUPS groups at
// a time), the others in the chunk's histogram row (which nothing reads
// afterwards).
constexpr int SCATTER_GROUPS = 8;

__global__ __launch_bounds__(64) void csr_scatter_kernel(const int32_t* __restrict__ labels, int seq_len, int num_sink,
                                                         int maxc, int label_bits, int lds_n, int chunk_len, int chunks,
                                                         const int32_t* __restrict__ offsets, int32_t* hist,
                                                         int32_t* __restrict__ member_positions) {
  extern __shared__ int cur_s[];
  const int chunk = blockIdx.x, g = blockIdx.y;
  const int lane = threadIdx.x;
  int32_t* h = hist + ((int64_t)g * chunks + chunk) * maxc;
  const int32_t* off = offsets + (int64_t)g * (maxc + 1);
  for (int c = lane; c < lds_n; c += 64) cur_s[c] = 0;
  wave_sync();
  const int32_t* row = labels + (int64_t)g * seq_len;
  int32_t* out = member_positions + (int64_t)g * (seq_len - num_sink);
  const int p0 = num_sink + chunk * chunk_len;
  const int p1 = min(p0 + chunk_len, seq_len);
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (int top0 = p1 - 1; top0 >= p0; top0 -= 64 * SCATTER_GROUPS) {
    int lab[SCATTER_GROUPS], first[SCATTER_GROUPS], later[SCATTER_GROUPS];
#pragma unroll
    for (int u = 0; u < SCATTER_GROUPS; ++u) lab[u] = gload_i32(row + max(top0 - 64 * u - lane, p0));
#pragma unroll
    for (int u = 0; u < SCATTER_GROUPS; ++u) {
      const int c = min(max(lab[u], 0), maxc - 1);
      first[u] = gload_i32(off + c);
      later[u] = gload_i32(h + c);
    }
#pragma unroll
    for (int u = 0; u < SCATTER_GROUPS; ++u) {
      const int p = top0 - 64 * u - lane;
      const int c = lab[u];
      const bool valid = p >= p0 && c >= 0 && c < maxc;
      uint64_t peers = __ballot(valid);
      if (peers == 0) continue;
      for (int b = 0; b < label_bits; ++b) {
        const bool bit = (c >> b) & 1;
        const uint64_t m = __ballot(bit);
        peers &= bit ? m : ~m;
      }
      const int rank = __popcll(peers & below), size = __popcll(peers);
      const bool in_lds = valid && c < lds_n;
      const bool in_row = valid && c >= lds_n;
      int at = 0;
      if (in_lds) at = first[u] + later[u] + cur_s[c];
      if (in_row) at = first[u] + __hip_atomic_load(h + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      wave_sync();
      if (rank == 0 && in_lds) cur_s[c] += size;
      if (__ballot(in_row)) {
        if (rank == 0 && in_row) __hip_atomic_fetch_add(h + c, size, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        wait_vm();  // the cursors are advanced before a later group reads them
      }
      wave_sync();
      if (valid) out[at + rank] = p;
    }
  }
}

// Sum and finish of a centroid row (lane = dims 2l and 2l+1): mean, clamp to
// +-448, then E4M3 or f32.
template <int CT>
__device__ __forceinline__ void store_mean(float s0, float s1, int size, bool divide, int64_t row, int lane,
                                           void* __restrict__ centroids, int32_t* __restrict__ sizes) {
  if (divide) {
    const float den = (float)max(size, 1);
    s0 = s0 / den;
    s1 = s1 / den;
  }
  s0 = fminf(fmaxf(s0, -448.0f), 448.0f);
  s1 = fminf(fmaxf(s1, -448.0f), 448.0f);
  if constexpr (CT == CKV_E4M3) {
    const uint16_t pair = (uint16_t)(ckv_f32_to_e4m3(s0) | ((uint16_t)ckv_f32_to_e4m3(s1) << 8));
    reinterpret_cast<uint16_t*>(centroids)[row * (D / 2) + lane] = pair;
  } else {
    float* dst = reinterpret_cast<float*>(centroids) + row * D + 2 * lane;
    dst[0] = s0;
    dst[1] = s1;
  }
  if (lane == 0) sizes[row] = size;
}

// Loads N rows (lanes past n of `mine` repeat the last member) in one round and
// adds the first n of them in order.
template <int KT, int N>
__device__ __forceinline__ void sum_rows(const void* __restrict__ keys, int64_t kb, int64_t token_stride, int mine,
                                         int n, float& s0, float& s1) {
  constexpr int W = KT == CKV_BF16 ? 1 : 2;
  uint32_t x[N][W];
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const int p = __builtin_amdgcn_readlane(mine, u);
    if constexpr (KT == CKV_BF16) {
      x[u][0] = (uint32_t)gload_i32(reinterpret_cast<const int32_t*>(reinterpret_cast<const uint16_t*>(keys) + kb +
                                                                     (int64_t)p * token_stride));
    } else {
      const float* kp = reinterpret_cast<const float*>(keys) + kb + (int64_t)p * token_stride;
      x[u][0] = ckv_f2u(gload_f32(kp));
      x[u][W - 1] = ckv_f2u(gload_f32(kp + 1));
    }
  }
#pragma unroll
  for (int u = 0; u < N; ++u) {
    if (u < n) {
      s0 = s0 + (KT == CKV_BF16 ? ckv_u2f(x[u][0] << 16) : ckv_u2f(x[u][0]));
      s1 = s1 + (KT == CKV_BF16 ? ckv_u2f(x[u][0] & 0xffff0000u) : ckv_u2f(x[u][W - 1]));
    }
  }
}

// One wave per (retrieval head, 64-member block): members 64k .. 64k+63 of
// community c in ascending position order (the CSR lists them newest first),
// summed in order in f32, lane = dims 2l and 2l+1.  All rows are loaded
// before the sum, so a block costs one gather round; a block of few members
// loads 4 or 16 rows instead of 64 (communities of a Leiden partition have two
// or three members on average: 120 us with 64 rows each, 8 x 13,000 of them, 54 us
// so).  A community of one block is finished here.
template <int KT, int CT>
__global__ __launch_bounds__(64 * CENTROID_WAVES) void block_sum_kernel(
    const void* __restrict__ keys, int64_t head_stride, int64_t token_stride, const int32_t* __restrict__ to_graph,
    const int32_t* __restrict__ to_kv, const int32_t* __restrict__ offsets, const int32_t* __restrict__ positions,
    const int32_t* __restrict__ blk_first, const int32_t* __restrict__ blk_comm, int64_t max_blocks, int seq_len,
    int num_sink, int maxc, int capacity, float* __restrict__ partial, void* __restrict__ centroids,
    int32_t* __restrict__ sizes) {
  const int r = blockIdx.y;
  const int64_t b = (int64_t)blockIdx.x * CENTROID_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int g = to_graph[r];
  const int kvh = to_kv[r];
  if (b >= blk_first[(int64_t)g * (maxc + 1) + maxc]) return;  // past this graph's blocks
  const int c = blk_comm[(int64_t)g * max_blocks + b];
  const int k = (int)(b - blk_first[(int64_t)g * (maxc + 1) + c]);
  const int lo = offsets[(int64_t)g * (maxc + 1) + c];
  const int hi = offsets[(int64_t)g * (maxc + 1) + c + 1];
  const int i0 = SUM_BLOCK * k;  // ascending member index of the block's first member
  const int n = min(SUM_BLOCK, hi - lo - i0);
  const int32_t* mem = positions + (int64_t)g * (seq_len - num_sink);
  const int mine = mem[hi - 1 - (i0 + min(lane, n - 1))];
  const int64_t kb = (int64_t)kvh * head_stride + 2 * lane;
  float s0 = 0.0f, s1 = 0.0f;  // (+0 start: an all-negative-zero block sums to +0, as scatter_add_ does)
  if (n <= 4) sum_rows<KT, 4>(keys, kb, token_stride, mine, n, s0, s1);
  else if (n <= 16) sum_rows<KT, 16>(keys, kb, token_stride, mine, n, s0, s1);
  else sum_rows<KT, SUM_BLOCK>(keys, kb, token_stride, mine, n, s0, s1);
  if (hi - lo <= SUM_BLOCK) {
    store_mean<CT>(s0, s1, hi - lo, true, (int64_t)r * capacity + c, lane, centroids, sizes);
    return;
  }
  float* dst = partial + ((int64_t)r * max_blocks + b) * D + 2 * lane;
  dst[0] = s0;
  dst[1] = s1;
}

// One wave per (retrieval head, community row) of several blocks or none: the
// block sums added in order, divided by its size.  Rows at or past maxc hold
// zeros.
template <int CT>
__global__ __launch_bounds__(64 * CENTROID_WAVES) void centroid_kernel(
    const int32_t* __restrict__ to_graph, const int32_t* __restrict__ offsets, const int32_t* __restrict__ blk_first,
    const float* __restrict__ partial, int64_t max_blocks, int maxc, int capacity, void* __restrict__ centroids,
    int32_t* __restrict__ sizes) {
  const int r = blockIdx.y;
  const int c = blockIdx.x * CENTROID_WAVES + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (c >= capacity) return;
  const int g = to_graph[r];
  int size = 0, b0 = 0, nb = 0;
  if (c < maxc) {
    size = offsets[(int64_t)g * (maxc + 1) + c + 1] - offsets[(int64_t)g * (maxc + 1) + c];
    b0 = blk_first[(int64_t)g * (maxc + 1) + c];
    nb = blk_first[(int64_t)g * (maxc + 1) + c + 1] - b0;
    if (nb == 1) return;  // finished by block_sum_kernel
  }
  const float* src = partial + ((int64_t)r * max_blocks + b0) * D + 2 * lane;
  float s0 = 0.0f, s1 = 0.0f;
  for (int j0 = 0; j0 < nb; j0 += 16) {
    float y0[16], y1[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const float* q = src + (int64_t)min(j0 + u, nb - 1) * D;
      y0[u] = gload_f32(q);
      y1[u] = gload_f32(q + 1);
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      if (j0 + u < nb) {
        s0 = s0 + y0[u];
        s1 = s1 + y1[u];
      }
    }
  }
  store_mean<CT>(s0, s1, size, c < maxc, (int64_t)r * capacity + c, lane, centroids, sizes);
}

// Community degree weights and 2m: each edge (graph * seq_len + position
// endpoints) adds its weight to both endpoint communities and twice to its
// graph's total.  A workgroup takes EDGES_PER_WG consecutive edges (the list
// is grouped by graph): the weights of the graph of its first edge gather in
// LDS and leave with one global atomic per touched community; edges of other
// graphs (at most a boundary's worth) add straight to global memory.
constexpr int EDGES_PER_WG = 8192;

__global__ __launch_bounds__(EDGE_THREADS) void edge_weight_kernel(
    const int32_t* __restrict__ labels, int seq_len, int graphs, int capacity, int lds_n,
    const int32_t* __restrict__ src, const int32_t* __restrict__ dst, const float* __restrict__ w, int64_t edges,
    float* __restrict__ weight, float* __restrict__ total) {
  extern __shared__ float w_s[];  // communities [0, lds_n) of the first edge's graph
  const int64_t e0 = (int64_t)blockIdx.x * EDGES_PER_WG;
  const int64_t e1 = min(edges, e0 + EDGES_PER_WG);
  const int g0 = src[e0] / seq_len;
  for (int c = threadIdx.x; c < lds_n; c += EDGE_THREADS) w_s[c] = 0.0f;
  __syncthreads();
  float mine = 0.0f;
  for (int64_t e = e0 + threadIdx.x; e < e1; e += EDGE_THREADS) {
    const int s = src[e], d = dst[e];
    const int g = s / seq_len;
    if (g < 0 || g >= graphs || d / seq_len != g) continue;
    const float x = w[e];
    const int sc = labels[(int64_t)g * seq_len + s % seq_len];
    const int dc = labels[(int64_t)g * seq_len + d % seq_len];
    if (g == g0) {
      if (sc >= 0 && sc < lds_n) atomicAdd(w_s + sc, x);
      else if (sc >= lds_n && sc < capacity) atomicAdd(weight + (int64_t)g * capacity + sc, x);
      if (dc >= 0 && dc < lds_n) atomicAdd(w_s + dc, x);
      else if (dc >= lds_n && dc < capacity) atomicAdd(weight + (int64_t)g * capacity + dc, x);
      mine = mine + 2.0f * x;
    } else {
      if (sc >= 0 && sc < capacity) atomicAdd(weight + (int64_t)g * capacity + sc, x);
      if (dc >= 0 && dc < capacity) atomicAdd(weight + (int64_t)g * capacity + dc, x);
      atomicAdd(total + g, 2.0f * x);
    }
  }
  __shared__ float s_part[EDGE_THREADS / 64];
  mine = wave_sum_tree(mine);
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = mine;
  __syncthreads();
  if (g0 >= 0 && g0 < graphs) {
    for (int c = threadIdx.x; c < lds_n; c += EDGE_THREADS) {
      const float v = w_s[c];
      if (v != 0.0f) atomicAdd(weight + (int64_t)g0 * capacity + c, v);
    }
    if (threadIdx.x == 0) {
      float t = 0.0f;
      for (int i = 0; i < EDGE_THREADS / 64; ++i) t = t + s_part[i];
      atomicAdd(total + g0, t);
    }
  }
}

// The same weights where the vertices' degrees are known (row sums of the
// graph, a self loop counted twice): an edge's two ends add its weight to
// their communities, so a community weighs the sum of its members' degrees.
// 262,144 degrees in place of 9.8 M edges with two label reads and LDS adds
// each: 488 us (8 graphs of 32,768, 13,000 communities) and 1,434 us (32 of
// 8,192) in edge_weight_kernel, 110 us with the totals here.
constexpr int DEGREE_THREADS = 256;

__global__ __launch_bounds__(DEGREE_THREADS) void degree_weight_kernel(
    const int32_t* __restrict__ labels, const double* __restrict__ degree, int seq_len, int graphs, int capacity,
    float* __restrict__ weight) {
  const int64_t v = (int64_t)blockIdx.x * DEGREE_THREADS + threadIdx.x;
  if (v >= (int64_t)graphs * seq_len) return;
  const int g = (int)(v / seq_len);
  const int c = labels[v];
  const float w = (float)degree[v];
  if (c >= 0 && c < capacity && w != 0.0f) unsafeAtomicAdd(weight + (int64_t)g * capacity + c, w);
}

// The graphs' totals.  In edge_weight_kernel a block of EDGES_PER_WG edges
// sends one sum to the graph of its first edge, and the edges of the graphs
// that begin inside the block are added to their totals one by one, 8,000
// atomics on one word (430 us); the block sums arrive after about 1,500 of them
// with 8 graphs, after 4,000 with 32 (whose atomics queue with theirs).  Float
// totals of 10^5 depend on that order by up to 3e-5 (a single edge is smaller
// than half their last bit), so it is kept, with the single edges added in a
// register: one wave per graph, before and after the blocks (within 7e-6 of
// the atomics on 4,000 to 32,768 positions, 2 to 32 graphs; 100 us in all at
// 9.8 M edges: the look 14, a wave's 4,096 additions 25 twice, the blocks 36).
//
// That needs a list grouped by ascending graph with every source in a graph.
// edge_order_kernel looks; of any other list the totals add up edge by edge,
// sources outside the graphs left out.  Each of its workgroups leaves its
// finding in a word of the weights, which are cleared afterwards: no word
// needs clearing before it and the entry needs no workspace.
constexpr int REST_EARLY_PER_GRAPH = 192, REST_EARLY_MOST = 4096;
constexpr int ORDER_MOST = 1024;  // words a workgroup reads to know what was found

__global__ __launch_bounds__(EDGE_THREADS) void edge_order_kernel(const int32_t* __restrict__ src, int64_t edges,
                                                                  int seq_len, int64_t vertices,
                                                                  int* __restrict__ found) {
  constexpr int U = 8;
  const int64_t step = (int64_t)gridDim.x * EDGE_THREADS;
  bool loose = false;
  for (int64_t e0 = (int64_t)blockIdx.x * EDGE_THREADS + threadIdx.x; e0 < edges; e0 += U * step) {
    int a[U], b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t e = min(e0 + u * step, edges - 1);
      b[u] = gload_i32(src + e);
      a[u] = gload_i32(src + (e > 0 ? e - 1 : 0));
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      loose = loose || b[u] < 0 || b[u] >= vertices || (a[u] > b[u] && a[u] / seq_len > b[u] / seq_len);
  }
  const int any = __syncthreads_or(loose ? 1 : 0);
  if (threadIdx.x == 0) found[blockIdx.x] = any ? 1 : 0;
}

// Whether any of the n words holds a finding (every thread of the workgroup calls).
__device__ inline bool any_found(const int* __restrict__ found, int n) {
  int mine = 0;
#pragma unroll 4
  for (int i = threadIdx.x; i < n; i += blockDim.x) mine |= found[i];
  return __syncthreads_or(mine) != 0;
}

__global__ __launch_bounds__(EDGE_THREADS) void edge_total_kernel(const int32_t* __restrict__ src,
                                                                  const float* __restrict__ w, int64_t edges,
                                                                  int seq_len, int graphs,
                                                                  const int* __restrict__ found, int founds,
                                                                  float* __restrict__ total) {
  constexpr int U = 8;
  const int64_t e0 = (int64_t)blockIdx.x * EDGES_PER_WG;
  const int64_t e1 = min(edges, e0 + EDGES_PER_WG);
  const bool loose = any_found(found, founds);
  const int g0 = src[e0] / seq_len;
  const bool whole = !loose && src[e1 - 1] / seq_len == g0;
  const bool g0_ok = !loose || (src[e0] >= 0 && g0 < graphs);
  float mine = 0.0f;
  for (int64_t b = e0 + threadIdx.x; b < e1; b += U * EDGE_THREADS) {
    float x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t e = min(b + u * EDGE_THREADS, e1 - 1);
      x[u] = gload_f32(w + e);
      if (!whole) {
        const int s = src[e];
        const int g = s / seq_len;
        if (loose && s >= 0 && g < graphs && (g != g0 || !g0_ok) && b + u * EDGE_THREADS < e1)
          unsafeAtomicAdd(total + g, 2.0f * x[u]);
        if (s < 0 || g != g0) x[u] = 0.0f;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (b + u * EDGE_THREADS < e1) mine = mine + 2.0f * x[u];
    }
  }
  __shared__ float s_part[EDGE_THREADS / 64];
  mine = wave_sum_tree(mine);
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = mine;
  __syncthreads();
  if (threadIdx.x == 0 && g0_ok) {
    float t = 0.0f;
    for (int i = 0; i < EDGE_THREADS / 64; ++i) t = t + s_part[i];
    unsafeAtomicAdd(total + g0, t);
  }
}

// t plus the edges [e0, last) of graph g in order, up to the graph's end.  The
// next 64 edges are on their way while these are added, from LDS four a read:
// the additions wait for each other alone.
__device__ inline float add_edges(const int32_t* __restrict__ src, const float* __restrict__ w, int64_t e0,
                                  int64_t last, int g, int seq_len, float t) {
  __shared__ __align__(16) float x_s[64];
  const int lane = lane_id();
  if (e0 >= last) return t;
  float x = gload_f32(w + min(e0 + lane, last - 1));
  int s = gload_i32(src + min(e0 + lane, last - 1));
  for (; e0 < last; e0 += 64) {
    const int64_t next = min(e0 + 64 + lane, last - 1);
    const float xn = gload_f32(w + next);
    const int sn = gload_i32(src + next);
    const int n = __popcll(__ballot(e0 + lane < last && s / seq_len == g));
    wave_sync();  // (the reads before are done)
    x_s[lane] = 2.0f * x;
    wave_sync();
    if (n == 64) {
      float4 y[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) y[i] = reinterpret_cast<const float4*>(x_s)[i];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        t = t + y[i].x;
        t = t + y[i].y;
        t = t + y[i].z;
        t = t + y[i].w;
      }
    } else {
      for (int i = 0; i < n; ++i) t = t + x_s[i];
      break;
    }
    x = xn;
    s = sn;
  }
  return t;
}

// One wave per graph: its edges that lie in an earlier graph's block, the
// first `early` of them into a cleared total (late == 0) or the others; of a
// list in another order the cleared total alone.
__global__ __launch_bounds__(64) void edge_rest_kernel(const int32_t* __restrict__ src, const float* __restrict__ w,
                                                       int64_t edges, int seq_len, int early, int late,
                                                       const int* __restrict__ found, int founds,
                                                       float* __restrict__ total) {
  const int g = blockIdx.x;
  const int lane = threadIdx.x;
  if (any_found(found, founds)) {
    if (!late && lane == 0) total[g] = 0.0f;
    return;
  }
  const int64_t v0 = (int64_t)g * seq_len;
  // the first edge of this graph or a later one, 64 probes a round
  int64_t lo = 0, hi = edges;
  while (lo < hi) {
    const int64_t step = (hi - lo + 63) / 64;
    const int64_t at = lo + (int64_t)lane * step;
    const uint64_t here = __ballot(at >= hi || src[min(at, hi - 1)] >= v0);
    const int f = here ? __builtin_ctzll(here) : 64;  // probe f is the first at or past the graph
    const int64_t top = lo + (int64_t)f * step;
    if (f > 0) lo = lo + (int64_t)(f - 1) * step + 1;
    hi = min(hi, top);
  }
  const int64_t last = min(edges, (lo + EDGES_PER_WG - 1) / EDGES_PER_WG * EDGES_PER_WG);
  const int64_t mid = min(last, lo + early);
  const float t = late ? add_edges(src, w, mid, last, g, seq_len, total[g]) : add_edges(src, w, lo, mid, g, seq_len, 0.0f);
  if (lane == 0) total[g] = t;
}

__global__ void weight_zero_kernel(float* __restrict__ weight, int64_t n, float* __restrict__ total, int graphs) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) weight[i] = 0.0f;
  if (total != nullptr && i < graphs) total[i] = 0.0f;
}

// Modularity weights straight from the prefill top-k edges: one thread per
// (query head, row).  With the row's valid columns k (score p_k), S = sum p_k:
// the direct edges (position, column k) weigh lam/2 p_k, the co-occurrence
// edges (k, l), k <= l, weigh (1 - lam) p_k p_l.  Column k's community gains
// lam/2 p_k + (1 - lam) p_k (S + p_k) (its own pair k = k counts at both
// ends), the row position's community gains lam/2 S, and the graph's total
// 2 x (edge weights) = lam S + (1 - lam) (S^2 + sum p_k^2).  A workgroup's
// rows share one head, hence one graph: weights gather in LDS first.
//
// A workgroup walks TOPK_THREADS rows at a time over a share of its head's
// rows chosen so that about TOPK_WORKGROUPS run: what it gathered leaves with
// one global atomic per touched community, and with 256 rows per workgroup
// those (2.1 M at 32 heads x 32,751 rows, 512 communities) were most of the
// launch.  Rows of 8 or 16 edges at 16-byte aligned addresses are read with
// 16-byte loads.
//
// What bounds it are the LDS atomics: an f32 add takes some three cycles a
// lane (9.4 M of them: 115,000 of a compute unit's 142,000 cycles), an f64 add
// half of that.  So the weights gather in doubles up to TOPK_F64_COMMUNITIES,
// in floats above, where only those fit a workgroup's 64 KB.  67 MB of edges,
// 512 communities: 82 us at first, 58 us with the shares and loads above, 32 us
// in doubles.  The whole state build at 512 / 2,000 / 3,900 / 7,500
// communities: 157 / 169 / 187 / 217 us in floats, 123 / 134 / 151 / 187 in
// doubles.  (Labels kept in LDS in 16 bits instead of read from L2: 63 us.)
constexpr int TOPK_THREADS = 256;
constexpr int TOPK_WORKGROUPS = 1024;
constexpr int TOPK_F64_COMMUNITIES = 8192;  // 64 KB

template <int VEC, class W>  // VEC: 16-byte pieces of a row's edges (0: any kappa, scalar loads); W: the sums' type
__global__ __launch_bounds__(TOPK_THREADS) void topk_weight_kernel(
    const int32_t* __restrict__ labels, int seq_len, int capacity, int lds_n, const int32_t* __restrict__ idx,
    const float* __restrict__ sc, int rows, int rows_per_wg, int kappa, int group, int row0, float lam,
    float* __restrict__ weight, float* __restrict__ total) {
  constexpr int K = VEC ? 4 * VEC : 16;
  extern __shared__ double topk_lds[];
  W* w_s = reinterpret_cast<W*>(topk_lds);  // communities [0, lds_n)
  const int h = blockIdx.y;
  const int g = h / group;
  for (int c = threadIdx.x; c < lds_n; c += TOPK_THREADS) w_s[c] = W(0);
  __syncthreads();
  const int32_t* lab = labels + (int64_t)g * seq_len;
  auto add = [&](int c, float v) {
    if (c >= 0 && c < lds_n) unsafeAtomicAdd(w_s + c, (W)v);
    else if (c >= lds_n && c < capacity) unsafeAtomicAdd(weight + (int64_t)g * capacity + c, v);
  };
  const float half = 0.5f * lam, co = 1.0f - lam;
  double mine = 0.0;
  const int r1 = min(rows, (int)(blockIdx.x + 1) * rows_per_wg);
  for (int r = blockIdx.x * rows_per_wg + threadIdx.x; r < r1; r += TOPK_THREADS) {
    const int64_t at = ((int64_t)h * rows + r) * kappa;
    int col[K];
    float p[K];
    if constexpr (VEC > 0) {
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        const uint4 i4 = gload16(idx + at + 4 * v), p4 = gload16(sc + at + 4 * v);
        col[4 * v] = (int)i4.x; col[4 * v + 1] = (int)i4.y; col[4 * v + 2] = (int)i4.z; col[4 * v + 3] = (int)i4.w;
        p[4 * v] = ckv_u2f(p4.x); p[4 * v + 1] = ckv_u2f(p4.y);
        p[4 * v + 2] = ckv_u2f(p4.z); p[4 * v + 3] = ckv_u2f(p4.w);
      }
    } else {
#pragma unroll
      for (int k = 0; k < K; ++k) {
        col[k] = k < kappa ? idx[at + k] : -1;
        p[k] = k < kappa ? sc[at + k] : 0.0f;
      }
    }
    int com[K];
#pragma unroll
    for (int k = 0; k < K; ++k) com[k] = gload_i32(lab + min(max(col[k], 0), seq_len - 1));
    const int pos = row0 + r;
    const bool pos_ok = pos >= 0 && pos < seq_len;
    const int pos_com = pos_ok ? lab[pos] : -1;
    float s = 0.0f, s2 = 0.0f;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (col[k] >= 0 && col[k] < seq_len) {
        s = s + p[k];
        s2 = s2 + p[k] * p[k];
      }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (col[k] >= 0 && col[k] < seq_len) add(com[k], half * p[k] + co * (p[k] * (s + p[k])));
    }
    if (pos_ok) add(pos_com, half * s);
    mine += (double)(lam * s + co * (s * s + s2));
  }
  __shared__ double s_part[TOPK_THREADS / 64];
  for (int o = 32; o >= 1; o >>= 1) mine += __shfl_xor(mine, o);
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = mine;
  __syncthreads();
  for (int c = threadIdx.x; c < lds_n; c += TOPK_THREADS) {
    const float v = (float)w_s[c];
    if (v != 0.0f) unsafeAtomicAdd(weight + (int64_t)g * capacity + c, v);
  }
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int i = 0; i < TOPK_THREADS / 64; ++i) t += s_part[i];
    unsafeAtomicAdd(total + g, (float)t);
  }
}

int launch_check() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : ckv_internal::set_error(CKV_E_LAUNCH, hipGetErrorString(e));
}

}  // namespace
}  // namespace ckv

using namespace ckv;

extern "C" size_t ckv_state_workspace_bytes(int32_t graphs, int32_t retrieval_heads, int32_t seq_len,
                                            int32_t num_sink, int32_t max_communities) {
  if (graphs <= 0 || retrieval_heads <= 0 || seq_len <= num_sink || num_sink < 0 || max_communities <= 0) return 0;
  return state_ws_words(graphs, retrieval_heads, seq_len, num_sink, max_communities, nullptr, nullptr) *
         sizeof(int32_t);
}

extern "C" int ckv_label_counts(const int32_t* labels, int32_t graphs, int32_t seq_len, int32_t num_sink,
                                int32_t* community_counts, void* stream) {
  if (!labels || !community_counts) return ckv_internal::set_error(CKV_E_INVALID, "null label-count argument");
  if (graphs <= 0 || seq_len <= 0 || num_sink < 0)
    return ckv_internal::set_error(CKV_E_INVALID, "graphs and seq_len must be positive, num_sink nonnegative");
  hipLaunchKernelGGL(label_count_kernel, dim3(graphs), dim3(COUNT_THREADS), 0, (hipStream_t)stream, labels, seq_len,
                     num_sink, community_counts);
  return launch_check();
}

extern "C" int ckv_build_layer_state(const ckv_state_build_args* a, void* stream) {
  if (!a) return ckv_internal::set_error(CKV_E_INVALID, "null state-build argument");
  if (!a->labels || !a->keys || !a->retrieval_to_graph || !a->retrieval_to_kv || !a->member_offsets ||
      !a->member_positions || !a->centroids || !a->community_sizes || !a->token_communities || !a->workspace)
    return ckv_internal::set_error(CKV_E_INVALID, "null state-build pointer");
  if (a->graphs <= 0 || a->seq_len <= 0 || a->num_sink < 0 || a->num_sink >= a->seq_len ||
      a->retrieval_heads <= 0 || a->kv_heads <= 0)
    return ckv_internal::set_error(CKV_E_INVALID, "bad graph, head or sequence sizes (num_sink < seq_len)");
  if (a->max_communities <= 0 || a->max_communities > CKV_MAX_COMMUNITIES)
    return ckv_internal::set_error(CKV_E_LIMIT, "max_communities must be in [1, 65536]");
  if (a->community_capacity < a->max_communities)
    return ckv_internal::set_error(CKV_E_INVALID, "community_capacity must cover max_communities");
  if (a->token_capacity < a->seq_len) return ckv_internal::set_error(CKV_E_INVALID, "token_capacity < seq_len");
  if (a->key_dtype != CKV_BF16 && a->key_dtype != CKV_F32)
    return ckv_internal::set_error(CKV_E_INVALID, "key dtype must be bf16 or f32");
  if (a->centroid_dtype != CKV_E4M3 && a->centroid_dtype != CKV_F32)
    return ckv_internal::set_error(CKV_E_INVALID, "centroid dtype must be e4m3 or f32");
  if (a->head_stride <= 0 || a->token_stride < CKV_HEAD_DIM)
    return ckv_internal::set_error(CKV_E_INVALID, "bad key strides");
  if (a->edges < 0 || (a->edges > 0 && (!a->edge_src || !a->edge_dst || !a->edge_weight)))
    return ckv_internal::set_error(CKV_E_INVALID, "edges need src, dst and weight");
  if (a->edges > 0 && (!a->community_weight || !a->total_weight))
    return ckv_internal::set_error(CKV_E_INVALID, "edges need community_weight and total_weight outputs");
  if (a->topk_indices) {
    if (a->edges > 0) return ckv_internal::set_error(CKV_E_INVALID, "give either an edge list or top-k edges");
    if (!a->topk_scores || !a->community_weight || !a->total_weight)
      return ckv_internal::set_error(CKV_E_INVALID, "top-k edges need scores and the weight outputs");
    if (a->topk_kappa < 1 || a->topk_kappa > 16 || a->topk_heads <= 0 || a->topk_rows < 0 || a->topk_group <= 0 ||
        a->topk_heads > a->topk_group * a->graphs)
      return ckv_internal::set_error(CKV_E_INVALID, "bad top-k edge shape (kappa 1..16, heads <= group * graphs)");
  }
  const hipStream_t s = (hipStream_t)stream;
  const int maxc = a->max_communities;
  const int chunk_len = state_chunk(a->seq_len, a->num_sink);
  const int chunks = state_chunks(a->seq_len, a->num_sink);
  const int64_t mb = state_max_blocks(a->seq_len, a->num_sink, maxc);
  StateWorkspace w;
  state_ws_words(a->graphs, a->retrieval_heads, a->seq_len, a->num_sink, maxc, &w, a->workspace);
  // communities past lds_n are counted in global memory (64 KB of LDS per kernel)
  const int lds_n = std::min(maxc, STATE_LDS_COMMUNITIES);
  const size_t lds = (size_t)lds_n * sizeof(int);
  const bool weights = a->community_weight && a->total_weight;
  const int64_t nw = (int64_t)a->graphs * a->community_capacity;
  const int64_t fill = std::max((int64_t)a->graphs * a->token_capacity, weights ? nw : 0);
  const unsigned prep = (unsigned)(chunks * a->graphs + std::min<int64_t>((fill + 4 * HIST_THREADS - 1) / (4 * HIST_THREADS), 1024));
  hipLaunchKernelGGL(state_prep_kernel, dim3(prep), dim3(HIST_THREADS), lds, s, a->labels, a->seq_len, a->num_sink,
                     maxc, lds_n, chunk_len, chunks, a->graphs, w.hist, a->token_capacity, a->token_communities,
                     weights ? a->community_weight : nullptr, nw, a->total_weight);
  hipLaunchKernelGGL(chunk_scan_kernel, dim3((maxc + HIST_THREADS - 1) / HIST_THREADS, a->graphs), dim3(HIST_THREADS),
                     0, s, maxc, chunks, w.hist, a->member_offsets);
  hipLaunchKernelGGL(csr_scan_kernel, dim3(a->graphs), dim3(SCAN_THREADS), 0, s, maxc, mb, a->member_offsets,
                     w.blk_first, w.blk_comm);
  int label_bits = 1;
  while (label_bits < 31 && ((maxc - 1) >> label_bits) != 0) ++label_bits;
  hipLaunchKernelGGL(csr_scatter_kernel, dim3(chunks, a->graphs), dim3(64), lds, s, a->labels, a->seq_len,
                     a->num_sink, maxc, label_bits, lds_n, chunk_len, chunks, (const int32_t*)a->member_offsets, w.hist,
                     a->member_positions);
  const dim3 bgrid((unsigned)((mb + CENTROID_WAVES - 1) / CENTROID_WAVES), a->retrieval_heads);
  auto sums = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, bgrid, dim3(64 * CENTROID_WAVES), 0, s, a->keys, a->head_stride, a->token_stride,
                       a->retrieval_to_graph, a->retrieval_to_kv, (const int32_t*)a->member_offsets,
                       (const int32_t*)a->member_positions, (const int32_t*)w.blk_first,
                       (const int32_t*)w.blk_comm, mb, a->seq_len, a->num_sink, maxc, a->community_capacity,
                       w.partial, a->centroids, a->community_sizes);
  };
  if (a->key_dtype == CKV_BF16) {
    if (a->centroid_dtype == CKV_E4M3) sums(block_sum_kernel<CKV_BF16, CKV_E4M3>);
    else sums(block_sum_kernel<CKV_BF16, CKV_F32>);
  } else {
    if (a->centroid_dtype == CKV_E4M3) sums(block_sum_kernel<CKV_F32, CKV_E4M3>);
    else sums(block_sum_kernel<CKV_F32, CKV_F32>);
  }
  const dim3 cgrid((a->community_capacity + CENTROID_WAVES - 1) / CENTROID_WAVES, a->retrieval_heads);
  auto cent = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, cgrid, dim3(64 * CENTROID_WAVES), 0, s, a->retrieval_to_graph,
                       (const int32_t*)a->member_offsets, (const int32_t*)w.blk_first, (const float*)w.partial, mb,
                       maxc, a->community_capacity, a->centroids, a->community_sizes);
  };
  if (a->centroid_dtype == CKV_E4M3) cent(centroid_kernel<CKV_E4M3>); else cent(centroid_kernel<CKV_F32>);
  if (weights) {
    if (a->topk_indices && a->topk_rows > 0) {
      const int per_head = std::max(1, TOPK_WORKGROUPS / a->topk_heads);
      const int rows_per_wg = ((a->topk_rows + per_head - 1) / per_head + TOPK_THREADS - 1) / TOPK_THREADS * TOPK_THREADS;
      const dim3 tgrid((a->topk_rows + rows_per_wg - 1) / rows_per_wg, a->topk_heads);
      const bool f64 = lds_n <= TOPK_F64_COMMUNITIES;
      auto topk = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, tgrid, dim3(TOPK_THREADS), (size_t)lds_n * (f64 ? 8 : 4), s, a->labels, a->seq_len,
                           a->community_capacity, lds_n, a->topk_indices, a->topk_scores, a->topk_rows, rows_per_wg,
                           a->topk_kappa, a->topk_group, a->topk_row0, a->lam, a->community_weight, a->total_weight);
      };
      const bool aligned = (((uintptr_t)a->topk_indices | (uintptr_t)a->topk_scores) & 15) == 0;
      if (aligned && a->topk_kappa == 8) f64 ? topk(topk_weight_kernel<2, double>) : topk(topk_weight_kernel<2, float>);
      else if (aligned && a->topk_kappa == 16)
        f64 ? topk(topk_weight_kernel<4, double>) : topk(topk_weight_kernel<4, float>);
      else f64 ? topk(topk_weight_kernel<0, double>) : topk(topk_weight_kernel<0, float>);
    }
    if (a->edges > 0) {
      hipLaunchKernelGGL(edge_weight_kernel, dim3((unsigned)((a->edges + EDGES_PER_WG - 1) / EDGES_PER_WG)),
                         dim3(EDGE_THREADS), (size_t)lds_n * sizeof(float), s, a->labels, a->seq_len, a->graphs,
                         a->community_capacity, lds_n, a->edge_src, a->edge_dst, a->edge_weight, a->edges, a->community_weight, a->total_weight);
    }
  }
  return launch_check();
}

extern "C" int ckv_degree_weights(const int32_t* labels, const double* degree, const int32_t* edge_src,
                                  const float* edge_weight, int64_t edges, int32_t graphs, int32_t seq_len,
                                  int32_t community_capacity, float* community_weight, float* total_weight,
                                  void* stream) {
  if (!labels || !degree || !community_weight || !total_weight || (edges > 0 && (!edge_src || !edge_weight)))
    return ckv_internal::set_error(CKV_E_INVALID, "null degree-weight argument");
  if (graphs <= 0 || seq_len <= 0 || community_capacity <= 0 || edges < 0)
    return ckv_internal::set_error(CKV_E_INVALID, "graphs, seq_len and community_capacity must be positive");
  const hipStream_t s = (hipStream_t)stream;
  const int64_t n = (int64_t)graphs * community_capacity, v = (int64_t)graphs * seq_len;
  if (edges > 0) {
    const int early = std::min(REST_EARLY_MOST, REST_EARLY_PER_GRAPH * graphs);
    const int64_t passes = (edges + 8 * EDGE_THREADS - 1) / (8 * EDGE_THREADS);
    const int founds = (int)std::min<int64_t>(std::min<int64_t>(passes, ORDER_MOST), n);
    int* found = reinterpret_cast<int*>(community_weight);
    hipLaunchKernelGGL(edge_order_kernel, dim3(founds), dim3(EDGE_THREADS), 0, s, edge_src, edges, seq_len, v,
                       found);
    hipLaunchKernelGGL(edge_rest_kernel, dim3(graphs), dim3(64), 0, s, edge_src, edge_weight, edges, seq_len, early, 0,
                       (const int*)found, founds, total_weight);
    hipLaunchKernelGGL(edge_total_kernel, dim3((unsigned)((edges + EDGES_PER_WG - 1) / EDGES_PER_WG)),
                       dim3(EDGE_THREADS), 0, s, edge_src, edge_weight, edges, seq_len, graphs, (const int*)found,
                       founds, total_weight);
    hipLaunchKernelGGL(edge_rest_kernel, dim3(graphs), dim3(64), 0, s, edge_src, edge_weight, edges, seq_len, early, 1,
                       (const int*)found, founds, total_weight);
  }
  const int64_t clear = edges > 0 ? n : std::max<int64_t>(n, graphs);
  hipLaunchKernelGGL(weight_zero_kernel, dim3((unsigned)((clear + 255) / 256)), dim3(256), 0, s, community_weight, n,
                     edges > 0 ? nullptr : total_weight, graphs);
  hipLaunchKernelGGL(degree_weight_kernel, dim3((unsigned)((v + DEGREE_THREADS - 1) / DEGREE_THREADS)),
                     dim3(DEGREE_THREADS), 0, s, labels, degree, seq_len, graphs, community_capacity,
                     community_weight);
  return launch_check();
}
