// graph.hip - device-resident CSR for the walker, common-neighbour counts and
// per-entry acceptance thresholds.
//
// Replaces GraphEngine::load_graph (include/graph.hpp:642-824) for a single
// partition: the whole graph lives in one GPU's HBM, so the MPI edge shuffle
// and vertex-range partitioning (:542-640, :723-773) disappear.  Neighbour
// order is part of the walk result (the walker indexes adj.begin + i,
// include/walk.hpp:899), so the CSR keeps the reference order: the doubled
// edge list [e0, rev e0, e1, rev e1, ...] (:671-686), stable by source
// (build_edge_container, :509-540).
//
// HBM layout
//   d_row_ptr : uint64[V+1]  row offsets (edge_id_t)
//   d_nbr     : uint32[m]    neighbour ids, reference order
//   d_cn      : uint32[m]    common-neighbour count |N(u) & N(v) \ {u,v}|
//   d_adj     : uint4[m]     walker view {neighbour, acceptance threshold,
//                            the neighbour's row offset and degree}: what a
//                            step needs by one 16-byte read (the reference's
//                            AdjUnit<real_t>, include/graph.hpp:32-37, holds
//                            the first two)
//   d_deg     : uint32[V]    degree (= row length)
//
// Common neighbours (src/tools/gcn.cpp:250-373, the offline tool whose
// output the reference walker reads back as edge data, walk.hpp:920) are
// computed on the device over the distinct neighbours: one wavefront per
// source vertex hashes N(u) into LDS, then probes the neighbour lists of 64
// entries at a time laid end to end over the lanes; a source with more than
// kSmallDeg neighbours gets a hash table in global memory and its entries are
// shared out to many wavefronts.  On a simple undirected graph each pair is
// counted once, from its larger-degree endpoint scanning the smaller list.
//
// Acceptance threshold: the walker bounces back when tanh(pa) <= p with
// p = u / (2^31 - 1), u the 31-bit draw (walk.hpp:928-938).  pa depends only
// on (deg u, deg v, cn), so per entry the smallest u that satisfies the test
// is found once (u / M is monotone in u under correctly rounded division),
// and the walker tests `u >= threshold` - the same decision bit
// for bit, without tanh or the neighbour's degree in the step loop.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>

#include "dg_internal.h"
#include "dg_math.h"

namespace {

constexpr uint32_t kEmpty = 0xffffffffu;
constexpr int kSmallDeg = 256;           // wave path: hash of 512 slots per wave
constexpr int kSmallSlots = 512;

// Multiplicative (Fibonacci) hashing keeps the high bits of the product:
// the low bits depend only on the low bits of w, and vertex ids of generated
// graphs (R-MAT in particular) are far from uniform in their low bits.
__device__ __forceinline__ uint32_t slot_hash(uint32_t w, uint32_t mask) {
  return (w * 2654435761u) >> __builtin_clz(mask);  // mask = 2^k - 1, k >= 6
}

// Returns true if w was in the table already.
__device__ __forceinline__ bool hash_insert(uint32_t* tbl, uint32_t mask, uint32_t w) {
  uint32_t s = slot_hash(w, mask);
  while (true) {
    uint32_t prev = atomicCAS(&tbl[s], kEmpty, w);
    if (prev == kEmpty) return false;
    if (prev == w) return true;
    s = (s + 1) & mask;
  }
}

__device__ __forceinline__ bool hash_find(const uint32_t* tbl, uint32_t mask, uint32_t w) {
  uint32_t s = slot_hash(w, mask);
  while (true) {
    uint32_t x = tbl[s];
    if (x == w) return true;
    if (x == kEmpty) return false;
    s = (s + 1) & mask;
  }
}

// A pair's count is |N(u) & N(v) \ {u, v}| over the distinct neighbours.
// With SYM (simple undirected graph, rev[k] = position of the reverse entry
// of k) each pair is counted once, from its larger-degree endpoint (ties by
// id): the smaller list is scanned against the hash of the larger one and
// the count written to both entries.  Cost: the sum over edges of
// min(deg u, deg v) instead of the sum of squared degrees.
// Counts of up to 64 entries [k0, k1) of row u against the hash of N(u).
// The neighbour lists to scan are laid end to end: lane j takes entry k0 + j's
// list, a prefix sum over the lanes gives each list's first element, and the
// 64 lanes then take kFlat elements each per pass (the list of an element by
// binary search over the sums), so that the loads of a whole pass are in
// flight together.  Bound by the latency of three dependent loads per pass.
// One list at a time instead (those loads per entry, most lanes idle on the
// short lists of a power-law graph): 6.2 ms against 1.1 ms (small rows and hubs
// 0.55 each) at 131,072 vertices and 2.7M entries.
constexpr int kFlat = 4;

struct CnLists {
  uint64_t beg[64];
  uint64_t off[64];
  uint32_t v[64];
  uint32_t cnt[64];
};

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <bool SYM>
__device__ __forceinline__ void cn_entries(const uint64_t* rp, const uint32_t* nbr, uint32_t u, uint32_t du,
                                           uint64_t k0, uint64_t k1, const uint32_t* tbl, uint32_t mask,
                                           CnLists& L, const uint64_t* rev, uint32_t* cn) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t k = k0 + lane;
  bool mine = k < k1;
  uint32_t v = 0, len = 0;
  uint64_t vb = 0;
  if (mine) {
    v = nbr[k];
    vb = rp[v];
    len = (uint32_t)(rp[v + 1] - vb);
    // the other endpoint counts this pair
    if (SYM && v != u && (len > du || (len == du && v > u))) mine = false;
    if (!mine) len = 0;
  }
  uint64_t inc = len;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint64_t o = __shfl_up(inc, d, 64);
    if ((int)lane >= d) inc += o;
  }
  L.beg[lane] = vb;
  L.off[lane] = inc - len;
  L.v[lane] = v;
  L.cnt[lane] = 0;
  const uint64_t total = __shfl(inc, 63, 64);
  wave_lds_sync();
  for (uint64_t t0 = 0; t0 < total; t0 += 64 * kFlat) {
    uint32_t w[kFlat], j[kFlat];
#pragma unroll
    for (int r = 0; r < kFlat; ++r) {
      const uint64_t e = t0 + 64 * r + lane;
      // the last list that starts at or before e (an empty list starts where
      // the next one does, and is not the last)
      uint32_t lo = 0;
#pragma unroll
      for (int h = 32; h >= 1; h >>= 1)
        if (L.off[lo + h] <= e) lo += h;
      j[r] = lo;
      w[r] = e < total ? nbr[L.beg[lo] + (e - L.off[lo])] : u;
    }
#pragma unroll
    for (int r = 0; r < kFlat; ++r)
      if (w[r] != u && w[r] != L.v[j[r]] && hash_find(tbl, mask, w[r])) atomicAdd(&L.cnt[j[r]], 1u);
  }
  wave_lds_sync();
  if (mine) {
    const uint32_t c = L.cnt[lane];
    cn[k] = c;
    if (SYM && v != u) cn[rev[k]] = c;
  }
  wave_lds_sync();
}

// One wavefront per source vertex with degree <= kSmallDeg.  *not_simple is
// set when a row lists a neighbour twice or its own vertex.
template <bool SYM>
__global__ __launch_bounds__(256) void cn_small_kernel(const uint64_t* rp, const uint32_t* nbr,
                                                       uint32_t v_num, const uint64_t* rev,
                                                       uint32_t* cn, uint32_t* not_simple) {
  __shared__ uint32_t s_tbl[4][kSmallSlots];
  __shared__ CnLists s_lists[4];
  const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t* tbl = s_tbl[wave];
  const uint64_t waves = (uint64_t)gridDim.x * 4;
  bool odd = false;
  for (uint64_t u0 = (uint64_t)blockIdx.x * 4 + wave; u0 < v_num; u0 += waves) {
    const uint32_t u = (uint32_t)u0;
    const uint64_t b = rp[u], e = rp[u + 1];
    const uint64_t d = e - b;
    if (d > (uint64_t)kSmallDeg || d == 0) continue;  // wave-uniform
    const uint32_t du = (uint32_t)d;
    uint32_t slots = 64;
    while (slots < 2 * du) slots <<= 1;
    const uint32_t mask = slots - 1;
    for (uint32_t i = lane; i < slots; i += 64) tbl[i] = kEmpty;
    wave_lds_sync();
    for (uint32_t i = lane; i < du; i += 64) {
      const uint32_t w = nbr[b + i];
      if (w == u || hash_insert(tbl, mask, w)) odd = true;
    }
    wave_lds_sync();
    for (uint64_t k = b; k < e; k += 64)
      cn_entries<SYM>(rp, nbr, u, du, k, k + 64 < e ? k + 64 : e, tbl, mask, s_lists[wave], rev, cn);
  }
  if (not_simple && __ballot(odd) != 0 && lane == 0) atomicOr(not_simple, 1u);
}

// Sources with degree > kSmallDeg (hubs): N(u) goes into a hash table of its
// own in global memory (hub_hash_kernel, one workgroup per hub), and the
// hub's entries are cut into items of kHubItem consecutive entries, one
// wavefront per item, so a hub's work spreads over many wavefronts.
constexpr uint32_t kHubItem = 64;

__global__ __launch_bounds__(256) void hub_hash_kernel(const uint64_t* rp, const uint32_t* nbr,
                                                       const uint32_t* big, uint32_t n_big,
                                                       const uint64_t* toff, const uint32_t* tsize,
                                                       uint32_t* tab, uint32_t* not_simple) {
  bool odd = false;
  for (uint32_t bi = blockIdx.x; bi < n_big; bi += gridDim.x) {
    const uint32_t u = big[bi];
    uint32_t* t = tab + toff[bi];
    const uint32_t mask = tsize[bi] - 1;
    for (uint64_t i = rp[u] + threadIdx.x; i < rp[u + 1]; i += 256) {
      const uint32_t w = nbr[i];
      if (w == u || hash_insert(t, mask, w)) odd = true;
    }
  }
  if (not_simple && __ballot(odd) != 0 && (threadIdx.x & 63u) == 0) atomicOr(not_simple, 1u);
}

template <bool SYM>
__global__ __launch_bounds__(256) void hub_cn_kernel(const uint64_t* rp, const uint32_t* nbr,
                                                     const uint32_t* big, const uint64_t* toff,
                                                     const uint32_t* tsize, const uint32_t* tab,
                                                     const uint32_t* it_hub, const uint64_t* it_k0,
                                                     uint64_t n_items, const uint64_t* rev, uint32_t* cn) {
  __shared__ CnLists s_lists[4];
  const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint64_t nwaves = (uint64_t)gridDim.x * 4;
  for (uint64_t it = (uint64_t)blockIdx.x * 4 + wv; it < n_items; it += nwaves) {
    const uint32_t bi = it_hub[it];
    const uint32_t u = big[bi];
    const uint64_t e = rp[u + 1];
    const uint64_t k0 = it_k0[it];
    cn_entries<SYM>(rp, nbr, u, (uint32_t)(e - rp[u]), k0, k0 + kHubItem < e ? k0 + kHubItem : e,
                    tab + toff[bi], tsize[bi] - 1, s_lists[wv], rev, cn);
  }
}

__global__ void fill_kernel(uint32_t* p, uint64_t n, uint32_t v) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

__global__ void degree_kernel(const uint64_t* rp, uint32_t v_num, uint32_t* deg) {
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < v_num; v += gridDim.x * blockDim.x)
    deg[v] = (uint32_t)(rp[v + 1] - rp[v]);
}

// Smallest u in [0, 2^31 - 1] with tanh(pa) <= u / (2^31 - 1), pa as in
// walk.hpp:933 (times the edge weight w on a weighted graph: tanh(pa * w));
// 2^31 (never reached by a 31-bit draw) if no u qualifies.
__device__ __forceinline__ uint32_t bounce_threshold(int sd, int dd, int cnv, const float* w,
                                                     uint64_t e) {
  const double M = 2147483647.0;
  const double pa = (1.0 / (double)(sd - cnv)) * (double)(sd > dd ? sd : dd) /
                    (double)(sd < dd ? sd : dd);
  const double pn = dg_tanh(w ? pa * (double)w[e] : pa);
  if (pn != pn) return 0x80000000u;
  if (!(pn <= 1.0)) return 0x80000000u;
  // u / M rounds to within 2^-53 of itself, far less than the 1 / M between
  // two candidates, so the smallest u lies within two of pn * M
  const double g = pn * M;
  uint32_t u = g > 2.0 ? (uint32_t)g - 2u : 0u;
  while (u < 2147483647u && !(pn <= (double)u / M)) ++u;
  return u;
}

// src: the source vertex of every entry, or null (found by binary search).
__global__ void threshold_kernel(const uint64_t* rp, const uint32_t* src, const uint32_t* nbr, const uint32_t* cn,
                                 const float* w, const uint32_t* deg, uint32_t v_num, uint64_t m,
                                 uint4* adj) {
  for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < m;
       e += (uint64_t)gridDim.x * blockDim.x) {
    uint32_t u;
    if (src) {
      u = src[e];
    } else {  // last u with rp[u] <= e
      uint32_t lo = 0, hi = v_num - 1;
      while (lo < hi) {
        const uint32_t mid = lo + (hi - lo + 1) / 2;
        if (rp[mid] <= e)
          lo = mid;
        else
          hi = mid - 1;
      }
      u = lo;
    }
    const uint32_t v = nbr[e];
    const uint64_t vb = rp[v];
    const uint32_t dv = deg[v];
    const uint2 row = dg_pack_row(vb, dv, dv == 2 && nbr[vb] == v);
    adj[e] = make_uint4(v, bounce_threshold((int)deg[u], (int)dv, (int)cn[e], w, e), row.x, row.y);
  }
}

__global__ void take_thresholds_kernel(const uint4* adj, uint64_t m, uint32_t* thr) {
  for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < m;
       e += (uint64_t)gridDim.x * blockDim.x)
    thr[e] = adj[e].y;
}

// ---- CSR on the device ---------------------------------------------------------
// Bound by the copy of the edges and three radix passes (0.05 ms each at 2.7M
// entries); counting and placing on the host took 45 ms of a 53 ms build at
// 131,072 vertices, this one 0.4 ms of 6.8 ms (the copies in and out and the
// allocations are the rest).  The doubled edge list sorted stably by source: LSD radix passes over
// (source, entry) pairs, each pass a histogram per tile, one scan over
// (digit, tile) and the scatter.  The entry (2 i for edge i, 2 i + 1 for its
// reverse) says where the neighbour, the data and the reverse entry come from.

// Index of the first edge with an endpoint out of range (by atomicMin).
__global__ void edge_check_kernel(const dg_edge* edges, uint64_t n, uint32_t v_num, unsigned long long* bad) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    if (edges[i].src >= v_num || edges[i].dst >= v_num) atomicMin(bad, (unsigned long long)i);
}

__global__ void set_u64_kernel(unsigned long long* p, unsigned long long v) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *p = v;
}

__global__ void entry_keys_kernel(const dg_edge* edges, uint64_t n, int undirected, uint32_t* keys,
                                  uint32_t* ids) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const dg_edge e = edges[i];
    if (undirected) {
      reinterpret_cast<uint2*>(keys)[i] = make_uint2(e.src, e.dst);
      reinterpret_cast<uint2*>(ids)[i] = make_uint2(2u * (uint32_t)i, 2u * (uint32_t)i + 1u);
    } else {
      keys[i] = e.src;
      ids[i] = (uint32_t)i;
    }
  }
}

constexpr int kSortThreads = 512;
constexpr int kSortWaves = kSortThreads / 64;
constexpr int kSortIpt = 8;
constexpr int kSortTile = kSortThreads * kSortIpt;  // 4,096 keys
constexpr int kDigits = 256;

// hist[digit * n_tiles + tile]
__global__ __launch_bounds__(kSortThreads) void sort_hist_kernel(const uint32_t* keys, uint64_t n, int shift,
                                                                 uint32_t n_tiles, uint32_t* hist) {
  __shared__ uint32_t h[kDigits];
  for (int d = threadIdx.x; d < kDigits; d += kSortThreads) h[d] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * kSortTile;
#pragma unroll
  for (int i = 0; i < kSortIpt; ++i) {
    const uint64_t k = base + (uint64_t)i * kSortThreads + threadIdx.x;
    if (k < n) atomicAdd(&h[(keys[k] >> shift) & (kDigits - 1)], 1u);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < kDigits; d += kSortThreads) hist[(uint64_t)d * n_tiles + blockIdx.x] = h[d];
}

// base[digit * n_tiles + tile]: where the tile's keys of that digit go.
// Wavefront w ranks keys [w * 512, (w + 1) * 512) of the tile, 64 at a time in
// order; lanes of one digit are ranked by a ballot match.
__global__ __launch_bounds__(kSortThreads) void sort_scatter_kernel(const uint32_t* keys, const uint32_t* ids,
                                                                    uint64_t n, int shift, uint32_t n_tiles,
                                                                    const uint64_t* base, uint32_t* okeys,
                                                                    uint32_t* oids) {
  __shared__ uint32_t cnt[kSortWaves][kDigits];
  __shared__ uint64_t gbase[kDigits];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < kSortWaves * kDigits; i += kSortThreads) (&cnt[0][0])[i] = 0;
  for (int d = threadIdx.x; d < kDigits; d += kSortThreads) gbase[d] = base[(uint64_t)d * n_tiles + blockIdx.x];
  __syncthreads();
  const uint64_t first = (uint64_t)blockIdx.x * kSortTile + wave * 64 * kSortIpt;
  const uint64_t below = (1ull << lane) - 1ull;
  uint32_t kk[kSortIpt], vv[kSortIpt], pos[kSortIpt];
#pragma unroll
  for (int i = 0; i < kSortIpt; ++i) {
    const uint64_t k = first + i * 64 + lane;
    kk[i] = k < n ? keys[k] : 0u;
    vv[i] = k < n ? ids[k] : 0u;
  }
#pragma unroll
  for (int i = 0; i < kSortIpt; ++i) {
    const bool valid = first + i * 64 + lane < n;
    const uint32_t dig = (kk[i] >> shift) & (kDigits - 1);
    uint64_t same = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const uint64_t bal = __ballot(((dig >> b) & 1u) != 0u);
      same &= ((dig >> b) & 1u) ? bal : ~bal;
    }
    const uint32_t before = cnt[wave][dig];
    const uint32_t rank = (uint32_t)__popcll(same & below);
    wave_lds_sync();
    if (valid && rank == 0) cnt[wave][dig] = before + (uint32_t)__popcll(same);
    wave_lds_sync();
    pos[i] = before + rank;
  }
  __syncthreads();
  for (int d = threadIdx.x; d < kDigits; d += kSortThreads) {
    uint32_t run = 0;
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) {
      const uint32_t c = cnt[w][d];
      cnt[w][d] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kSortIpt; ++i) {
    if (first + i * 64 + lane < n) {
      const uint32_t dig = (kk[i] >> shift) & (kDigits - 1);
      const uint64_t dst = gbase[dig] + cnt[wave][dig] + pos[i];
      okeys[dst] = kk[i];
      oids[dst] = vv[i];
    }
  }
}

// rp[v] = first sorted position whose source is v or above.
__global__ void row_ptr_kernel(const uint32_t* src, uint64_t m, uint32_t v_num, uint64_t* rp) {
  for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v <= v_num;
       v += (uint64_t)gridDim.x * blockDim.x) {
    uint64_t lo = 0, hi = m;
    while (lo < hi) {
      const uint64_t mid = (lo + hi) / 2;
      if (src[mid] < v)
        lo = mid + 1;
      else
        hi = mid;
    }
    rp[v] = lo;
  }
}

// The edge data as the walker's integer (walk.hpp:920), converted as the
// host's float-to-int conversion does out of range.
__device__ __forceinline__ uint32_t data_to_cn(float d) {
  return d >= -2147483648.0f && d < 2147483648.0f ? (uint32_t)(int)d : 0x80000000u;
}

__global__ void entry_gather_kernel(const dg_edge* edges, const uint32_t* ids, uint64_t m, int undirected,
                                    uint32_t* nbr, uint32_t* cn, float* w, uint32_t* where) {
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < m;
       p += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t id = ids[p];
    const dg_edge e = edges[undirected ? id >> 1 : id];
    nbr[p] = (undirected && (id & 1u)) ? e.src : e.dst;
    if (cn) cn[p] = data_to_cn(e.data);
    if (w) w[p] = e.data;
    if (where) where[id] = (uint32_t)p;
  }
}

// rev[p] = position of p's reverse entry.
__global__ void reverse_kernel(const uint32_t* ids, const uint32_t* where, uint64_t m, uint64_t* rev) {
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < m;
       p += (uint64_t)gridDim.x * blockDim.x)
    rev[p] = where[ids[p] ^ 1u];
}

// ---- the hot set and the hubs ---------------------------------------------------
// hist[d] = vertices of degree d, the last bin those of kDegBins - 1 or more.
constexpr uint32_t kDegBins = 8192;

__global__ __launch_bounds__(256) void degree_hist_kernel(const uint32_t* deg, uint32_t v_num, uint32_t* hist) {
  __shared__ uint32_t h[kDegBins];
  for (uint32_t i = threadIdx.x; i < kDegBins; i += 256) h[i] = 0;
  __syncthreads();
  for (uint64_t v = (uint64_t)blockIdx.x * 256 + threadIdx.x; v < v_num; v += (uint64_t)gridDim.x * 256)
    atomicAdd(&h[deg[v] < kDegBins ? deg[v] : kDegBins - 1], 1u);
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < kDegBins; i += 256)
    if (h[i]) atomicAdd(&hist[i], h[i]);
}

// The lowest degree whose vertices, with those above it, fit n_hot slots
// (cut[0]; kDegBins if even the last bin does not), and zeroed slot counters
// (cut[1]: those above the cut, cut[2]: those just below it).
__global__ __launch_bounds__(256) void hot_cut_kernel(const uint32_t* hist, uint32_t n_hot, uint32_t* cut) {
  __shared__ uint32_t part[256];
  constexpr uint32_t per = kDegBins / 256;
  const uint32_t hi = kDegBins - threadIdx.x * per;  // thread t: bins [hi - per, hi)
  uint32_t s = 0;
  for (uint32_t i = 0; i < per; ++i) s += hist[hi - 1 - i];
  part[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x != 0) return;
  uint32_t run = 0, t = 0;
  while (t < 256 && run + part[t] <= n_hot) run += part[t++];
  uint32_t c = kDegBins - t * per;
  while (c > 0 && run + hist[c - 1] <= n_hot) run += hist[--c];
  cut[0] = c;
  cut[1] = 0;
  cut[2] = run;
}

// Slots of the highest-degree vertices: every vertex at or above the cut,
// then vertices of the next lower bin while slots are left (walks visit
// vertices in proportion to degree; which vertex has which slot, and which of
// that bin have one, does not change any count).  Without a cut every vertex
// has one.
__global__ void hot_slots_kernel(const uint32_t* deg, uint32_t v_num, uint32_t n_hot, uint32_t* cut,
                                 uint16_t* slot, uint32_t* hot_id) {
  const uint32_t c = cut ? cut[0] : 0u;
  for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < v_num;
       v += (uint64_t)gridDim.x * blockDim.x) {
    if (!cut) {
      slot[v] = (uint16_t)v;
      hot_id[v] = (uint32_t)v;
      continue;
    }
    const uint32_t d = deg[v] < kDegBins ? deg[v] : kDegBins - 1;
    uint32_t k = kNotHot;
    if (d >= c) {
      k = atomicAdd(&cut[1], 1u);
    } else if (d + 1 == c && __hip_atomic_load(&cut[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < n_hot) {
      k = atomicAdd(&cut[2], 1u);
      if (k >= n_hot) k = kNotHot;
    }
    slot[v] = (uint16_t)k;
    if (k != kNotHot) hot_id[k] = (uint32_t)v;
  }
}

// Vertices of degree above kSmallDeg, in no order: count, then {id, degree,
// row} of the first `cap`.
struct HubRec {
  uint32_t v, deg;
  uint64_t row;
};

__global__ void hub_list_kernel(const uint64_t* rp, uint32_t v_num, uint32_t* count, uint32_t cap, HubRec* out) {
  for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < v_num;
       v += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t b = rp[v], d = rp[v + 1] - b;
    if (d <= (uint64_t)kSmallDeg) continue;
    const uint32_t i = atomicAdd(count, 1u);
    if (i < cap) out[i] = HubRec{(uint32_t)v, (uint32_t)d, b};
  }
}

int grid_for(dg_ctx* ctx, uint64_t n, int block) {
  uint64_t g = (n + block - 1) / block;
  uint64_t cap = (uint64_t)ctx->num_cus * 32;
  if (g > cap) g = cap;
  return g == 0 ? 1 : (int)g;
}

}  // namespace

void dg_graph_free(dg_ctx* ctx) {
  void* bufs[] = {ctx->d_row_ptr, ctx->d_nbr, ctx->d_cn, ctx->d_adj, ctx->d_deg, ctx->d_hot_slot,
                  ctx->d_hot_id};
  for (void* p : bufs)
    if (p) hipFree(p);
  ctx->d_hot_slot = nullptr;
  ctx->d_hot_id = nullptr;
  ctx->n_hot = 0;
  ctx->d_row_ptr = nullptr;
  ctx->d_nbr = nullptr;
  ctx->d_cn = nullptr;
  ctx->d_adj = nullptr;
  ctx->d_deg = nullptr;
  ctx->v_num = 0;
  ctx->m = 0;
}

// Rows in parallel on the host: lo .. hi of [0, n) per thread.
template <typename F>
static void host_rows(uint32_t n, F f) {
  unsigned t = std::thread::hardware_concurrency();
  t = t == 0 ? 1 : (t > 16 ? 16 : t);
  if (n < 4096) t = 1;
  std::vector<std::thread> th;
  for (unsigned i = 0; i < t; ++i) {
    const uint32_t lo = (uint32_t)((uint64_t)n * i / t), hi = (uint32_t)((uint64_t)n * (i + 1) / t);
    th.emplace_back([=] { f(lo, hi); });
  }
  for (auto& x : th) x.join();
}

namespace {

// An allocation: without room the call ends with DG_ERR_NOMEM (and the
// allocation's error is not the next launch's).
#define DG_ROOM(ctx, expr)                                                              \
  do {                                                                                  \
    hipError_t _e = (expr);                                                             \
    if (_e != hipSuccess) {                                                             \
      (void)hipGetLastError();                                                          \
      return dg_fail((ctx), _e == hipErrorOutOfMemory ? DG_ERR_NOMEM : DG_ERR_HIP,      \
                     "%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e), __FILE__, __LINE__); \
    }                                                                                   \
  } while (0)

// Device memory of one call, freed with it.
struct Scratch {
  std::vector<void*> bufs;
  ~Scratch() {
    for (void* b : bufs) hipFree(b);
  }
  template <typename T>
  hipError_t get(T** p, uint64_t n) {
    const hipError_t e = hipMalloc((void**)p, sizeof(T) * (n ? n : 1));
    if (e == hipSuccess) bufs.push_back(*p);
    return e;
  }
};

}  // namespace

// Counts of every entry of the CSR (d_rp, d_nbr) into d_cn, on the stream;
// with d_rev (position of every entry's reverse) each pair is counted once.
// *d_not_simple (zeroed here, may be null) is set for a row that repeats a
// neighbour or lists its own vertex.  Buffers come from `mem`.
static int enqueue_cn(dg_ctx* ctx, Scratch& mem, uint32_t v_num, uint64_t m, const uint64_t* d_rp,
                      const uint32_t* d_nbr, const uint64_t* d_rev, uint32_t* d_cn, uint32_t* d_not_simple) {
  // hubs: listed on the device, hash-table offsets and work items laid out here
  const uint64_t cap = std::min<uint64_t>(v_num, m / (kSmallDeg + 1));
  std::vector<HubRec> hubs;
  if (cap) {
    uint32_t* d_count = nullptr;
    HubRec* d_hubs = nullptr;
    DG_ROOM(ctx, mem.get(&d_count, 2));
    DG_ROOM(ctx, mem.get(&d_hubs, cap));
    fill_kernel<<<1, 64, 0, ctx->stream>>>(d_count, 1, 0u);
    hub_list_kernel<<<grid_for(ctx, v_num, 256), 256, 0, ctx->stream>>>(d_rp, v_num, d_count, (uint32_t)cap,
                                                                       d_hubs);
    uint32_t n = 0;
    DG_HIP(ctx, hipMemcpyAsync(&n, d_count, sizeof(n), hipMemcpyDeviceToHost, ctx->stream));
    DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    hubs.resize(n);
    if (n) DG_HIP(ctx, hipMemcpy(hubs.data(), d_hubs, sizeof(HubRec) * n, hipMemcpyDeviceToHost));
  }
  std::vector<uint32_t> big, tsize, it_hub;
  std::vector<uint64_t> toff, it_k0;
  uint64_t tslots = 0;
  for (const HubRec& h : hubs) {
    uint64_t sz = 64;
    while (sz < 2 * (uint64_t)h.deg) sz <<= 1;
    const uint32_t bi = (uint32_t)big.size();
    big.push_back(h.v);
    tsize.push_back((uint32_t)sz);
    toff.push_back(tslots);
    tslots += sz;
    for (uint64_t k0 = h.row; k0 < h.row + h.deg; k0 += kHubItem) {
      it_hub.push_back(bi);
      it_k0.push_back(k0);
    }
  }
  uint32_t *d_big = nullptr, *d_tsize = nullptr, *d_tab = nullptr, *d_it_hub = nullptr;
  uint64_t *d_toff = nullptr, *d_it_k0 = nullptr;
  if (!big.empty()) {
    DG_ROOM(ctx, mem.get(&d_big, big.size()));
    DG_ROOM(ctx, mem.get(&d_tsize, big.size()));
    DG_ROOM(ctx, mem.get(&d_toff, big.size()));
    DG_ROOM(ctx, mem.get(&d_tab, tslots));
    DG_ROOM(ctx, mem.get(&d_it_hub, it_hub.size()));
    DG_ROOM(ctx, mem.get(&d_it_k0, it_k0.size()));
    DG_HIP(ctx, hipMemcpy(d_big, big.data(), sizeof(uint32_t) * big.size(), hipMemcpyHostToDevice));
    DG_HIP(ctx, hipMemcpy(d_tsize, tsize.data(), sizeof(uint32_t) * big.size(), hipMemcpyHostToDevice));
    DG_HIP(ctx, hipMemcpy(d_toff, toff.data(), sizeof(uint64_t) * big.size(), hipMemcpyHostToDevice));
    DG_HIP(ctx, hipMemcpy(d_it_hub, it_hub.data(), sizeof(uint32_t) * it_hub.size(), hipMemcpyHostToDevice));
    DG_HIP(ctx, hipMemcpy(d_it_k0, it_k0.data(), sizeof(uint64_t) * it_k0.size(), hipMemcpyHostToDevice));
  }
  size_t tc;
  DG_CHECK(dg_time_begin(ctx, "cn", &tc));
  if (d_not_simple) fill_kernel<<<1, 64, 0, ctx->stream>>>(d_not_simple, 1, 0u);
  const unsigned gs = (unsigned)grid_for(ctx, (uint64_t)v_num, 4);
  if (!big.empty()) {
    fill_kernel<<<grid_for(ctx, tslots, 256), 256, 0, ctx->stream>>>(d_tab, tslots, kEmpty);
    hub_hash_kernel<<<(unsigned)std::min<size_t>(big.size(), (size_t)ctx->num_cus * 8), 256, 0, ctx->stream>>>(
        d_rp, d_nbr, d_big, (uint32_t)big.size(), d_toff, d_tsize, d_tab, d_not_simple);
  }
  const unsigned gh = (unsigned)grid_for(ctx, (uint64_t)it_hub.size() * 64, 256);
  if (d_rev) {
    cn_small_kernel<true><<<gs, 256, 0, ctx->stream>>>(d_rp, d_nbr, v_num, d_rev, d_cn, d_not_simple);
    if (!big.empty())
      hub_cn_kernel<true><<<gh, 256, 0, ctx->stream>>>(d_rp, d_nbr, d_big, d_toff, d_tsize, d_tab, d_it_hub,
                                                       d_it_k0, it_hub.size(), d_rev, d_cn);
  } else {
    cn_small_kernel<false><<<gs, 256, 0, ctx->stream>>>(d_rp, d_nbr, v_num, nullptr, d_cn, d_not_simple);
    if (!big.empty())
      hub_cn_kernel<false><<<gh, 256, 0, ctx->stream>>>(d_rp, d_nbr, d_big, d_toff, d_tsize, d_tab, d_it_hub,
                                                        d_it_k0, it_hub.size(), nullptr, d_cn);
  }
  DG_HIP(ctx, hipGetLastError());
  DG_CHECK(dg_time_end(ctx, tc));
  return DG_OK;
}

// Counts of a graph with repeated edges or self-loops: taken on the distinct
// neighbour lists (sorted, without the vertex itself), each entry taking the
// count of its pair - the set semantics of gcn.cpp:329-346.
static int cn_of_multigraph(dg_ctx* ctx, uint32_t v_num, uint64_t m) {
  std::vector<uint64_t> rp(v_num + 1ull);
  std::vector<uint32_t> nbr(m);
  DG_HIP(ctx, hipMemcpy(rp.data(), ctx->d_row_ptr, sizeof(uint64_t) * (v_num + 1ull), hipMemcpyDeviceToHost));
  if (m) DG_HIP(ctx, hipMemcpy(nbr.data(), ctx->d_nbr, sizeof(uint32_t) * m, hipMemcpyDeviceToHost));
  std::vector<uint64_t> srp(v_num + 1ull, 0);
  std::vector<uint32_t> snbr;
  {
    std::vector<std::vector<uint32_t>> rows(v_num);
    host_rows(v_num, [&](uint32_t lo, uint32_t hi) {
      for (uint32_t u = lo; u < hi; ++u) {
        std::vector<uint32_t>& r = rows[u];
        r.assign(nbr.begin() + rp[u], nbr.begin() + rp[u + 1]);
        std::sort(r.begin(), r.end());
        r.erase(std::unique(r.begin(), r.end()), r.end());
        r.erase(std::remove(r.begin(), r.end(), u), r.end());
      }
    });
    for (uint32_t u = 0; u < v_num; ++u) srp[u + 1] = srp[u] + rows[u].size();
    snbr.resize(srp[v_num]);
    for (uint32_t u = 0; u < v_num; ++u) std::copy(rows[u].begin(), rows[u].end(), snbr.begin() + srp[u]);
  }
  const uint64_t cm = srp[v_num];
  std::vector<uint32_t> scn(cm), cn(m);
  {
    Scratch mem;
    uint64_t* d_rp = nullptr;
    uint32_t *d_nbr = nullptr, *d_cn = nullptr;
    DG_ROOM(ctx, mem.get(&d_rp, v_num + 1ull));
    DG_ROOM(ctx, mem.get(&d_nbr, cm));
    DG_ROOM(ctx, mem.get(&d_cn, cm));
    DG_HIP(ctx, hipMemcpy(d_rp, srp.data(), sizeof(uint64_t) * (v_num + 1ull), hipMemcpyHostToDevice));
    if (cm) DG_HIP(ctx, hipMemcpy(d_nbr, snbr.data(), sizeof(uint32_t) * cm, hipMemcpyHostToDevice));
    DG_CHECK(enqueue_cn(ctx, mem, v_num, cm, d_rp, d_nbr, nullptr, d_cn, nullptr));
    DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (cm) DG_HIP(ctx, hipMemcpy(scn.data(), d_cn, sizeof(uint32_t) * cm, hipMemcpyDeviceToHost));
  }
  host_rows(v_num, [&](uint32_t lo, uint32_t hi) {
    for (uint32_t u = lo; u < hi; ++u) {
      const uint32_t* row = snbr.data() + srp[u];
      const uint64_t len = srp[u + 1] - srp[u];
      for (uint64_t k = rp[u]; k < rp[u + 1]; ++k) {
        const uint32_t v = nbr[k];
        if (v == u) {  // |N(u) \ {u}|
          cn[k] = (uint32_t)len;
          continue;
        }
        const uint32_t* it = std::lower_bound(row, row + len, v);
        cn[k] = scn[srp[u] + (uint64_t)(it - row)];
      }
    }
  });
  if (m) DG_HIP(ctx, hipMemcpy(ctx->d_cn, cn.data(), sizeof(uint32_t) * m, hipMemcpyHostToDevice));
  return DG_OK;
}

// The rest of the graph from ctx's row pointers and neighbours (and, from the
// edge data, counts): degrees, the hot set, the counts, the thresholds.
// d_w: weights or null; d_rev: reverse positions or null; d_src: every
// entry's source or null.
static int finish_graph(dg_ctx* ctx, const float* d_w, const uint64_t* d_rev, const uint32_t* d_src, int cn_mode) {
  const uint32_t v_num = ctx->v_num;
  const uint64_t m = ctx->m;
  Scratch mem;
  degree_kernel<<<grid_for(ctx, v_num, 256), 256, 0, ctx->stream>>>(ctx->d_row_ptr, v_num, ctx->d_deg);
  {
    // hot set for visit counting: walks visit vertices in proportion to degree
    const uint32_t n_hot = v_num < kHotMax ? v_num : kHotMax;
    uint32_t* d_cut = nullptr;
    if (v_num > kHotMax) {
      uint32_t* d_hist = nullptr;
      DG_ROOM(ctx, mem.get(&d_hist, kDegBins + 4));
      d_cut = d_hist + kDegBins;
      fill_kernel<<<grid_for(ctx, kDegBins + 4, 256), 256, 0, ctx->stream>>>(d_hist, kDegBins + 4, 0u);
      const unsigned gd = (unsigned)std::min<uint64_t>((uint64_t)ctx->num_cus, ((uint64_t)v_num + 255) / 256);
      degree_hist_kernel<<<gd, 256, 0, ctx->stream>>>(ctx->d_deg, v_num, d_hist);
      hot_cut_kernel<<<1, 256, 0, ctx->stream>>>(d_hist, n_hot, d_cut);
    }
    hot_slots_kernel<<<grid_for(ctx, v_num, 256), 256, 0, ctx->stream>>>(ctx->d_deg, v_num, n_hot, d_cut,
                                                                        ctx->d_hot_slot, ctx->d_hot_id);
    ctx->n_hot = n_hot;
  }
  DG_HIP(ctx, hipGetLastError());
  if (cn_mode == DG_CN_COMPUTE || cn_mode == DG_CN_COMPUTE_WEIGHTED) {
    uint32_t* d_flag = nullptr;
    DG_ROOM(ctx, mem.get(&d_flag, 1));
    DG_CHECK(enqueue_cn(ctx, mem, v_num, m, ctx->d_row_ptr, ctx->d_nbr, d_rev, ctx->d_cn, d_flag));
    uint32_t not_simple = 0;
    DG_HIP(ctx, hipMemcpyAsync(&not_simple, d_flag, sizeof(not_simple), hipMemcpyDeviceToHost, ctx->stream));
    DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (not_simple) DG_CHECK(cn_of_multigraph(ctx, v_num, m));
  }
  size_t tt;
  DG_CHECK(dg_time_begin(ctx, "threshold", &tt));
  if (m)
    threshold_kernel<<<grid_for(ctx, m, 256), 256, 0, ctx->stream>>>(
        ctx->d_row_ptr, d_src, ctx->d_nbr, ctx->d_cn, d_w, ctx->d_deg, v_num, m, ctx->d_adj);
  DG_HIP(ctx, hipGetLastError());
  DG_CHECK(dg_time_end(ctx, tt));
  DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return DG_OK;
}

// The graph's own arrays (the previous graph and its walker state are given up).
static int alloc_graph(dg_ctx* ctx, uint32_t v_num, uint64_t m) {
  dg_walk_free(ctx);  // walker state belongs to the previous graph
  dg_graph_free(ctx);
  const uint64_t n = m ? m : 1;
  DG_ROOM(ctx, hipMalloc((void**)&ctx->d_row_ptr, sizeof(uint64_t) * (v_num + 1ull)));
  DG_ROOM(ctx, hipMalloc((void**)&ctx->d_nbr, sizeof(uint32_t) * n));
  DG_ROOM(ctx, hipMalloc((void**)&ctx->d_cn, sizeof(uint32_t) * n));
  DG_ROOM(ctx, hipMalloc((void**)&ctx->d_adj, sizeof(uint4) * n));
  DG_ROOM(ctx, hipMalloc((void**)&ctx->d_deg, sizeof(uint32_t) * v_num));
  DG_ROOM(ctx, hipMalloc((void**)&ctx->d_hot_slot, sizeof(uint16_t) * v_num));
  DG_ROOM(ctx, hipMalloc((void**)&ctx->d_hot_id, sizeof(uint32_t) * kHotMax));
  ctx->v_num = v_num;
  ctx->m = m;
  return DG_OK;
}

static int edge_range_error(dg_ctx* ctx, const dg_edge* edges, uint64_t i, uint32_t v_num) {
  return dg_fail(ctx, DG_ERR_ARG, "edge %llu (%u, %u) out of range for %u vertices", (unsigned long long)i,
                 edges[i].src, edges[i].dst, v_num);
}

// The working memory of the device build: per entry two (source, entry)
// pairs and the reverse position, per edge its record, per tile the digit
// counts and their scan.
struct CsrScratch {
  uint64_t n_tiles = 0;
  dg_edge* edges = nullptr;
  uint32_t *keys[2] = {nullptr, nullptr}, *ids[2] = {nullptr, nullptr}, *hist = nullptr;
  uint64_t *base = nullptr, *rev = nullptr;
  float* w = nullptr;
  unsigned long long* bad = nullptr;

  bool get(Scratch& mem, uint64_t e_num, uint64_t m, bool want_rev, bool weighted) {
    n_tiles = (m + kSortTile - 1) / kSortTile;
    bool ok = mem.get(&edges, e_num) == hipSuccess && mem.get(&bad, 1) == hipSuccess;
    for (int b = 0; b < 2; ++b)
      ok = ok && mem.get(&keys[b], m) == hipSuccess && mem.get(&ids[b], m) == hipSuccess;
    ok = ok && mem.get(&hist, n_tiles * kDigits) == hipSuccess;
    ok = ok && mem.get(&base, n_tiles * kDigits + 1) == hipSuccess;
    if (want_rev) ok = ok && mem.get(&rev, m) == hipSuccess;
    if (weighted) ok = ok && mem.get(&w, m) == hipSuccess;
    return ok;
  }
};

// The edges on the device, and none of them out of range.
static int send_edges(dg_ctx* ctx, CsrScratch& t, uint32_t v_num, const dg_edge* edges, uint64_t e_num) {
  unsigned long long bad = ~0ull;
  set_u64_kernel<<<1, 64, 0, ctx->stream>>>(t.bad, bad);
  DG_HIP(ctx, hipMemcpyAsync(t.edges, edges, sizeof(dg_edge) * e_num, hipMemcpyHostToDevice, ctx->stream));
  edge_check_kernel<<<grid_for(ctx, e_num, 256), 256, 0, ctx->stream>>>(t.edges, e_num, v_num, t.bad);
  DG_HIP(ctx, hipGetLastError());
  DG_HIP(ctx, hipMemcpyAsync(&bad, t.bad, sizeof(bad), hipMemcpyDeviceToHost, ctx->stream));
  DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return bad == ~0ull ? DG_OK : edge_range_error(ctx, edges, bad, v_num);
}

// CSR built on the device from edges that are there: only the hubs and one
// flag come back.
static int build_on_device(dg_ctx* ctx, CsrScratch& t, uint32_t v_num, uint64_t e_num, int undirected, int cn_mode) {
  const uint64_t m = e_num * (undirected ? 2 : 1);
  DG_CHECK(alloc_graph(ctx, v_num, m));
  entry_keys_kernel<<<grid_for(ctx, e_num, 256), 256, 0, ctx->stream>>>(t.edges, e_num, undirected, t.keys[0],
                                                                       t.ids[0]);
  int bits = 1, cur = 0;
  while (bits < 32 && (1ull << bits) < v_num) ++bits;
  for (int shift = 0; shift < bits; shift += 8) {
    sort_hist_kernel<<<(unsigned)t.n_tiles, kSortThreads, 0, ctx->stream>>>(t.keys[cur], m, shift,
                                                                           (uint32_t)t.n_tiles, t.hist);
    DG_CHECK(dg_scan_lengths(ctx, t.hist, t.n_tiles * kDigits, t.base));
    sort_scatter_kernel<<<(unsigned)t.n_tiles, kSortThreads, 0, ctx->stream>>>(
        t.keys[cur], t.ids[cur], m, shift, (uint32_t)t.n_tiles, t.base, t.keys[1 - cur], t.ids[1 - cur]);
    cur = 1 - cur;
  }
  const uint32_t *src = t.keys[cur], *ids = t.ids[cur];
  row_ptr_kernel<<<grid_for(ctx, v_num + 1ull, 256), 256, 0, ctx->stream>>>(src, m, v_num, ctx->d_row_ptr);
  uint32_t* where = t.rev ? t.ids[1 - cur] : nullptr;
  entry_gather_kernel<<<grid_for(ctx, m, 256), 256, 0, ctx->stream>>>(
      t.edges, ids, m, undirected, ctx->d_nbr, cn_mode == DG_CN_FROM_DATA ? ctx->d_cn : nullptr, t.w, where);
  if (t.rev) reverse_kernel<<<grid_for(ctx, m, 256), 256, 0, ctx->stream>>>(ids, where, m, t.rev);
  DG_HIP(ctx, hipGetLastError());
  return finish_graph(ctx, t.w, t.rev, src, cn_mode);
}

// The device build takes some twenty launches and a dozen allocations whatever
// the size, the host's grows with it: a ring of 1,000 vertices (2,000 entries)
// 140 us on the host and 219 on the device, a Chung-Lu graph of 1,000 (16,000)
// 222 and 302, of 4,000 (64,000) 640 and 593, of 16,000 1,455 and 1,040.
constexpr uint64_t kDeviceSize = 1u << 15;  // entries and vertices together

// CSR built on the host (a small graph, entries past 32 bits, or no room for the
// device build and its working memory): include/graph.hpp:671-699 then :509-540, the
// doubled list counted and placed in order.
static int build_on_host(dg_ctx* ctx, uint32_t v_num, const dg_edge* edges, uint64_t e_num, int undirected,
                         int cn_mode) {
  const uint64_t m = e_num * (undirected ? 2 : 1);
  std::vector<uint64_t> rp(v_num + 1ull, 0);
  for (uint64_t i = 0; i < e_num; ++i) {
    rp[edges[i].src + 1ull]++;
    if (undirected) rp[edges[i].dst + 1ull]++;
  }
  for (uint32_t v = 0; v < v_num; ++v) rp[v + 1ull] += rp[v];
  std::vector<uint64_t> fill(rp.begin(), rp.end() - 1);
  std::vector<uint32_t> nbr(m);
  std::vector<uint32_t> cn;
  std::vector<float> weight;
  std::vector<uint64_t> rev;  // undirected: position of each entry's reverse entry
  const bool want_rev = undirected && cn_mode != DG_CN_FROM_DATA;
  if (want_rev) rev.resize(m);
  const bool from_data = cn_mode == DG_CN_FROM_DATA, weighted = cn_mode == DG_CN_COMPUTE_WEIGHTED;
  if (from_data) cn.resize(m);
  if (weighted) weight.resize(m);
  for (uint64_t i = 0; i < e_num; ++i) {
    const uint64_t p = fill[edges[i].src]++;
    nbr[p] = edges[i].dst;
    // walk.hpp:920 converts the float edge data to int
    const uint32_t c = from_data ? (uint32_t)(int)edges[i].data : 0u;
    if (from_data) cn[p] = c;
    if (weighted) weight[p] = edges[i].data;
    if (undirected) {
      const uint64_t q = fill[edges[i].dst]++;
      nbr[q] = edges[i].src;
      if (from_data) cn[q] = c;
      if (weighted) weight[q] = edges[i].data;
      if (want_rev) {
        rev[p] = q;
        rev[q] = p;
      }
    }
  }
  DG_CHECK(alloc_graph(ctx, v_num, m));
  Scratch mem;
  uint64_t* d_rev = nullptr;
  float* d_w = nullptr;
  DG_HIP(ctx, hipMemcpy(ctx->d_row_ptr, rp.data(), sizeof(uint64_t) * (v_num + 1ull), hipMemcpyHostToDevice));
  if (m) {
    DG_HIP(ctx, hipMemcpy(ctx->d_nbr, nbr.data(), sizeof(uint32_t) * m, hipMemcpyHostToDevice));
    if (from_data) DG_HIP(ctx, hipMemcpy(ctx->d_cn, cn.data(), sizeof(uint32_t) * m, hipMemcpyHostToDevice));
    if (want_rev) {
      DG_ROOM(ctx, mem.get(&d_rev, m));
      DG_HIP(ctx, hipMemcpy(d_rev, rev.data(), sizeof(uint64_t) * m, hipMemcpyHostToDevice));
    }
    if (weighted) {  // only needed for the thresholds, so not kept
      DG_ROOM(ctx, mem.get(&d_w, m));
      DG_HIP(ctx, hipMemcpy(d_w, weight.data(), sizeof(float) * m, hipMemcpyHostToDevice));
    }
  }
  return finish_graph(ctx, d_w, d_rev, nullptr, cn_mode);
}

extern "C" int dg_graph_from_edges(dg_ctx* ctx, uint32_t v_num, const dg_edge* edges,
                                   uint64_t e_num, int undirected, int cn_mode) {
  if (!ctx || (!edges && e_num) || v_num == 0) return DG_ERR_ARG;
  if (cn_mode != DG_CN_FROM_DATA && cn_mode != DG_CN_COMPUTE && cn_mode != DG_CN_COMPUTE_WEIGHTED)
    return dg_fail(ctx, DG_ERR_ARG, "unknown cn_mode %d", cn_mode);
  DG_HIP(ctx, hipSetDevice(ctx->device));
  const uint64_t m = e_num * (undirected ? 2 : 1);
  int rc = DG_ERR_NOMEM;
  if (m > 0 && m + v_num >= kDeviceSize && m < (1ull << 32)) {
    Scratch mem;
    CsrScratch t;
    if (t.get(mem, e_num, m, undirected && cn_mode != DG_CN_FROM_DATA, cn_mode == DG_CN_COMPUTE_WEIGHTED)) {
      DG_CHECK(send_edges(ctx, t, v_num, edges, e_num));  // the graph before stays
      rc = build_on_device(ctx, t, v_num, e_num, undirected, cn_mode);
    } else {
      (void)hipGetLastError();
    }
  }
  if (rc == DG_ERR_NOMEM) {
    for (uint64_t i = 0; i < e_num; ++i)
      if (edges[i].src >= v_num || edges[i].dst >= v_num) return edge_range_error(ctx, edges, i, v_num);
    rc = build_on_host(ctx, v_num, edges, e_num, undirected, cn_mode);
  }
  if (rc != DG_OK) dg_graph_free(ctx);  // never a part of one
  return rc;
}

extern "C" int dg_graph_load_bin(dg_ctx* ctx, const char* path, uint32_t v_num, int undirected,
                                 int cn_mode) {
  if (!ctx || !path) return DG_ERR_ARG;
  FILE* f = fopen(path, "rb");
  if (!f) return dg_fail(ctx, DG_ERR_IO, "cannot open %s", path);
  fseek(f, 0, SEEK_END);
  long sz = ftell(f);
  fseek(f, 0, SEEK_SET);
  if (sz < 0 || sz % (long)sizeof(dg_edge) != 0) {
    fclose(f);
    return dg_fail(ctx, DG_ERR_IO, "%s: size %ld is not a multiple of %zu", path, sz,
                   sizeof(dg_edge));
  }
  const uint64_t e_num = (uint64_t)sz / sizeof(dg_edge);
  std::vector<dg_edge> edges(e_num);
  const size_t got = e_num ? fread(edges.data(), sizeof(dg_edge), e_num, f) : 0;
  fclose(f);
  if (got != e_num) return dg_fail(ctx, DG_ERR_IO, "%s: short read", path);
  return dg_graph_from_edges(ctx, v_num, edges.data(), e_num, undirected, cn_mode);
}

extern "C" int dg_graph_info(dg_ctx* ctx, uint32_t* v_num, uint64_t* m) {
  if (!ctx) return DG_ERR_ARG;
  if (v_num) *v_num = ctx->v_num;
  if (m) *m = ctx->m;
  return DG_OK;
}

extern "C" int dg_graph_get_csr(dg_ctx* ctx, uint64_t* row_ptr, uint32_t* nbr, uint32_t* cn) {
  if (!ctx) return DG_ERR_ARG;
  if (!ctx->d_row_ptr) return dg_fail(ctx, DG_ERR_STATE, "no graph loaded");
  DG_HIP(ctx, hipSetDevice(ctx->device));
  DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (row_ptr)
    DG_CHECK(dg_copy_to_host(ctx, row_ptr, ctx->d_row_ptr, sizeof(uint64_t) * (ctx->v_num + 1ull)));
  if (nbr && ctx->m) DG_CHECK(dg_copy_to_host(ctx, nbr, ctx->d_nbr, sizeof(uint32_t) * ctx->m));
  if (cn && ctx->m) DG_CHECK(dg_copy_to_host(ctx, cn, ctx->d_cn, sizeof(uint32_t) * ctx->m));
  return DG_OK;
}

extern "C" int dg_graph_get_thresholds(dg_ctx* ctx, uint32_t* thr) {
  if (!ctx || !thr) return DG_ERR_ARG;
  if (!ctx->d_adj) return dg_fail(ctx, DG_ERR_STATE, "no graph loaded");
  DG_HIP(ctx, hipSetDevice(ctx->device));
  DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (ctx->m == 0) return DG_OK;
  Scratch mem;
  uint32_t* d_thr = nullptr;
  DG_ROOM(ctx, mem.get(&d_thr, ctx->m));
  take_thresholds_kernel<<<grid_for(ctx, ctx->m, 256), 256, 0, ctx->stream>>>(ctx->d_adj, ctx->m, d_thr);
  DG_HIP(ctx, hipGetLastError());
  DG_CHECK(dg_copy_to_host(ctx, thr, d_thr, sizeof(uint32_t) * ctx->m));
  return DG_OK;
}
