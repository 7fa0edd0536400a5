// walker.hip - persistent information-oriented walker for gfx950, and the
// per-round corpus packing and relative-entropy kernels.
//
// Reference: WalkEngine::internal_random_walk / internal_walk_epoch
// (include/walk.hpp:608-782, :789-1043) with Correlation (:260-387), for one
// partition.  PathCollector/PathSet (include/path.hpp) become a device token
// buffer in walk-id order.
//
// Design (MI355X-first, not a translation of the OpenMP/MPI loop):
//   * One lane per walk, 64 walks per wavefront, in one persistent launch.
//     Walks have uneven lengths; a lane whose walk ends takes the next walk id
//     from its wave's pool, and a wave refills its pool with one atomic on its
//     shard of the device work queue, so every lane stays busy until the shard
//     drains and every wave then leaves the loop.
//   * Each lane keeps its walk in LDS (kPathLds vertices, in 16-byte groups of
//     four) and spills longer walks to a private global area.  The visit count
//     f_i of walk.hpp:816 (an unordered_map per walk) is a scan of that
//     buffer: six 16-byte LDS reads in flight together, unused places holding
//     an id no vertex has.
//   * An adjacency unit carries the neighbour's row offset and degree beside
//     its id and bounce threshold (16 bytes), so a step reads one random
//     address, not two in a row.
//   * A finished walk goes into its own slot (walk index * kPathLds tokens) by
//     16-byte stores of its own lane; only walks longer than a slot take space
//     from a shared overflow cursor.
//   * Visit counts are not taken in the walk loop: the packing pass counts
//     every token, the highest-degree vertices in per-workgroup LDS counters
//     and the rest with uncontended global atomics.
//   * Every draw comes from the walk's own Philox stream (dg_philox.h), and the
//     FP64 entropy/acceptance math uses dg_math.h, so the corpus is the same
//     bits as the CPU oracle's whatever the schedule.
#include <algorithm>

#include "dg_internal.h"
#include "dg_math.h"
#include "dg_philox.h"

namespace {

constexpr int kWalkBlock = 256;
constexpr int kPathLds = 24;    // vertices per lane kept in LDS; reference walks hold 22
constexpr int kPathVec = kPathLds / 4;
constexpr uint32_t kNoVertex = 0xffffffffu;  // never a vertex id (ids are below a 32-bit count)
constexpr int kTermTable = 32;  // entropy terms tabulated for walks shorter than 32
constexpr int kTermStride = kTermTable + 1;
constexpr uint32_t kPool = 64;
constexpr uint32_t kDefaultLengthLimit = DG_WALK_LENGTH_LIMIT_DEFAULT;

struct WalkArgs {
  const uint64_t* row_ptr;
  const uint4* adj;  // {neighbour, bounce threshold, neighbour's row} (dg_pack_row)
  const double* term_table;
  uint32_t v_num;
  uint32_t round;
  uint64_t seed;
  uint32_t walker_begin;
  uint32_t walker_num;
  uint32_t min_length;
  uint32_t max_length;
  uint32_t length_limit;
  uint32_t spill_per_slot;
  double mu;
  uint32_t* tokens;   // raw buffer: walker_num slots of kPathLds, then the overflow region
  uint64_t tok_cap;
  uint64_t slots_end;  // walker_num * kPathLds
  uint64_t* walk_off;
  uint32_t* walk_len;
  uint32_t* spill;
  dg_walk_queue* q;
  dg_walk_shard* shards;
};

// Running statistics of Correlation (include/walk.hpp:260-387).  Sn and N
// both equal the number of vertices on the walk, which the kernel keeps as an
// integer, and the moments of S alone (ES, ESS) depend only on it: they are
// tabulated up to kTermTable vertices and kept in registers past that.
struct WalkState {
  double H, EH, EHS, EHH;
  double ES, ESS;  // past kTermTable vertices only
};

// x / n for an integer n, given y = 1 / n correctly rounded: two corrections
// of x * y by the exact remainder give the correctly rounded quotient
// (Markstein 1990), in 5 operations instead of a division's dozen.  x and
// the remainders are far from the ends of the exponent range here.
__device__ __forceinline__ double div_by(double x, double n, double y) {
  double q = x * y;
  q = __builtin_fma(__builtin_fma(-n, q, x), y, q);
  return __builtin_fma(__builtin_fma(-n, q, x), y, q);
}

// log2 term of Correlation::iterateHn with step_k = 1 (include/walk.hpp:
// 284-304) for a walk of Sn vertices appending a vertex seen fi times before:
// log2(pow(Sn/(Sn+1), Sn) * pow(1/(Sn+1), 1) [* pow((fi+1)/fi, fi) * pow(fi+1, 1)]).
__device__ __forceinline__ double entropy_term(double Sn, double fi) {
  const double one = 1.0;
  const double Sn1 = Sn + one;
  const double prod = dg_pow(Sn / Sn1, Sn) * dg_pow(one / Sn1, one);
  if (fi == 0.0) return dg_log2(prod);
  const double fj = fi + one;
  const double fac = dg_pow(fj / fi, fi) * dg_pow(fj, one);
  return dg_log2(prod * fac);
}

// Rest of Correlation::iterate (include/walk.hpp:317-354), same operation
// order.  The correlation R itself is only read by the termination test
// (walk.hpp:979-985), which runs after min_length steps, so it is formed from
// the moments there (state_corr) instead of on every step.
// y = 1 / (Sn + 1), correctly rounded.
__device__ __forceinline__ void state_iterate(WalkState& w, double Sn, double t, double y) {
  const double S1 = Sn + 1.0;
  const double H1 = div_by(Sn * w.H - t, S1, y);
  w.EH = w.EH + div_by(H1 - w.EH, S1, y);
  w.EHS = w.EHS + div_by(H1 * S1 - w.EHS, S1, y);
  w.EHH = w.EHH + div_by(H1 * H1 - w.EHH, S1, y);
  w.H = H1;
}

// The same step of the moments of S.
__device__ __forceinline__ void size_iterate(double& ES, double& ESS, double Sn, double y) {
  const double S1 = Sn + 1.0;
  ES = ES + div_by(S1 - ES, S1, y);
  ESS = ESS + div_by(S1 * S1 - ESS, S1, y);
}

// Pearson R of the (H, S) history from the running moments (walk.hpp:342-354).
__device__ __forceinline__ double state_corr(const WalkState& w, double ES, double ESS) {
  const double DH = w.EHH - w.EH * w.EH;
  const double DS = ESS - ES * ES;
  const double cov = w.EHS - w.EH * ES;
  return cov == 0.0 ? 0.0 : cov / dg_sqrt(DH * DS);
}

// Tables of the walk: term[S * kTermStride + f] = entropy_term(S, f) for
// 1 <= S < kTermTable, 0 <= f <= S, computed by the same device code the
// walker would run inline; then for n <= kTermTable vertices 1 / n, ES and ESS.
constexpr int kTermWords = kTermTable * kTermStride;
constexpr int kTabInv = kTermWords, kTabES = kTabInv + kTermTable + 1, kTabESS = kTabES + kTermTable + 1;
constexpr int kTabWords = kTabESS + kTermTable + 1;

__global__ void term_table_kernel(double* tbl) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < kTermWords) {
    const int S = i / kTermStride, f = i % kTermStride;
    tbl[i] = (S >= 1 && f <= S) ? entropy_term((double)S, (double)f) : 0.0;
  }
  if (i == 0) {
    double ES = 1.0, ESS = 1.0;
    tbl[kTabInv] = tbl[kTabES] = tbl[kTabESS] = 0.0;
    for (int n = 1; n <= kTermTable; ++n) {
      const double y = 1.0 / (double)n;
      if (n > 1) size_iterate(ES, ESS, (double)(n - 1), y);
      tbl[kTabInv + n] = y;
      tbl[kTabES + n] = ES;
      tbl[kTabESS + n] = ESS;
    }
  }
}

// A lane's draws: the words of its stream (dg_stream), two Philox blocks deep.
// The lanes of a wavefront run out at different steps, and a block evaluated
// for one lane costs the wavefront as much as one for all: so when any lane
// has fewer than the two words a step takes, every lane with room evaluates
// its next block, and the wavefront evaluates one block per two steps at
// most (it was one or two per step).
struct WalkDraws {
  uint32_t k0, k1, c1, c2, block;
  uint32_t b[4], n[4];   // words in hand (shifted down), and the next block
  uint32_t avail;        // words in b
  bool next;             // n holds a block

  __device__ __forceinline__ void start(uint64_t seed, uint32_t walk, uint32_t round) {
    k0 = (uint32_t)seed;
    k1 = (uint32_t)(seed >> 32);
    c1 = walk;
    c2 = round;
    block = 0;
    avail = 0;
    next = false;
  }
  __device__ __forceinline__ bool low() const { return avail < 2 && !next; }
  __device__ __forceinline__ void refill() {
    if (next) return;
    const dg_u32x4 o = dg_philox4x32_10(block, c1, c2, DG_TAG_WALK, k0, k1);
    ++block;
    n[0] = o.x0;
    n[1] = o.x1;
    n[2] = o.x2;
    n[3] = o.x3;
    next = true;
  }
  // needs a word in hand or a next block
  __device__ __forceinline__ uint32_t take() {
    if (avail == 0) {
      b[0] = n[0];
      b[1] = n[1];
      b[2] = n[2];
      b[3] = n[3];
      avail = 4;
      next = false;
    }
    const uint32_t r = b[0];
    b[0] = b[1];
    b[1] = b[2];
    b[2] = b[3];
    --avail;
    return r;
  }
  // dg_stream_uniform; leaves at least one word for dg_stream_u31
  __device__ __forceinline__ uint32_t uniform(uint32_t range) {
    uint64_t m = (uint64_t)take() * (uint64_t)range;
    if ((uint32_t)m < range) {
      const uint32_t t = (uint32_t)(0u - range) % range;
      while ((uint32_t)m < t) {  // a rejected word: once in 2^32 / range draws
        if (low()) refill();
        m = (uint64_t)take() * (uint64_t)range;
      }
      if (low()) refill();
    }
    return (uint32_t)(m >> 32);
  }
};

__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) {
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}

// Bound: at small rounds (fewer walks than lanes) the latency of one walk's
// chain, per step one random adjacency read (about 1,100 cycles), the scan of
// the walk, the entropy arithmetic and half a Philox block (300 to 700
// each); at large ones the instructions of four wavefronts per SIMD.
// 10,000 vertices (50,000 walks): 107 -> 46 us; 262,144 vertices: 1.31M walks
// 655 -> 303 us, 262,144 walks 352 -> 75 us.  Most of it is the sharded queue;
// the one-read step, the 16-byte scan, the reciprocals and the shared Philox
// evaluations took 12% with the queue as it was.
__global__ __launch_bounds__(kWalkBlock) void walk_kernel(WalkArgs a) {
  __shared__ uint4 s_path[kPathVec * kWalkBlock];  // [group of four][thread]
  __shared__ double s_tab[kTabWords];
  for (int i = threadIdx.x; i < kTabWords; i += kWalkBlock) s_tab[i] = a.term_table[i];
  __syncthreads();

  const uint32_t lane = threadIdx.x & 63u;
  uint32_t* path = reinterpret_cast<uint32_t*>(s_path + threadIdx.x);
  const uint64_t slot = (uint64_t)blockIdx.x * kWalkBlock + threadIdx.x;
  uint32_t* spill = a.spill + slot * a.spill_per_slot;

  // this workgroup's shard of the walks, dealt out in pools of 64: pool p is
  // workgroup (p mod grid)'s, and a shard hands out its workgroups' pools in
  // order.  A contiguous range each leaves most shards without work where the
  // ids follow the degrees (walks start at id mod V): a round on R-MAT scale 25
  // 10.5 ms, and 9.1 so (8.95 with one counter and no shards).
  const uint32_t n_sh = gridDim.x < kWalkShards ? gridDim.x : kWalkShards;
  const uint32_t sh = blockIdx.x % n_sh, b_mine = gridDim.x / n_sh + (sh < gridDim.x % n_sh ? 1u : 0u);
  dg_walk_shard* const shard = a.shards + sh;

  bool active = false;
  bool drained = false;                   // wave-uniform
  uint64_t pool_next = 0, pool_end = 0;   // wave-uniform

  uint32_t wid = 0, cur = 0, cur_deg = 0, len = 0;
  uint64_t cur_rb = 0;
  bool cur_stuck = false;                 // degree 2, itself its first neighbour
  // this lane's totals over its walks, added to the queue once per wave at the end
  uint64_t tot_draw = 0, tot_move = 0, tot_tok = 0;
  uint32_t max_l = 0;
  bool pending_back = false;
  WalkState ws = {0, 0, 0, 0, 0, 0};
  WalkDraws rs;
  rs.start(a.seed, 0, 0);

  while (true) {
    // ---- hand new walk ids to idle lanes --------------------------------
    if (!drained) {
      const uint64_t want = __ballot(!active);
      if (want != 0) {
        const uint32_t nwant = (uint32_t)__popcll(want);
        const uint32_t rank = lanes_below(want);
        const uint64_t avail = pool_end - pool_next;
        uint64_t id;
        if (avail >= nwant) {
          id = pool_next + rank;
          pool_next += nwant;
        } else {
          uint32_t c = 0;
          if (lane == 0) c = atomicAdd(&shard->next, 1u);
          c = __builtin_amdgcn_readfirstlane(c);
          const uint64_t base = ((uint64_t)(c / b_mine) * gridDim.x + sh + (c % b_mine) * n_sh) * kPool;
          id = rank < avail ? pool_next + rank : base + (rank - avail);
          pool_next = base + (nwant - avail);
          pool_end = base + kPool;
        }
        if (!active && id < a.walker_num) {
          // walk.hpp:529-589 (start = id mod V), :661-669 (footprint, step 0),
          // :849-856 (first-visit state)
          wid = (uint32_t)id;
          const uint32_t w = a.walker_begin + wid;
          cur = w % a.v_num;
          cur_rb = a.row_ptr[cur];
          cur_deg = (uint32_t)(a.row_ptr[cur + 1] - cur_rb);
          cur_stuck = cur_deg == 2 && a.adj[cur_rb].x == cur;
#pragma unroll
          for (int j = 0; j < kPathVec; ++j)
            s_path[j * kWalkBlock + threadIdx.x] =
                make_uint4(j == 0 ? cur : kNoVertex, kNoVertex, kNoVertex, kNoVertex);
          len = 1;
          ++tot_move;
          pending_back = false;
          ws.H = 0.0;
          ws.EH = 0.0;
          ws.EHS = 0.0;
          ws.EHH = 0.0;
          rs.start(a.seed, w, a.round);
          active = true;
        }
        if (__ballot(!active) != 0) drained = true;
      }
    }
    if (__ballot(active) == 0) {
      if (drained) break;
      continue;
    }
    if (__ballot(active && rs.low()) != 0) rs.refill();

    // ---- one appended vertex per active lane ------------------------------
    bool finish = false;
    if (active) {
      if (a.max_length != 0 && len >= a.max_length) {
        finish = true;
      } else {
        bool append = false;
        bool trace = false;
        uint32_t v_app = 0;
        uint2 next_row = make_uint2(0u, 0u);  // row of the vertex moved to
        if (pending_back) {
          v_app = cur;  // walk.hpp:986-1017: back to the current vertex
          append = true;
        } else if (cur_deg == 0) {
          finish = true;  // walk.hpp:887-892
        } else {
          const uint32_t i = rs.uniform(cur_deg);  // walk.hpp:899
          const uint4 e = a.adj[cur_rb + i];
          ++tot_draw;
          if (cur_stuck) {
            finish = true;  // walk.hpp:900-902
          } else if (!(len == 1 && e.x == cur)) {  // walk.hpp:904-906 redraw at step 0
            const uint32_t u = rs.take() >> 1;  // walk.hpp:928
            trace = (u >= e.y);                // walk.hpp:933-938 via the threshold
            v_app = e.x;
            append = true;
            next_row = make_uint2(e.z, e.w);
          }
        }
        if (append) {
          // walk.hpp:961-985: footprint, f_i = visits so far, entropy update
          uint32_t f4[4] = {0u, 0u, 0u, 0u};  // four chains of adds
#pragma unroll
          for (int j = 0; j < kPathVec; ++j) {
            const uint4 p = s_path[j * kWalkBlock + threadIdx.x];
            f4[0] += p.x == v_app;
            f4[1] += p.y == v_app;
            f4[2] += p.z == v_app;
            f4[3] += p.w == v_app;
          }
          uint32_t fi = (f4[0] + f4[1]) + (f4[2] + f4[3]);
          for (uint32_t j = kPathLds; j < len; ++j) fi += (spill[j - kPathLds] == v_app);
          double t, y;
          if (len < (uint32_t)kTermTable) {
            t = s_tab[len * kTermStride + fi];
            y = s_tab[kTabInv + len + 1];
          } else {
            t = entropy_term((double)len, (double)fi);
            y = 1.0 / ((double)len + 1.0);
            if (len == (uint32_t)kTermTable) {
              ws.ES = s_tab[kTabES + kTermTable];
              ws.ESS = s_tab[kTabESS + kTermTable];
            }
            size_iterate(ws.ES, ws.ESS, (double)len, y);
          }
          state_iterate(ws, (double)len, t, y);
          if (len < (uint32_t)kPathLds)
            path[(len >> 2) * (kWalkBlock * 4) + (len & 3u)] = v_app;
          else
            spill[len - kPathLds] = v_app;
          ++len;
          const uint32_t step = len - 1;
          bool ends = false;
          if (step > a.min_length) {
            const bool tab = len <= (uint32_t)kTermTable;
            const double R = state_corr(ws, tab ? s_tab[kTabES + len] : ws.ES, tab ? s_tab[kTabESS + len] : ws.ESS);
            ends = R * R < a.mu || R < 0.0;
          }
          if (ends) {
            finish = true;
          } else if (a.max_length != 0 && len >= a.max_length) {
            finish = true;
          } else if (len >= a.length_limit) {
            finish = true;
            atomicOr(&a.q->flags, DG_QFLAG_LENGTH_LIMIT);
          } else if (len == (uint32_t)kPathLds && a.spill_per_slot == 0) {
            finish = true;  // the round is walked again, with spill space
            atomicOr(&a.q->flags, DG_QFLAG_NO_SPILL);
          } else if (pending_back) {
            pending_back = false;
          } else if (trace) {
            pending_back = true;
          } else {
            cur = v_app;  // walk.hpp:1018-1023
            cur_rb = dg_row_begin(next_row);
            cur_deg = dg_row_degree(next_row);
            cur_stuck = dg_row_stuck(next_row);
            if (cur_deg == kRowDegMax) {  // the packed degree is full: read the row
              cur_deg = (uint32_t)(a.row_ptr[cur + 1] - cur_rb);
              cur_stuck = false;
            }
            ++tot_move;
          }
        }
      }
    }

    // ---- write finished walks out, each by its own lane -------------------
    // A walk of up to kPathLds vertices goes to its own slot of the raw buffer
    // (walk index * kPathLds, whose place the packing knows); longer walks
    // take space after the slots from an overflow cursor.  No wave waits on a
    // shared counter for a short walk.
    if (finish) {
      tot_tok += len;
      max_l = len > max_l ? len : max_l;
      a.walk_len[wid] = len;
      if (len <= (uint32_t)kPathLds) {
        uint4* dst = reinterpret_cast<uint4*>(a.tokens + (uint64_t)wid * kPathLds);
#pragma unroll
        for (int j = 0; j < kPathVec; ++j) dst[j] = s_path[j * kWalkBlock + threadIdx.x];
      } else {
        const uint64_t off = a.slots_end + atomicAdd(&a.q->cursor, (unsigned long long)len);
        a.walk_off[wid] = off;
        if (off + len <= a.tok_cap) {
          for (uint32_t j = 0; j < (uint32_t)kPathLds; ++j)
            a.tokens[off + j] = path[(j >> 2) * (kWalkBlock * 4) + (j & 3u)];
          for (uint32_t j = kPathLds; j < len; ++j) a.tokens[off + j] = spill[j - kPathLds];
        } else {
          atomicOr(&a.q->flags, DG_QFLAG_TOKEN_OVERFLOW);
        }
      }
      active = false;
    }
  }
  // ---- the lane totals, added to the shard once per wave
  const uint64_t wd = wave_sum_u64(tot_draw), wm = wave_sum_u64(tot_move), wt = wave_sum_u64(tot_tok);
  uint32_t wmax = max_l;
  for (int d = 32; d >= 1; d >>= 1) {
    const uint32_t o = __shfl_xor(wmax, d, 64);
    wmax = o > wmax ? o : wmax;
  }
  if (lane == 0) {
    if (wd) atomicAdd(&shard->draws, (unsigned long long)wd);
    if (wm) atomicAdd(&shard->moves, (unsigned long long)wm);
    if (wt) atomicAdd(&shard->tokens, (unsigned long long)wt);
    if (wmax) atomicMax(&shard->max_len, wmax);
  }
}

// Empties a round that overflowed the token buffer, hit the length limit or
// lacked spill space (every walk length 0), so the kernels after it leave the
// visit counts and the tables as they were.
//
// Its first wavefront also adds the shards' totals into the queue.
__global__ void round_guard_kernel(dg_walk_queue* q, uint32_t* walk_len, uint32_t n, const dg_walk_shard* shards) {
  static_assert(kWalkShards == 64, "a lane per shard");
  if (blockIdx.x == 0 && threadIdx.x < 64) {
    const dg_walk_shard s = shards[threadIdx.x];
    const uint64_t draws = wave_sum_u64(s.draws), moves = wave_sum_u64(s.moves), tokens = wave_sum_u64(s.tokens);
    uint32_t most = s.max_len;
    for (int d = 32; d >= 1; d >>= 1) {
      const uint32_t o = __shfl_xor(most, d, 64);
      most = o > most ? o : most;
    }
    if (threadIdx.x == 0) {
      q->draws = draws;
      q->moves = moves;
      q->tokens = tokens;
      q->max_len = most;
    }
  }
  if (q->flags == 0) return;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    walk_len[i] = 0;
}

__global__ void zero_first_kernel(uint64_t* p) {
  if (threadIdx.x == 0 && blockIdx.x == 0) p[0] = 0;
}

__global__ __launch_bounds__(64) void queue_reset_kernel(dg_walk_queue* q, dg_walk_shard* shards) {
  shards[threadIdx.x] = dg_walk_shard{};
  if (threadIdx.x == 0) *q = dg_walk_queue{};
}

__global__ void fill_u32_kernel(uint32_t* p, uint64_t n, uint32_t v) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// ---- exclusive scan of walk lengths (three phases, 1024 items per block) ----
constexpr int kScanBlock = 256;
constexpr int kScanItems = 4;
constexpr int kScanTile = kScanBlock * kScanItems;

__device__ uint64_t block_exclusive_scan(uint64_t v, uint64_t* s_wave, uint64_t* total) {
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint64_t incl = v;
  for (int d = 1; d < 64; d <<= 1) {
    const uint64_t t = __shfl_up(incl, d, 64);
    if ((int)lane >= d) incl += t;
  }
  if (lane == 63) s_wave[wave] = incl;
  __syncthreads();
  uint64_t wave_prefix = 0, sum = 0;
  for (uint32_t w = 0; w < kScanBlock / 64; ++w) {
    if (w < wave) wave_prefix += s_wave[w];
    sum += s_wave[w];
  }
  __syncthreads();
  *total = sum;
  return wave_prefix + incl - v;
}

__global__ __launch_bounds__(kScanBlock) void scan_tile_sums(const uint32_t* len, uint64_t n,
                                                             uint64_t* tile_sums) {
  __shared__ uint64_t s_wave[kScanBlock / 64];
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  uint64_t s = 0;
  for (int k = 0; k < kScanItems; ++k)
    if (base + k < n) s += len[base + k];
  uint64_t total;
  block_exclusive_scan(s, s_wave, &total);
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

// Exclusive scan of the tile sums in one block; tile_sums[n_tiles] gets the total.
__global__ __launch_bounds__(kScanBlock) void scan_tile_prefix(uint64_t* tile_sums,
                                                               uint64_t n_tiles) {
  __shared__ uint64_t s_wave[kScanBlock / 64];
  const uint64_t per = (n_tiles + kScanBlock - 1) / kScanBlock;
  const uint64_t lo = threadIdx.x * per;
  const uint64_t hi = lo + per < n_tiles ? lo + per : n_tiles;
  uint64_t s = 0;
  for (uint64_t i = lo; i < hi; ++i) s += tile_sums[i];
  uint64_t total;
  uint64_t run = block_exclusive_scan(s, s_wave, &total);
  for (uint64_t i = lo; i < hi; ++i) {
    const uint64_t t = tile_sums[i];
    tile_sums[i] = run;
    run += t;
  }
  if (threadIdx.x == 0) tile_sums[n_tiles] = total;
}

__global__ __launch_bounds__(kScanBlock) void scan_tile_apply(const uint32_t* len, uint64_t n,
                                                              const uint64_t* tile_prefix,
                                                              uint64_t n_tiles, uint64_t* off) {
  __shared__ uint64_t s_wave[kScanBlock / 64];
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  uint64_t v[kScanItems];
  uint64_t s = 0;
  for (int k = 0; k < kScanItems; ++k) {
    v[k] = base + k < n ? len[base + k] : 0;
    s += v[k];
  }
  uint64_t total;
  uint64_t run = block_exclusive_scan(s, s_wave, &total) + tile_prefix[blockIdx.x];
  for (int k = 0; k < kScanItems; ++k) {
    if (base + k < n) off[base + k] = run;
    run += v[k];
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) off[n] = tile_prefix[n_tiles];
}

// ---- corpus packing in walk-id order, and the round's visit counts ------
// (path.hpp:91,95: context_map_freq / vertex_cn).  A wavefront takes 64
// consecutive walks, a lane each: the walk's slot is read into registers
// (six 16-byte loads), each of its distinct vertices counted once with its
// multiplicity (walks revisit their hub at every other step; equal pairs are
// found by comparing registers), and the 64 walks, which are one run of the
// packed corpus, leave through LDS as one coalesced copy.  A hot vertex
// (hot_slot != kNotHot) is counted in this workgroup's LDS counters, written
// out as one partial row at the end.
//
// The other vertices are what the counting costs: an atomic each on a random
// counter goes at about 30 G/s however the counters are spread (0.33 of the
// 0.45 ms of a 1.31M-walk round, the same with a counter array per XCD).  So
// with BIN a tile of walks sorts its (vertex, multiplicity) entries
// into kBins bins by vertex in LDS, and writes them over its own slots in the
// raw buffer (all read by then), with the bins' offsets in bin_off; a
// workgroup of bin_count_kernel then adds up the entries of one bin of many
// tiles in LDS counters.  That takes graphs whose vertices fit the bins'
// counters (kBinVertices); larger ones keep the atomics.
// Walks longer than a slot are copied and counted by the whole wavefront.
// The workgroup's threads are the tile's walks: 1,024 (a workgroup per CU), or
// 256 where a round has fewer walks than that fills the CUs with.
constexpr int kPackBig = 1024, kPackSmall = 256;
constexpr int kBins = 128;
constexpr uint32_t kBinCounters = 32768;  // counters of a bin: 128 KB of LDS
constexpr uint32_t kBinVertices = kBins * kBinCounters;

// Bin and place in it of a vertex: runs of 16 counters (64 bytes of the
// visit counts) go to the bins in turn, so that neighbouring ids, which often
// have similar degrees, spread over the bins.
__host__ __device__ __forceinline__ uint32_t bin_of(uint32_t v) { return (v >> 4) % kBins; }
__host__ __device__ __forceinline__ uint32_t bin_place(uint32_t v) { return (v >> 4) / kBins * 16u + (v & 15u); }
__host__ __device__ __forceinline__ uint32_t bin_vertex(uint32_t bin, uint32_t place) {
  return ((place >> 4) * kBins + bin) * 16u + (place & 15u);
}

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int kPackBlock, bool BIN>
__global__ __launch_bounds__(kPackBlock) void pack_count_kernel(
    uint32_t* raw, const uint64_t* walk_off, const uint32_t* walk_len, const uint64_t* out_off,
    uint64_t n_walks, uint32_t* tokens, const uint16_t* hot_slot, uint32_t n_hot, uint32_t* freq,
    uint32_t* hot_part, uint32_t* bin_off) {
  __shared__ uint32_t s_hot[kHotMax];
  __shared__ uint32_t s_out[kPackBlock * kPathLds];
  __shared__ uint32_t s_bin[kBins], s_first[kBins + 1];
  for (uint32_t k = threadIdx.x; k < n_hot; k += kPackBlock) s_hot[k] = 0;
  if (threadIdx.x < kBins) s_bin[threadIdx.x] = 0;
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63u, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t* out = s_out + wv * (64 * kPathLds);
  const uint64_t n_tiles = (n_walks + kPackBlock - 1) / kPackBlock;
  for (uint64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    const uint64_t w0 = tile * kPackBlock + wv * 64;
    const uint64_t w = w0 + lane;
    const bool ok = w < n_walks;
    const uint32_t len = ok ? walk_len[w] : 0u;
    const uint64_t dst = ok ? out_off[w] : 0ull;
    const uint64_t base = __shfl(dst, 0, 64);
    const uint64_t too_long = __ballot(len > (uint32_t)kPathLds);
    const bool mine = ok && len <= (uint32_t)kPathLds;
    uint32_t t[kPathLds];
    // entry of the vertex at place i (BIN): multiplicity, and above it its
    // rank in the tile's bin; 0 where it is not a bin's entry
    uint32_t n[kPathLds];
    if (mine) {
      const uint4* slot = reinterpret_cast<const uint4*>(raw + w * kPathLds);
#pragma unroll
      for (int j = 0; j < kPathVec; ++j) {
        const uint4 q = slot[j];
        t[4 * j] = q.x;
        t[4 * j + 1] = q.y;
        t[4 * j + 2] = q.z;
        t[4 * j + 3] = q.w;
      }
      // occurrences of the vertex at i from i on, and whether i is its first
      uint32_t again = 0;
#pragma unroll
      for (int i = 0; i < kPathLds; ++i) n[i] = 1;
#pragma unroll
      for (int i = 0; i < kPathLds; ++i)
#pragma unroll
        for (int j = i + 1; j < kPathLds; ++j) {
          const bool same = t[i] == t[j];
          n[i] += same ? 1u : 0u;
          again |= same ? 1u << j : 0u;
        }
#pragma unroll
      for (int i = 0; i < kPathLds; ++i) {
        if ((uint32_t)i >= len || ((again >> i) & 1u)) {
          n[i] = 0;
          continue;
        }
        const uint16_t hs = hot_slot[t[i]];
        if (hs != kNotHot) {
          atomicAdd(&s_hot[hs], n[i]);
          n[i] = 0;
        } else if constexpr (BIN) {
          n[i] |= atomicAdd(&s_bin[bin_of(t[i])], 1u) << 8;
        } else {
          atomicAdd(&freq[t[i]], n[i]);
        }
      }
      if (too_long == 0) {
        const uint32_t o = (uint32_t)(dst - base);
#pragma unroll
        for (int i = 0; i < kPathLds; ++i)
          if ((uint32_t)i < len) out[o + i] = t[i];
      } else {
#pragma unroll
        for (int i = 0; i < kPathLds; ++i)
          if ((uint32_t)i < len) tokens[dst + i] = t[i];
      }
    }
    if (too_long == 0) {
      uint32_t total = len;
#pragma unroll
      for (int d = 32; d >= 1; d >>= 1) total += __shfl_xor(total, d, 64);
      wave_lds_sync();
      for (uint32_t i = lane; i < total; i += 64) tokens[base + i] = out[i];
      wave_lds_sync();
    }
    for (uint64_t m = too_long; m != 0; m &= m - 1) {
      const int l = __builtin_ctzll(m);
      const uint64_t src = walk_off[w0 + l], d = __shfl(dst, l, 64);
      const uint32_t nl = __shfl(len, l, 64);
      for (uint32_t i = lane; i < nl; i += 64) {
        const uint32_t v = raw[src + i];
        tokens[d + i] = v;
        const uint16_t hs = hot_slot[v];
        if (hs != kNotHot)
          atomicAdd(&s_hot[hs], 1u);
        else
          atomicAdd(&freq[v], 1u);
      }
    }
    if constexpr (BIN) {
      __syncthreads();  // every rank is taken, every slot of the tile read
      if (wv == 0) {
        static_assert(kBins == 128, "two bins per lane");
        const uint32_t c0 = s_bin[2 * lane], c1 = s_bin[2 * lane + 1];
        uint32_t inc = c0 + c1;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const uint32_t u = __shfl_up(inc, d, 64);
          if ((int)lane >= d) inc += u;
        }
        s_first[2 * lane] = inc - c0 - c1;
        s_first[2 * lane + 1] = inc - c1;
        if (lane == 63) s_first[kBins] = inc;
        s_bin[2 * lane] = 0;
        s_bin[2 * lane + 1] = 0;
      }
      __syncthreads();
      if (mine) {
#pragma unroll
        for (int i = 0; i < kPathLds; ++i)
          if (n[i]) s_out[s_first[bin_of(t[i])] + (n[i] >> 8)] = bin_place(t[i]) | (n[i] & 0xffu) << 16;
      }
      if (threadIdx.x <= kBins) bin_off[tile * (kBins + 1) + threadIdx.x] = s_first[threadIdx.x];
      __syncthreads();
      const uint32_t total = s_first[kBins];
      for (uint32_t i = threadIdx.x; i < total; i += kPackBlock) raw[tile * (kPackBlock * kPathLds) + i] = s_out[i];
      __syncthreads();  // s_out is the next tile's
    }
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < n_hot; k += kPackBlock)
    hot_part[(uint64_t)blockIdx.x * n_hot + k] = s_hot[k];
}

// Workgroup (bin, part): the bin's entries of its share of the tiles, a
// wavefront per tile, added up in LDS and then to the visit counts.  Entries: place, and the multiplicity from bit 16.
constexpr int kBinBlock = 1024;

__global__ __launch_bounds__(kBinBlock) void bin_count_kernel(const uint32_t* raw, const uint32_t* bin_off,
                                                              uint64_t n_tiles, uint32_t tile_words, uint32_t v_num, uint32_t places,
                                                              uint32_t* freq) {
  extern __shared__ uint32_t s_cnt[];
  const uint32_t bin = blockIdx.x;
  for (uint32_t i = threadIdx.x; i < places; i += kBinBlock) s_cnt[i] = 0;
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63u, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr uint32_t waves = kBinBlock / 64;
  for (uint64_t tile = (uint64_t)blockIdx.y * waves + wv; tile < n_tiles; tile += (uint64_t)gridDim.y * waves) {
    const uint32_t lo = bin_off[tile * (kBins + 1) + bin], hi = bin_off[tile * (kBins + 1) + bin + 1];
    const uint32_t* e = raw + tile * tile_words;
    for (uint32_t i = lo + lane; i < hi; i += 64) {
      const uint32_t x = e[i];
      atomicAdd(&s_cnt[x & 0xffffu], x >> 16);
    }
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < places; i += kBinBlock) {
    const uint32_t v = bin_vertex(bin, i), c = s_cnt[i];
    if (c && v < v_num) atomicAdd(&freq[v], c);
  }
}

// Hot-vertex counts: the partial rows summed per slot.  Grid (slots / 64,
// rows / kHotRows): each thread adds kHotRows partial rows of one slot
// (coalesced across the slots of a wavefront, all loads in flight) and adds
// that to the vertex's count.
constexpr uint32_t kHotRows = 32;

__global__ __launch_bounds__(64) void hot_reduce_kernel(const uint32_t* hot_part, uint32_t n_parts,
                                                        uint32_t n_hot, const uint32_t* hot_id,
                                                        uint32_t* freq) {
  const uint32_t k = blockIdx.x * 64 + threadIdx.x;
  if (k >= n_hot) return;
  const uint32_t b0 = blockIdx.y * kHotRows;
  uint32_t v[kHotRows];
#pragma unroll
  for (uint32_t r = 0; r < kHotRows; ++r) v[r] = b0 + r < n_parts ? hot_part[(uint64_t)(b0 + r) * n_hot + k] : 0u;
  uint32_t c = 0;
#pragma unroll
  for (uint32_t r = 0; r < kHotRows; ++r) c += v[r];
  if (c) atomicAdd(&freq[hot_id[k]], c);
}

// ---- relative entropy (walk.hpp:693-725) in a fixed summation order -------
// Terms p_i (ln p_i - ln q_i); chunk sums of 1024 consecutive terms added
// left to right, then the chunk sums added left to right.
constexpr uint32_t kReChunk = 1024;

// One workgroup per chunk: its terms into LDS (four per thread), then the sum
// left to right by one lane.  The order makes a chunk 1,024 dependent FP64
// adds, so the sum is bound by their latency: reading them from LDS, several
// ahead, one add is all that is on the chain: 16 us plus 4 us for the chunk
// sums at 262,144 vertices, 114 us with the running sum taken through lane
// shuffles and the terms passed through memory.  wsum = the visits counted
// before this round plus the round's tokens (from the queue, so the host need
// not know the round's token count).  A vertex without a term adds 0, which
// leaves the running sum's bits as they are.
constexpr int kReBlock = 256;

// Sum of n LDS values left to right, sixteen values read ahead of the adds.
__device__ __forceinline__ double ordered_sum(const double* v, uint32_t n, double sum) {
  uint32_t i = 0;
  for (; i + 16 <= n; i += 16) {
    double t[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) t[u] = v[i + u];
#pragma unroll
    for (int u = 0; u < 16; ++u) sum = sum + t[u];
  }
  for (; i < n; ++i) sum = sum + v[i];
  return sum;
}

__global__ __launch_bounds__(kReBlock) void re_chunks_kernel(const uint32_t* deg, const uint32_t* freq,
                                                             uint32_t v_num, uint64_t dsum,
                                                             uint64_t wsum_before, double* chunks,
                                                             dg_walk_queue* q) {
  __shared__ __align__(16) double s_term[kReChunk];
  __shared__ uint32_t s_zeros;
  if (threadIdx.x == 0) s_zeros = 0;
  __syncthreads();
  const uint64_t wsum = wsum_before + q->tokens;
  const uint32_t lo = blockIdx.x * kReChunk;
  const uint32_t n = v_num - lo < kReChunk ? v_num - lo : kReChunk;
  uint32_t zeros = 0;
#pragma unroll
  for (uint32_t k = 0; k < kReChunk / kReBlock; ++k) {
    const uint32_t j = k * kReBlock + threadIdx.x;
    if (j >= n) break;
    const uint32_t d = deg[lo + j];
    const uint32_t f = freq[lo + j];
    double t = 0.0;
    if (d == 0 || f == 0) {
      ++zeros;
    } else {
      const double pi = (double)d / (double)dsum;
      const double qi = (double)f / (double)wsum;
      t = pi * (dg_log(pi) - dg_log(qi));
    }
    s_term[j] = t;
  }
  if (zeros) atomicAdd(&s_zeros, zeros);
  __syncthreads();
  if (threadIdx.x == 0) {
    chunks[blockIdx.x] = ordered_sum(s_term, n, 0.0);
    if (s_zeros) atomicAdd(&q->zero_terms, s_zeros);
  }
}

// The chunk sums left to right in the same way, by one workgroup.
__global__ __launch_bounds__(kReBlock) void re_final_kernel(const double* chunks, uint32_t n_chunks,
                                                            dg_walk_queue* q) {
  __shared__ __align__(16) double s_part[kReChunk];
  double total = 0.0;
  for (uint32_t c0 = 0; c0 < n_chunks; c0 += kReChunk) {
    const uint32_t n = n_chunks - c0 < kReChunk ? n_chunks - c0 : kReChunk;
    for (uint32_t j = threadIdx.x; j < n; j += kReBlock) s_part[j] = chunks[c0 + j];
    __syncthreads();
    if (threadIdx.x == 0) total = ordered_sum(s_part, n, total);
    __syncthreads();
  }
  if (threadIdx.x == 0) q->re = total;
}

__global__ void offsets_shift_kernel(const uint64_t* src, uint64_t n, uint64_t add,
                                     uint64_t* dst) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    dst[i] = src[i] + add;
}

// Places of a bin that a vertex below v_num can have.
uint32_t bin_places(uint32_t v_num) { return ((v_num - 1) / (16u * kBins) + 1u) * 16u; }

int grid_for(dg_ctx* ctx, uint64_t n, int block) {
  uint64_t g = (n + block - 1) / block;
  uint64_t cap = (uint64_t)ctx->num_cus * 16;
  if (g > cap) g = cap;
  return g == 0 ? 1 : (int)g;
}

}  // namespace

// A planned round (see plan_round below).
struct dg_walk_plan {
  WalkArgs a;
  uint64_t blocks = 0;        // walk_kernel grid
  uint32_t parts = 0;         // pack_count_kernel grid
  uint32_t pack_block = 0;    // and its workgroup
  bool bins = false;          // visits counted by bins (else by atomics)
  uint64_t bin_words = 0, tail_words = 0;  // the packing's words at the end of the raw buffer
  uint32_t *bin_off = nullptr, *hot_part = nullptr;
  uint32_t bin_parts = 1;     // bin_count_kernel workgroups per bin
  uint32_t round = 0;
  uint32_t walker_num = 0;
  uint32_t length_limit = 0;
  uint64_t freq_total_before = 0;
};


void dg_walk_free(dg_ctx* ctx) {
  void* bufs[] = {ctx->d_freq,   ctx->d_tok_raw,  ctx->d_walk_off, ctx->d_walk_len,
                  ctx->d_tokens, ctx->d_offsets,  ctx->d_spill,    ctx->d_scan_tmp,
                  ctx->d_re_chunks, ctx->d_train_tokens, ctx->d_train_offsets,
                  ctx->d_term_table};
  for (void* p : bufs)
    if (p) hipFree(p);
  ctx->d_freq = nullptr;
  ctx->d_tok_raw = nullptr;
  ctx->d_walk_off = nullptr;
  ctx->d_walk_len = nullptr;
  ctx->d_tokens = nullptr;
  ctx->d_offsets = nullptr;
  ctx->d_spill = nullptr;
  ctx->d_scan_tmp = nullptr;
  ctx->d_re_chunks = nullptr;
  ctx->d_train_tokens = nullptr;
  ctx->d_train_offsets = nullptr;
  ctx->d_term_table = nullptr;
  delete ctx->wplan;
  ctx->wplan = nullptr;
  ctx->tok_raw_cap = ctx->walk_cap = ctx->walk_len_cap = ctx->tokens_cap = ctx->offsets_cap = 0;
  ctx->walks_spill = false;
  ctx->spill_cap = ctx->scan_tmp_cap = ctx->re_cap = 0;
  ctx->train_tokens_cap = ctx->train_offsets_cap = 0;
  ctx->train_walks = ctx->train_tokens = 0;
  ctx->cur_walks = ctx->cur_tokens = 0;
  ctx->freq_total = 0;
  ctx->prev_re = 0.0;
  ctx->rounds_done = 0;
}

int dg_scan_lengths(dg_ctx* ctx, const uint32_t* d_len, uint64_t n, uint64_t* d_off) {
  const uint64_t n_tiles = (n + kScanTile - 1) / kScanTile;
  DG_CHECK(dg_reserve(ctx, &ctx->d_scan_tmp, &ctx->scan_tmp_cap, n_tiles + 1));
  if (n_tiles > 0) {
    scan_tile_sums<<<(unsigned)n_tiles, kScanBlock, 0, ctx->stream>>>(d_len, n, ctx->d_scan_tmp);
    scan_tile_prefix<<<1, kScanBlock, 0, ctx->stream>>>(ctx->d_scan_tmp, n_tiles);
    scan_tile_apply<<<(unsigned)n_tiles, kScanBlock, 0, ctx->stream>>>(d_len, n, ctx->d_scan_tmp,
                                                                       n_tiles, d_off);
  } else {
    zero_first_kernel<<<1, 64, 0, ctx->stream>>>(d_off);
  }
  DG_HIP(ctx, hipGetLastError());
  return DG_OK;
}

extern "C" void dg_walk_params_default(dg_walk_params* p, uint32_t v_num) {
  if (!p) return;
  p->seed = 1;
  p->walkers_per_round = v_num;
  p->init_round = 5;
  p->min_length = 20;
  p->max_length = 0;
  p->mu = 0.999;
  p->delta = 0.001;
  p->max_rounds = 30;
  p->rounds_mode = DG_ROUNDS_REFERENCE;
  p->length_limit = 0;
  p->reserved = 0;
}

extern "C" int dg_walk_reset(dg_ctx* ctx) {
  if (!ctx) return DG_ERR_ARG;
  if (!ctx->d_row_ptr) return dg_fail(ctx, DG_ERR_STATE, "no graph loaded");
  DG_HIP(ctx, hipSetDevice(ctx->device));
  if (!ctx->d_freq) {
    DG_HIP(ctx, hipMalloc((void**)&ctx->d_freq, sizeof(uint32_t) * ctx->v_num));
  }
  if (!ctx->d_term_table) {
    DG_HIP(ctx, hipMalloc((void**)&ctx->d_term_table, sizeof(double) * kTabWords));
    term_table_kernel<<<(kTermWords + 255) / 256, 256, 0, ctx->stream>>>(
        ctx->d_term_table);
    DG_HIP(ctx, hipGetLastError());
  }
  fill_u32_kernel<<<grid_for(ctx, ctx->v_num, 256), 256, 0, ctx->stream>>>(ctx->d_freq, ctx->v_num,
                                                                           0u);
  DG_HIP(ctx, hipGetLastError());
  ctx->freq_total = 0;
  ctx->prev_re = 0.0;
  ctx->rounds_done = 0;
  return DG_OK;
}

// ---- one round, in three parts ---------------------------------------------
// plan: validation, launch shapes and buffers (may allocate); enqueue: kernels
// only, no host waits, so a stream capture can record them; collect: the
// round's statistics once the stream has finished.  round_guard_kernel empties
// a round that did not complete, which is then planned and walked again
// (dg_walk_round; the captured step does the same, pipeline.hip).

static int plan_round(dg_ctx* ctx, const dg_walk_params* p, uint32_t round,
                      uint32_t walker_begin, uint32_t walker_num, dg_walk_plan* pl) {
  if (!ctx->d_freq) DG_CHECK(dg_walk_reset(ctx));
  const uint32_t length_limit = p->length_limit ? p->length_limit : kDefaultLengthLimit;
  if (p->max_length != 0 && p->max_length > length_limit)
    return dg_fail(ctx, DG_ERR_ARG, "max_length %u exceeds length_limit %u", p->max_length,
                   length_limit);
  if (p->min_length + 2 > length_limit)
    return dg_fail(ctx, DG_ERR_ARG, "min_length %u needs length_limit > %u", p->min_length,
                   p->min_length + 1);
  // the buffers below may be reallocated (their contents dropped): the
  // previous round's corpus is given up here, so a round that fails leaves an
  // empty corpus behind, never one whose buffers no longer hold it
  ctx->cur_walks = 0;
  ctx->cur_tokens = 0;

  // persistent grid: every resident block slot on the device, fewer for small rounds
  if (ctx->walk_per_cu == 0) {
    int per_cu = 0;
    DG_HIP(ctx, hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, walk_kernel, kWalkBlock, 0));
    ctx->walk_per_cu = per_cu < 1 ? 1 : per_cu;
  }
  uint64_t blocks = (uint64_t)ctx->num_cus * ctx->walk_per_cu;
  const uint64_t need_blocks = ((uint64_t)walker_num + kWalkBlock - 1) / kWalkBlock;
  if (blocks > need_blocks) blocks = need_blocks ? need_blocks : 1;
  // spill space for the longest walk, (limit - kPathLds) vertices per lane
  // (1 GB for the default limit): only once a walk has needed it, or where they
  // will (the reference's walks end at 22 vertices): past min_length, or with a
  // threshold well below the reference's 0.999, at which walks run on
  // (walk.hpp:979-985; of 50,000 walks on a Chung-Lu graph 1 passes 24 vertices
  // at 0.97, 138 at 0.95 and 4,698 at 0.9)
  const uint32_t longest = p->max_length != 0 ? p->max_length : length_limit;
  if (p->min_length + 1 >= (uint32_t)kPathLds || p->mu <= 0.95) ctx->walks_spill = true;
  const uint32_t spill_per_slot =
      ctx->walks_spill && longest > (uint32_t)kPathLds ? longest - (uint32_t)kPathLds : 0;

  DG_CHECK(dg_reserve(ctx, &ctx->d_walk_off, &ctx->walk_cap, (size_t)walker_num));
  DG_CHECK(dg_reserve(ctx, &ctx->d_walk_len, &ctx->walk_len_cap, (size_t)walker_num + 1));
  DG_CHECK(dg_reserve(ctx, &ctx->d_offsets, &ctx->offsets_cap, (size_t)walker_num + 1));
  DG_CHECK(dg_reserve(ctx, &ctx->d_spill, &ctx->spill_cap,
                      (size_t)blocks * kWalkBlock * spill_per_slot));
  // raw buffer: one slot of kPathLds tokens per walk, then room for longer
  // walks, and at its end the packing's own words (its bins' offsets and the
  // hot counters' rows)
  const uint64_t slots_end = (uint64_t)walker_num * kPathLds;
  {
    // packing: a workgroup of 1,024 walks per CU (LDS: the hot counters and 96 KB of tokens)
    pl->pack_block = walker_num < (uint64_t)ctx->num_cus * kPackBig ? kPackSmall : kPackBig;
    const uint64_t n_tiles = std::max<uint64_t>(1, ((uint64_t)walker_num + pl->pack_block - 1) / pl->pack_block);
    pl->parts = (uint32_t)std::min<uint64_t>((uint64_t)ctx->num_cus, n_tiles);
    pl->bins = ctx->v_num <= kBinVertices;
    pl->bin_words = 0;
    if (pl->bins) {
      pl->bin_words = n_tiles * (kBins + 1);
      // two workgroups of 1,024 threads per CU, fewer where their LDS does not fit
      const size_t lds = sizeof(uint32_t) * bin_places(ctx->v_num);
      DG_HIP(ctx, hipFuncSetAttribute((const void*)bin_count_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)lds));
      const uint64_t fill = (uint64_t)ctx->num_cus * (lds <= 80 * 1024 ? 2 : 1) / kBins;
      pl->bin_parts = (uint32_t)std::max<uint64_t>(1, std::min(fill, n_tiles));
    }
    pl->tail_words = pl->bin_words + (uint64_t)pl->parts * ctx->n_hot;
    const size_t need = (size_t)(slots_end + walker_num / 8 + 4096 + pl->tail_words);
    DG_CHECK(dg_reserve(ctx, &ctx->d_tok_raw, &ctx->tok_raw_cap, need));
    pl->bin_off = ctx->d_tok_raw + (ctx->tok_raw_cap - pl->tail_words);
    pl->hot_part = pl->bin_off + pl->bin_words;
  }
  const uint32_t n_chunks = (ctx->v_num + kReChunk - 1) / kReChunk;
  DG_CHECK(dg_reserve(ctx, &ctx->d_re_chunks, &ctx->re_cap, (size_t)n_chunks));
  DG_CHECK(dg_reserve(ctx, &ctx->d_scan_tmp, &ctx->scan_tmp_cap,
                      (size_t)((walker_num + kScanTile - 1) / kScanTile) + 1));

  WalkArgs& a = pl->a;
  a.row_ptr = ctx->d_row_ptr;
  a.adj = ctx->d_adj;
  a.term_table = ctx->d_term_table;
  a.v_num = ctx->v_num;
  a.round = round;
  a.seed = p->seed;
  a.walker_begin = walker_begin;
  a.walker_num = walker_num;
  a.min_length = p->min_length;
  a.max_length = p->max_length;
  a.length_limit = length_limit;
  a.spill_per_slot = spill_per_slot;
  a.mu = p->mu;
  a.walk_off = ctx->d_walk_off;
  a.walk_len = ctx->d_walk_len;
  a.spill = ctx->d_spill;
  a.q = ctx->d_queue;
  a.shards = ctx->d_shards;
  a.slots_end = slots_end;
  a.tokens = ctx->d_tok_raw;
  a.tok_cap = ctx->tok_raw_cap - pl->tail_words;
  pl->blocks = blocks;
  pl->round = round;
  pl->walker_num = walker_num;
  pl->length_limit = length_limit;
  pl->freq_total_before = ctx->freq_total;
  return DG_OK;
}

// The walk itself: queue reset and the persistent launch.
static int enqueue_walk(dg_ctx* ctx, const dg_walk_plan& pl, bool timed) {
  queue_reset_kernel<<<1, 64, 0, ctx->stream>>>(ctx->d_queue, ctx->d_shards);
  size_t tk = 0;
  if (timed) DG_CHECK(dg_time_begin(ctx, "walk", &tk));
  walk_kernel<<<(unsigned)pl.blocks, kWalkBlock, 0, ctx->stream>>>(pl.a);
  DG_HIP(ctx, hipGetLastError());
  if (timed) DG_CHECK(dg_time_end(ctx, tk));
  // a round that did not complete becomes empty here, so the rest of it
  // changes nothing and it can run again
  round_guard_kernel<<<grid_for(ctx, pl.walker_num, 256), 256, 0, ctx->stream>>>(
      ctx->d_queue, ctx->d_walk_len, pl.walker_num, ctx->d_shards);
  DG_HIP(ctx, hipGetLastError());
  return DG_OK;
}

// Everything after the walk: packing in walk-id order with the round's visits
// added to the cumulative counts (a round that failed packs nothing), and the
// relative entropy.  Reads only device
// state, so it needs no host knowledge of the round's token count.
static int enqueue_tail(dg_ctx* ctx, const dg_walk_plan& pl, bool timed) {
  const uint32_t walker_num = pl.walker_num;
  size_t tp = 0;
  if (timed) DG_CHECK(dg_time_begin(ctx, "pack", &tp));
  DG_CHECK(dg_scan_lengths(ctx, ctx->d_walk_len, walker_num, ctx->d_offsets));
  const auto pack = [&](auto kern) {
    kern<<<pl.parts, pl.pack_block, 0, ctx->stream>>>(
        ctx->d_tok_raw, ctx->d_walk_off, ctx->d_walk_len, ctx->d_offsets, walker_num, ctx->d_tokens,
        ctx->d_hot_slot, ctx->n_hot, ctx->d_freq, pl.hot_part, pl.bin_off);
  };
  const bool big = pl.pack_block == (uint32_t)kPackBig;
  if (pl.bins) {
    big ? pack(pack_count_kernel<kPackBig, true>) : pack(pack_count_kernel<kPackSmall, true>);
    const uint64_t n_tiles = ((uint64_t)walker_num + pl.pack_block - 1) / pl.pack_block;
    const uint32_t places = bin_places(ctx->v_num);
    bin_count_kernel<<<dim3(kBins, pl.bin_parts), kBinBlock, sizeof(uint32_t) * places, ctx->stream>>>(
        ctx->d_tok_raw, pl.bin_off, n_tiles, pl.pack_block * kPathLds, ctx->v_num, places, ctx->d_freq);
  } else {
    big ? pack(pack_count_kernel<kPackBig, false>) : pack(pack_count_kernel<kPackSmall, false>);
  }
  if (ctx->n_hot) {
    const dim3 grid((ctx->n_hot + 63) / 64, (pl.parts + kHotRows - 1) / kHotRows);
    hot_reduce_kernel<<<grid, 64, 0, ctx->stream>>>(pl.hot_part, pl.parts, ctx->n_hot,
                                                    ctx->d_hot_id, ctx->d_freq);
  }
  DG_HIP(ctx, hipGetLastError());
  if (timed) DG_CHECK(dg_time_end(ctx, tp));

  // relative entropy against the cumulative visit counts
  const uint32_t n_chunks = (ctx->v_num + kReChunk - 1) / kReChunk;
  size_t tr = 0;
  if (timed) DG_CHECK(dg_time_begin(ctx, "re", &tr));
  re_chunks_kernel<<<n_chunks, kReBlock, 0, ctx->stream>>>(ctx->d_deg, ctx->d_freq, ctx->v_num, ctx->m,
                                                           pl.freq_total_before, ctx->d_re_chunks,
                                                           ctx->d_queue);
  re_final_kernel<<<1, kReBlock, 0, ctx->stream>>>(ctx->d_re_chunks, n_chunks, ctx->d_queue);
  DG_HIP(ctx, hipGetLastError());
  if (timed) DG_CHECK(dg_time_end(ctx, tr));
  return DG_OK;
}

// The round's statistics from the queue mirror (the stream has finished and
// h_queue holds the final queue).  Advances the host-side round state.
static int collect_round(dg_ctx* ctx, const dg_walk_plan& pl, double walk_ms, double total_ms,
                         dg_round_stats* out) {
  const dg_walk_queue& q = *ctx->h_queue;
  const uint64_t n_tok = q.tokens;
  ctx->freq_total = pl.freq_total_before + n_tok;
  ctx->cur_walks = pl.walker_num;
  ctx->cur_tokens = n_tok;
  const double re = q.re;
  const double delta = ctx->rounds_done == 0 ? re : re - ctx->prev_re;
  ctx->prev_re = re;
  ctx->rounds_done += 1;
  if (out) {
    out->round = pl.round;
    out->walkers = pl.walker_num;
    out->tokens = n_tok;
    out->steps = n_tok - pl.walker_num;
    out->re = re;
    out->delta_re = delta;
    out->walk_ms = walk_ms;
    out->total_ms = total_ms;
    out->max_walk_len = q.max_len;
    out->draws = q.draws;
    out->moves = q.moves;
    out->stop = 0;
  }
  if (q.zero_terms != 0)
    return dg_fail(ctx, DG_ERR_RE_UNDEFINED,
                   "relative entropy undefined: %u vertices with degree 0 or no visits",
                   q.zero_terms);
  return DG_OK;
}

static int read_queue(dg_ctx* ctx) {
  DG_HIP(ctx, hipMemcpyAsync(ctx->h_queue, ctx->d_queue, sizeof(dg_walk_queue),
                             hipMemcpyDeviceToHost, ctx->stream));
  DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return DG_OK;
}

// What the flags of a round that did not complete ask for: more token space,
// spill space, or an error.  *retry: the round is to be walked again.
static int check_flags(dg_ctx* ctx, const dg_walk_plan& pl, bool* retry) {
  const dg_walk_queue& q = *ctx->h_queue;
  *retry = false;
  if (q.flags & DG_QFLAG_LENGTH_LIMIT)
    return dg_fail(ctx, DG_ERR_WALK_TOO_LONG,
                   "round %u: a walk reached the length limit %u (raise length_limit)", pl.round,
                   pl.length_limit);
  if (q.flags & DG_QFLAG_NO_SPILL) {
    ctx->walks_spill = true;  // the next plan reserves it
    *retry = true;
  }
  if (q.flags & DG_QFLAG_TOKEN_OVERFLOW) {
    const size_t need = (size_t)(pl.a.slots_end + q.cursor + q.cursor / 8 + 1024 + pl.tail_words);
    DG_CHECK(dg_reserve(ctx, &ctx->d_tok_raw, &ctx->tok_raw_cap, need));
    *retry = true;
  }
  return DG_OK;
}

// The packed corpus can hold every token the raw buffer can, whatever share of
// it the packing's words take: a round of fewer walks leaves them less, and a
// buffer sized for the tokens alone was allocated anew in a job's second round
// (0.3 to 0.4 ms).
static int reserve_tokens(dg_ctx* ctx) {
  return dg_reserve(ctx, &ctx->d_tokens, &ctx->tokens_cap, ctx->tok_raw_cap);
}

static int walk_round_impl(dg_ctx* ctx, const dg_walk_params* p, uint32_t round,
                           uint32_t walker_begin, uint32_t walker_num, dg_round_stats* out) {
  dg_walk_plan pl;
  // at most one repeat for spill space and two for token space
  for (int attempt = 0; attempt < 4; ++attempt) {
    DG_CHECK(plan_round(ctx, p, round, walker_begin, walker_num, &pl));
    // where the packed corpus has to be allocated, a round that needs more room
    // is known before that (one host wait more, once per size)
    const bool fits = ctx->d_tokens && ctx->tokens_cap >= ctx->tok_raw_cap;
    DG_CHECK(enqueue_walk(ctx, pl, true));
    bool retry = false;
    int rc = DG_OK;
    if (!fits) {
      DG_CHECK(read_queue(ctx));
      rc = check_flags(ctx, pl, &retry);
    }
    if (rc == DG_OK && !retry) {
      DG_CHECK(reserve_tokens(ctx));
      DG_CHECK(enqueue_tail(ctx, pl, true));
      DG_CHECK(read_queue(ctx));
      rc = check_flags(ctx, pl, &retry);
    }
    if (rc != DG_OK || retry) {
      DG_CHECK(dg_time_resolve(ctx));
      if (rc != DG_OK) return rc;
      continue;
    }
    double walk_ms = 0.0, total_ms = 0.0;
    for (auto& pe : ctx->pending) {
      float ms = 0.f;
      DG_HIP(ctx, hipEventElapsedTime(&ms, pe.start, pe.stop));
      if (pe.name == "walk") walk_ms = ms;
      total_ms += ms;
    }
    DG_CHECK(dg_time_resolve(ctx));
    return collect_round(ctx, pl, walk_ms, total_ms, out);
  }
  return dg_fail(ctx, DG_ERR_STATE, "token buffer sizing did not converge");
}

extern "C" int dg_walk_round(dg_ctx* ctx, const dg_walk_params* p, uint32_t round,
                             uint32_t walker_begin, uint32_t walker_num, dg_round_stats* out) {
  if (!ctx || !p) return DG_ERR_ARG;
  if (!ctx->d_row_ptr) return dg_fail(ctx, DG_ERR_STATE, "no graph loaded");
  if (!(p->mu > 0.0)) return dg_fail(ctx, DG_ERR_ARG, "mu must be positive");
  DG_HIP(ctx, hipSetDevice(ctx->device));
  return walk_round_impl(ctx, p, round, walker_begin, walker_num, out);
}

// ---- the round as the captured pipeline step runs it -----------------------

int dg_walk_graph_plan(dg_ctx* ctx, const dg_walk_params* p, uint32_t round,
                       uint32_t walker_begin, uint32_t walker_num, uint64_t* tok_bound,
                       uint64_t* slot_tokens, uint64_t* overflow_tokens) {
  if (!ctx->d_row_ptr) return dg_fail(ctx, DG_ERR_STATE, "no graph loaded");
  if (!(p->mu > 0.0)) return dg_fail(ctx, DG_ERR_ARG, "mu must be positive");
  if (!ctx->wplan) ctx->wplan = new dg_walk_plan();
  DG_CHECK(plan_round(ctx, p, round, walker_begin, walker_num, ctx->wplan));
  DG_CHECK(reserve_tokens(ctx));
  *tok_bound = ctx->wplan->a.tok_cap;
  *slot_tokens = kPathLds;
  *overflow_tokens = ctx->wplan->a.tok_cap - ctx->wplan->a.slots_end;
  return DG_OK;
}

int dg_walk_graph_enqueue(dg_ctx* ctx, bool timed) {
  const dg_walk_plan& pl = *ctx->wplan;
  DG_CHECK(enqueue_walk(ctx, pl, timed));
  return enqueue_tail(ctx, pl, timed);
}

int dg_walk_graph_collect(dg_ctx* ctx, double walk_ms, double total_ms, dg_round_stats* out,
                          bool* retry) {
  DG_CHECK(read_queue(ctx));
  DG_CHECK(check_flags(ctx, *ctx->wplan, retry));
  if (*retry) return DG_OK;
  return collect_round(ctx, *ctx->wplan, walk_ms, total_ms, out);
}

extern "C" int dg_corpus_append(dg_ctx* ctx) {
  if (!ctx) return DG_ERR_ARG;
  DG_HIP(ctx, hipSetDevice(ctx->device));
  const uint64_t nw = ctx->cur_walks, nt = ctx->cur_tokens;
  DG_CHECK(dg_grow_keep(ctx, &ctx->d_train_tokens, &ctx->train_tokens_cap,
                        (size_t)(ctx->train_tokens + nt), (size_t)ctx->train_tokens));
  DG_CHECK(dg_grow_keep(ctx, &ctx->d_train_offsets, &ctx->train_offsets_cap,
                        (size_t)(ctx->train_walks + nw + 1), (size_t)(ctx->train_walks + 1)));
  if (ctx->train_walks == 0)
    DG_HIP(ctx, hipMemsetAsync(ctx->d_train_offsets, 0, sizeof(uint64_t), ctx->stream));
  if (nt)
    DG_HIP(ctx, hipMemcpyAsync(ctx->d_train_tokens + ctx->train_tokens, ctx->d_tokens,
                               sizeof(uint32_t) * nt, hipMemcpyDeviceToDevice, ctx->stream));
  if (nw)
    offsets_shift_kernel<<<grid_for(ctx, nw, 256), 256, 0, ctx->stream>>>(
        ctx->d_offsets + 1, nw, ctx->train_tokens, ctx->d_train_offsets + ctx->train_walks + 1);
  DG_HIP(ctx, hipGetLastError());
  ctx->train_walks += nw;
  ctx->train_tokens += nt;
  return DG_OK;
}

extern "C" int dg_train_corpus_info(dg_ctx* ctx, uint64_t* n_walks, uint64_t* n_tokens) {
  if (!ctx) return DG_ERR_ARG;
  if (n_walks) *n_walks = ctx->train_walks;
  if (n_tokens) *n_tokens = ctx->train_tokens;
  return DG_OK;
}

extern "C" int dg_train_corpus_clear(dg_ctx* ctx) {
  if (!ctx) return DG_ERR_ARG;
  ctx->train_walks = 0;
  ctx->train_tokens = 0;
  return DG_OK;
}

extern "C" int dg_walk_run(dg_ctx* ctx, const dg_walk_params* p, dg_round_stats* per_round,
                           uint32_t max_stats, uint32_t* n_rounds, int keep_corpus) {
  if (!ctx || !p) return DG_ERR_ARG;
  if (!ctx->d_row_ptr) return dg_fail(ctx, DG_ERR_STATE, "no graph loaded");
  if (p->walkers_per_round == 0 || p->init_round == 0)
    return dg_fail(ctx, DG_ERR_ARG, "walkers_per_round and init_round must be positive");
  DG_HIP(ctx, hipSetDevice(ctx->device));
  DG_CHECK(dg_walk_reset(ctx));
  uint32_t iter = 1;
  uint32_t done = 0;
  const uint32_t max_rounds = p->max_rounds ? p->max_rounds : 30;
  while (true) {
    // walk.hpp:614 (round 1: walker_num * init_round), :764-775 (later rounds)
    const uint64_t nw64 = (iter == 1) ? (uint64_t)p->walkers_per_round * p->init_round
                                      : (uint64_t)p->walkers_per_round;
    if (nw64 > 0xffffffffull) return dg_fail(ctx, DG_ERR_ARG, "too many walkers per round");
    dg_round_stats st;
    DG_CHECK(walk_round_impl(ctx, p, iter, 0, (uint32_t)nw64, &st));
    if (keep_corpus) DG_CHECK(dg_corpus_append(ctx));
    // walk.hpp:735-749: stop after round max_rounds; optionally on |delta RE| <= delta
    bool stop = (iter + 1 > max_rounds);
    if (p->rounds_mode == DG_ROUNDS_CONVERGE && (st.delta_re < 0 ? -st.delta_re : st.delta_re) <= p->delta)
      stop = true;
    st.stop = stop ? 1u : 0u;
    if (per_round && done < max_stats) per_round[done] = st;
    ++done;
    ++iter;
    if (stop) break;
  }
  if (n_rounds) *n_rounds = done;
  return DG_OK;
}

extern "C" int dg_corpus_info(dg_ctx* ctx, uint64_t* n_walks, uint64_t* n_tokens) {
  if (!ctx) return DG_ERR_ARG;
  if (n_walks) *n_walks = ctx->cur_walks;
  if (n_tokens) *n_tokens = ctx->cur_tokens;
  return DG_OK;
}

extern "C" int dg_corpus_copy(dg_ctx* ctx, uint32_t* tokens, uint64_t* offsets) {
  if (!ctx) return DG_ERR_ARG;
  DG_HIP(ctx, hipSetDevice(ctx->device));
  DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (tokens && ctx->cur_tokens)
    DG_CHECK(dg_copy_to_host(ctx, tokens, ctx->d_tokens, sizeof(uint32_t) * ctx->cur_tokens));
  if (offsets && ctx->d_offsets)
    DG_CHECK(dg_copy_to_host(ctx, offsets, ctx->d_offsets, sizeof(uint64_t) * (ctx->cur_walks + 1)));
  return DG_OK;
}

extern "C" int dg_vertex_freq(dg_ctx* ctx, uint32_t* freq) {
  if (!ctx || !freq) return DG_ERR_ARG;
  if (!ctx->d_freq) return dg_fail(ctx, DG_ERR_STATE, "no walk has run");
  DG_HIP(ctx, hipSetDevice(ctx->device));
  DG_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return dg_copy_to_host(ctx, freq, ctx->d_freq, sizeof(uint32_t) * ctx->v_num);
}

// Walk text file of include/path.hpp:67-119.  Formatting is done into a large
// buffer with a hand-rolled decimal conversion; the bytes equal fprintf's.
extern "C" int dg_corpus_write_text(dg_ctx* ctx, const char* path, uint32_t threads) {
  if (!ctx || !path) return DG_ERR_ARG;
  if (threads == 0) threads = 1;
  std::vector<uint32_t> tok(ctx->cur_tokens);
  std::vector<uint64_t> off(ctx->cur_walks + 1);
  DG_CHECK(dg_corpus_copy(ctx, tok.data(), off.data()));
  FILE* f = fopen(path, "w");
  if (!f) return dg_fail(ctx, DG_ERR_IO, "cannot open %s for writing", path);
  std::vector<char> buf;
  buf.reserve(1 << 22);
  auto flush = [&]() -> bool {
    bool ok = buf.empty() || fwrite(buf.data(), 1, buf.size(), f) == buf.size();
    buf.clear();
    return ok;
  };
  bool ok = true;
  for (uint32_t t = 0; t < threads && ok; ++t) {
    for (uint64_t w = t; w < ctx->cur_walks && ok; w += threads) {
      for (uint64_t i = off[w]; i < off[w + 1]; ++i) {
        char digits[12];
        int nd = 0;
        uint32_t v = tok[i];
        do {
          digits[nd++] = (char)('0' + v % 10);
          v /= 10;
        } while (v);
        buf.push_back(' ');
        while (nd) buf.push_back(digits[--nd]);
      }
      buf.push_back('\n');
      if (buf.size() > (1u << 22) - 4096) ok = flush();
    }
  }
  ok = flush() && ok;
  if (fclose(f) != 0) ok = false;
  return ok ? DG_OK : dg_fail(ctx, DG_ERR_IO, "write to %s failed", path);
}
