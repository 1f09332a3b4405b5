// perft.hip -- batched perft on gfx950.
//
// Replaces perft_gpu (src/zetaperft.cl:801-1477), which walks ONE root with
// one 64-lane work-group, and its host driver (src/search.c:225-271,
// src/clrun.c:979-1147).  Design: a level-synchronous frontier over all roots
// of the batch (SoA in HBM); the last level is never materialised: its moves
// are applied to their parents and the children's legal moves counted (bulk
// counting at depth-1) into the roots' u64 counters.  Every leaf-level lane
// does the same branch-free set-wise counting, so the uneven subtree sizes of a
// batch cost no SIMD divergence.  Two drivers:
//   the chain (fast_perft) queues all levels without waiting for their sizes,
//   and counts positions that several move orders reach once;
//   the chunked one (process) reads each level's size, splits levels that
//   exceed the frontier budget into chunks (depth-first over chunks), and works
//   in fixed buffers where the call may not allocate.  Its levels:
//     count -> exclusive scan -> expand writes (parent, move) pairs of level
//     L+1 -> apply materialises level L+1 and counts its moves.
#include <string.h>

#include <type_traits>
#include <vector>

#include "chess.h"
#include "runtime.h"
#include "wave.h"

using namespace zc;

namespace {

struct Front {  // a frontier level, structure of arrays (coalesced per field)
  u64 *b0, *b1, *b2, *b3, *cr;
  u32 *meta;  // root index << 1 | side to move
  u32 *cnt;   // number of legal moves
};

__device__ __forceinline__ Pos load_pos(const Front &f, size_t i) {
  Pos p;
  p.b0 = f.b0[i];
  p.b1 = f.b1[i];
  p.b2 = f.b2[i];
  p.b3 = f.b3[i];
  p.cr = f.cr[i];
  p.stm = f.meta[i] & 1u;
  return p;
}

__device__ __forceinline__ void store_pos(const Front &f, size_t i, const Pos &p, u32 root) {
  f.b0[i] = p.b0;
  f.b1[i] = p.b1;
  f.b2[i] = p.b2;
  f.b3[i] = p.b3;
  f.cr[i] = p.cr;
  f.meta[i] = (root << 1) | p.stm;
}

constexpr int TPB = 256;

__global__ __launch_bounds__(TPB) void k_roots(const u64 *__restrict__ in, int n, Front f) {
  const int i = blockIdx.x * TPB + threadIdx.x;
  if (i >= n) return;
  const u64 *q = in + (size_t)i * 8;  // zeta_pos = 7 x u64 + stm + pad
  Pos p;
  p.b0 = q[0];
  p.b1 = q[1];
  p.b2 = q[2];
  p.b3 = q[3];
  p.cr = q[4];
  p.stm = (u32)(q[7] & 1u);
  store_pos(f, i, p, (u32)i);
  Legal L;
  analyse(p, L);
  f.cnt[i] = (u32)count_legal(p, L, false);
}

// ---- exclusive scan of u32 counts into u64 offsets (off[n] = total)
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = TPB * SCAN_ITEMS;

__device__ __forceinline__ u64 block_exscan(u64 v, u64 *lds, u64 &total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  u64 x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    u64 y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) lds[w] = x;
  __syncthreads();
  u64 wo = 0;
  for (int k = 0; k < w; k++) wo += lds[k];
  total = lds[0] + lds[1] + lds[2] + lds[3];
  __syncthreads();
  return wo + x - v;
}

__global__ __launch_bounds__(TPB) void k_scan_reduce(const u32 *__restrict__ cnt, size_t n, u64 *bsum) {
  __shared__ u64 lds[4];
  const size_t base = (size_t)blockIdx.x * SCAN_TILE + (size_t)threadIdx.x * SCAN_ITEMS;
  u64 s = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; k++)
    if (base + k < n) s += cnt[base + k];
  u64 tot;
  block_exscan(s, lds, tot);
  if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

__global__ __launch_bounds__(TPB) void k_scan_top(u64 *bsum, size_t nb, u64 *total_out) {
  __shared__ u64 lds[4];
  u64 carry = 0;
  for (size_t t0 = 0; t0 < nb; t0 += TPB) {
    const size_t i = t0 + threadIdx.x;
    u64 v = i < nb ? bsum[i] : 0;
    u64 tot;
    u64 ex = block_exscan(v, lds, tot);
    if (i < nb) bsum[i] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0) *total_out = carry;
}

__global__ __launch_bounds__(TPB) void k_scan_down(const u32 *__restrict__ cnt, size_t n, const u64 *bsum,
                                                   u64 *off) {
  __shared__ u64 lds[4];
  const size_t base = (size_t)blockIdx.x * SCAN_TILE + (size_t)threadIdx.x * SCAN_ITEMS;
  u32 v[SCAN_ITEMS];
  u64 s = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; k++) {
    v[k] = base + k < n ? cnt[base + k] : 0u;
    s += v[k];
  }
  u64 tot;
  u64 ex = block_exscan(s, lds, tot) + bsum[blockIdx.x];
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; k++) {
    if (base + k < n) off[base + k] = ex;
    ex += v[k];
  }
  // the thread covering element n-1 also writes the total into off[n]
  if (base < n && base + SCAN_ITEMS >= n) off[n] = ex;
}

// ---- expand: (parent, move) pairs of every legal move, at the scanned offsets.
// A block's parents own one contiguous range of pairs.  Each lane enumerates
// its parent's moves into LDS (move code + the lane that owns the parent),
// then the block writes the range out with coalesced 8-byte stores: stored
// straight from the enumeration loop, the pairs of 64 lanes land on 64
// different cache lines per store instruction.  Moves beyond the LDS capacity
// (a block whose parents have more than XCAP moves in all) are stored directly.
constexpr int XTPB = 128;
constexpr int XCAP = 4096;  // 16 KiB of codes + 4 KiB of lane indices per block
__global__ __launch_bounds__(XTPB) void k_expand(Front f, size_t i0, size_t i1, const u64 *__restrict__ off,
                                                 u64 base, u64 *__restrict__ pm, const u64 *__restrict__ gtotal,
                                                 u64 gcap) {
  __shared__ u32 lcode[XCAP];
  __shared__ u8 llane[XCAP];
  // launched before the host knows the level's pair total: the whole grid
  // leaves when the total does not fit the pair buffer (the host relaunches)
  if (gtotal && *gtotal > gcap) return;
  const size_t bi0 = i0 + (size_t)blockIdx.x * XTPB;
  const size_t bi1 = bi0 + XTPB < i1 ? bi0 + XTPB : i1;
  const u64 blo = off[bi0], total = off[bi1] - blo;
  u64 *const out = pm + (blo - base);
  const size_t i = bi0 + threadIdx.x;
  if (i < bi1) {
    const Pos p = load_pos(f, i);
    Legal L;
    analyse(p, L);
    u64 o = off[i] - blo;
    const u64 parent = (u64)i << 32;
    const u8 lane = (u8)threadIdx.x;
    for_each_legal(p, L, [&](u32 code) {
      if (o < (u64)XCAP) {
        lcode[o] = code;
        llane[o] = lane;
      } else {
        out[o] = parent | code;
      }
      o++;
    });
  }
  __syncthreads();
  const u32 n = total < (u64)XCAP ? (u32)total : (u32)XCAP;
  const u32 last = (u32)(bi1 - bi0) - 1;  // every slot below n has an owner; the clamp only bounds the index
  for (u32 j = threadIdx.x; j < n; j += XTPB) {
    const u32 l = llane[j] < last ? llane[j] : last;
    out[j] = ((u64)(bi0 + l) << 32) | lcode[j];
  }
}

// ---- chunk cuts of an oversized level: bucket b holds the parents whose pairs
// start in [b * bp, (b + 1) * bp), so a chunk has at most bp + 218 pairs (the
// most legal moves of a position).  cut_idx[b] = first parent of bucket b
// (relative to the level range), cut_off[b] = its offset; buckets past the
// last parent get (n, total).  Every b in [0, nb] is written exactly once.
__global__ __launch_bounds__(TPB) void k_cuts(const u64 *__restrict__ off, size_t n, u64 bp, u64 nb,
                                              u64 *__restrict__ cut_idx, u64 *__restrict__ cut_off) {
  const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
  if (i >= n) return;
  const u64 b = off[i] / bp;
  const u64 first = i ? off[i - 1] / bp + 1 : 0;
  for (u64 j = first; j <= b && j <= nb; j++) {
    cut_idx[j] = i;
    cut_off[j] = off[i];
  }
  if (i + 1 == n)
    for (u64 j = b + 1; j <= nb; j++) {
      cut_idx[j] = n;
      cut_off[j] = off[n];
    }
}

// ---- apply: materialise the next level and count its moves
__global__ __launch_bounds__(TPB) void k_apply(Front f, const u64 *__restrict__ pm,
                                               size_t m, Front g) {
  const size_t j = (size_t)blockIdx.x * TPB + threadIdx.x;
  if (j >= m) return;
  const u64 e = pm[j];
  const u32 pi = (u32)(e >> 32);
  const Pos p = load_pos(f, pi);
  const Pos c = apply_v(p, (u32)e);
  store_pos(g, j, c, f.meta[pi] >> 1);
  Legal L;
  analyse(c, L);
  g.cnt[j] = (u32)count_legal(c, L, false);
}

// sum over the wave (all lanes active); a wave's per-root share is at most
// 64 x 218 legal moves, so 32-bit DPP sums suffice
__device__ __forceinline__ u64 wave_sum(u32 v) {
  return (u64)(u32)__builtin_amdgcn_readlane(zw::wave_scan_add((int)v), 63);
}

// ---- leaf level: apply + count, accumulate per root
__global__ __launch_bounds__(TPB) void k_leaf(Front f, const u64 *__restrict__ pm,
                                              size_t m, u64 *__restrict__ rootcnt, int nobulk) {
  const size_t j = (size_t)blockIdx.x * TPB + threadIdx.x;
  bool active = j < m;
  u64 v = 0;
  u32 root = 0;
  if (active) {
    const u64 e = pm[j];
    const u32 pi = (u32)(e >> 32);
    const Pos p = load_pos(f, pi);
    const Pos c = apply_v(p, (u32)e);
    Legal L;
    analyse(c, L);
    if (nobulk) {
      // the reference visits every leaf: it generates the leaf's (quiescence)
      // moves and counts one node (src/zetaperft.cl:1316-1326)
      const int n = count_legal(c, L, true);
      v = 1ULL + (u64)(n > 4096);
    } else {
      v = (u64)count_legal(c, L, false);
    }
    root = f.meta[pi] >> 1;
  }
  // wavefront-aggregated accumulation: one atomic per distinct root in the wave
  const int lane = threadIdx.x & 63;
  u64 pending = __ballot(active);
  while (pending) {
    const int leader = __builtin_ctzll(pending);
    const u32 rl = __shfl(root, leader, 64);
    const bool mine = active && root == rl;
    const u64 mask = __ballot(mine);
    const u64 s = wave_sum(mine ? (u32)v : 0u);
    if (lane == leader) atomicAdd((unsigned long long *)&rootcnt[rl], (unsigned long long)s);
    pending &= ~mask;
    active = active && !mine;
  }
}

// ========================================================== the chain
// A call's levels in one chain of launches without a wait between them: the
// host sizes the buffers by what earlier calls needed, every kernel reads its
// level's count from device memory, and a level that did not fit reports its
// size at the end (the chain then runs again with room for it, or, past the
// frontier budget, the chunked driver takes the call).
//   wide    one wavefront a parent, lane = square, then lane = move: few
//           positions in few microseconds
//   spread  one parent a lane, the moves of 128 parents meet in LDS and are
//           made one a lane: many positions
// Levels 3 and deeper merge transpositions: positions of a root reached by
// several move orders become one node that carries their number (k_merge).
// Measured against the chunked driver (host waits for every level, three scan
// launches each): one position at depth 4 146 -> 54 us, at depth 6 (119 M and
// 8 G leaves) 2.05 -> 0.39 and 5.8 -> 0.52 ms.  Of the first, 46 us are its four
// kernels (7, 10, 26 and 4), the rest launches and the host's one wait; the
// others are bound by the leaves' VALU issue.
struct Level {
  u64 *b0, *b1, *b2, *b3, *cr;
  u64 *wt;    // paths from the root that the node stands for
  u32 *meta;  // root index << 1 | side to move
  u32 *mv;    // the move that led to it, where k_spread's list in LDS was full
  u32 *par;   // its parent's index in the level above
  u64 *count; // nodes wanted so far (those past the capacity are not stored)
  u64 cap;
};

__device__ __forceinline__ Pos level_pos(const Level &f, size_t i) {
  Pos p;
  p.b0 = f.b0[i];
  p.b1 = f.b1[i];
  p.b2 = f.b2[i];
  p.b3 = f.b3[i];
  p.cr = f.cr[i];
  p.stm = f.meta[i] & 1u;
  return p;
}
__device__ __forceinline__ void level_store(const Level &f, size_t i, const Pos &c, u32 root, u32 par, u64 wt) {
  f.b0[i] = c.b0;
  f.b1[i] = c.b1;
  f.b2[i] = c.b2;
  f.b3[i] = c.b3;
  f.cr[i] = c.cr;
  f.meta[i] = (root << 1) | c.stm;
  f.par[i] = par;
  f.wt[i] = wt;
}
// (a level that did not fit counts as empty: nothing below it is worked on)
__device__ __forceinline__ u64 level_size(const Level &f) {
  const u64 n = *f.count;
  return n <= f.cap ? n : 0;
}
__device__ __forceinline__ Pos root_pos(const u64 *in, size_t i) {
  const u64 *q = in + i * 8;  // zeta_pos = 7 x u64 + stm + pad
  Pos p;
  p.b0 = q[0];
  p.b1 = q[1];
  p.b2 = q[2];
  p.b3 = q[3];
  p.cr = q[4];
  p.stm = (u32)(q[7] & 1u);
  return p;
}

// ---- depth 1: the roots' own move counts
__global__ __launch_bounds__(64) void k_count_roots(const u64 *__restrict__ in, int n, u64 *__restrict__ counts) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  if (i >= n) return;
  const Pos p = root_pos(in, i);
  Legal L;
  analyse(p, L);
  counts[i] = (u64)count_legal(p, L, false);
}

// ---- wide: the legal moves of one position, spread over a wavefront: lane
// takes move number `lane` + 64 k of list[0 .. n).  Boards that the per-square
// form takes otherwise than the counts do (lanes_serve) are enumerated by one
// lane.
__device__ __forceinline__ int wide_moves(const Pos &p, int lane, u32 *list) {
  Node0 B;
  node_basics(p, B);
  if (!lanes_serve(p, B)) {
    int n = 0;
    if (lane == 0) {
      Legal L;
      analyse(p, L);
      for_each_legal(p, L, [&](u32 code) { list[n++] = code; });
    }
    return __shfl(n, 0, 64);
  }
  const u64 A = __ballot(attacked_nk(B, lane));
  u64 t = (B.own >> lane) & 1 ? lane_targets(p, B, A, lane, false) : 0;
  const int incl = zw::wave_scan_add(popc(t));
  int k = incl - popc(t);
  while (t) {
    list[k++] = make_code(p, lane, lsb(t));
    t &= t - 1;
  }
  return __builtin_amdgcn_readlane(incl, 63);
}

// most moves of a position with one king to move, on any board: a piece has at
// most 27 (the king 10), a square can be reached from at most 8 lines, 8
// knights, a king and 2 more pawns: with k pieces no more than
// min(27 k + 10, 19 (64 - k)), below 740 for every k
constexpr int MAXMOVES = 768;
constexpr int WIDE_TPB = 512;

// level 0 (in != null) or f -> g; also clears the counts of the roots
__global__ __launch_bounds__(WIDE_TPB) void k_wide(const u64 *__restrict__ in, int nroots, Level f, Level g,
                                                   u64 *__restrict__ counts) {
  __shared__ u32 list[WIDE_TPB / 64][MAXMOVES];
  __shared__ u32 num[WIDE_TPB / 64];
  __shared__ u64 lbase;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const u64 n = in ? (u64)nroots : level_size(f);
  for (u64 i0 = (u64)blockIdx.x * (WIDE_TPB / 64); i0 < n; i0 += (u64)gridDim.x * (WIDE_TPB / 64)) {
    const u64 i = i0 + w;
    Pos p = {};
    u32 root = 0;
    u64 wt = 1;
    int m = 0;
    if (i < n) {
      p = in ? root_pos(in, i) : level_pos(f, i);
      root = in ? (u32)i : f.meta[i] >> 1;
      if (!in) wt = f.wt[i];
      if (in && lane == 0) counts[i] = 0;
      m = wide_moves(p, lane, list[w]);
    }
    if (lane == 0) num[w] = (u32)m;
    __syncthreads();
    // one atomic a block: they are a chain of 10 ns each
    u32 before = 0, total = 0;
#pragma unroll
    for (int k = 0; k < WIDE_TPB / 64; k++) {
      before += k < w ? num[k] : 0u;
      total += num[k];
    }
    if (threadIdx.x == 0) lbase = total ? atomicAdd((unsigned long long *)g.count, (unsigned long long)total) : 0;
    __syncthreads();
    const u64 base = lbase + before;
    for (int k = lane; k < m; k += 64)
      if (base + k < g.cap) level_store(g, base + k, apply_count(p, list[w][k]), root, (u32)i, wt);
    __syncthreads();
  }
}

// the last level below few parents: each lane makes a child and counts its
// moves (nobulk: generates them and counts the child itself).
// Bound: latency of one wavefront's work on a parent: 1000 parents are 128 blocks
// on 256 CUs, and 0.6 of their cycles wait (26 us).
__global__ __launch_bounds__(WIDE_TPB) void k_wide_leaf(const u64 *__restrict__ in, int nroots, Level f,
                                                        u64 *__restrict__ counts, int nobulk) {
  __shared__ u32 list[WIDE_TPB / 64][MAXMOVES];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const u64 n = in ? (u64)nroots : level_size(f);
  const u64 step = (u64)gridDim.x * (WIDE_TPB / 64);
  for (u64 i = (u64)blockIdx.x * (WIDE_TPB / 64) + w; i < n; i += step) {
    const Pos p = in ? root_pos(in, i) : level_pos(f, i);
    const int m = wide_moves(p, lane, list[w]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    u32 v = 0;
    for (int k = lane; k < m; k += 64) {
      const Pos c = apply_v(p, list[w][k]);
      Legal L;
      analyse(c, L);
      v += nobulk ? 1u + (u32)(count_legal(c, L, true) > 4096) : (u32)count_legal(c, L, false);
    }
    const u64 s = (u64)(u32)__builtin_amdgcn_readlane(zw::wave_scan_add((int)v), 63);
    if (lane == 0) {
      if (in) counts[i] = s;
      else if (s) atomicAdd((unsigned long long *)&counts[f.meta[i] >> 1], (unsigned long long)(s * f.wt[i]));
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

// ---- spread: 128 parents a block, one a lane; their moves meet in LDS (those
// beyond its list wait in the output itself) and are made one a lane, so that
// the stores are coalesced.  PAIRS: the moves are not made but written as
// (parent << 32 | move) for the leaf kernel.  Takes the parents [i0, i1).
// Bound: VALU issue of the move loops, where a wavefront runs as many steps as
// its busiest lane has of each kind (3.97 M parents, 128.9 M pairs: 0.57 ms; the
// stores alone would take 0.22).
template <bool PAIRS>
__global__ __launch_bounds__(XTPB) void k_spread(Level f, u64 i0, u64 i1, Level g, u64 *__restrict__ pm) {
  __shared__ u32 lcode[XCAP];
  __shared__ u8 llane[XCAP];
  __shared__ u64 lb0[XTPB], lb1[XTPB], lb2[XTPB], lb3[XTPB], lcr[XTPB], lwt[XTPB];
  __shared__ u32 lmeta[XTPB];
  __shared__ u32 wsum[XTPB / 64];
  __shared__ u64 lbase;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const u64 size = level_size(f), n = size < i1 ? size : i1;
  for (u64 c0 = i0 + (u64)blockIdx.x * XTPB; c0 < n; c0 += (u64)gridDim.x * XTPB) {
    const u64 i = c0 + tid;
    Pos p;
    Legal L;
    u32 cnt = 0;
    if (i < n) {
      p = level_pos(f, i);
      if (!PAIRS) {
        lb0[tid] = p.b0;
        lb1[tid] = p.b1;
        lb2[tid] = p.b2;
        lb3[tid] = p.b3;
        lcr[tid] = p.cr;
        lwt[tid] = f.wt[i];
        lmeta[tid] = f.meta[i];
      }
      analyse(p, L);
      cnt = (u32)count_emitted(p, L);
    }
    const u32 incl = (u32)zw::wave_scan_add((int)cnt);
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    const u32 total = wsum[0] + wsum[1];
    if (tid == 0) lbase = atomicAdd((unsigned long long *)g.count, (unsigned long long)total);
    __syncthreads();
    const u64 base = lbase;
    if (i < n) {
      u32 o = incl - cnt + (w ? wsum[0] : 0u);
      for_each_legal(p, L, [&](u32 code) {
        if (o < (u32)XCAP) {
          lcode[o] = code;
          llane[o] = (u8)tid;
        } else if (base + o < g.cap) {
          if (PAIRS) {
            pm[base + o] = i << 32 | code;
          } else {
            g.mv[base + o] = code;
            g.par[base + o] = (u32)i;
          }
        }
        o++;
      });
    }
    __syncthreads();
    for (u32 k = tid; k < total && base + k < g.cap; k += XTPB) {
      if (PAIRS) {
        if (k >= (u32)XCAP) break;
        pm[base + k] = (c0 + llane[k]) << 32 | lcode[k];
      } else {
        const u32 l = k < (u32)XCAP ? llane[k] : (u32)(g.par[base + k] - c0);
        const u32 code = k < (u32)XCAP ? lcode[k] : g.mv[base + k];
        Pos q;
        q.b0 = lb0[l];
        q.b1 = lb1[l];
        q.b2 = lb2[l];
        q.b3 = lb3[l];
        q.cr = lcr[l];
        q.stm = lmeta[l] & 1u;
        level_store(g, base + k, apply_count(q, code), lmeta[l] >> 1, (u32)(c0 + l), lwt[l]);
      }
    }
    __syncthreads();
  }
}

// ---- leaf: the children of `f` that the pairs name, counted into their roots.
// Bound: VALU issue (0.97-0.99 of the peak): a child costs 865 lane-instructions,
// 128.9 M of them 2.85-2.93 ms.
// A wavefront takes runs of 512 pairs in turn, one atomic a root of the run; of
// the grid about three blocks a CU are resident, and the rest of its 48 a CU
// fills the places of those that end first (a grid of the resident ones took
// 12 % longer).
// WT: f is a merged level, whose nodes count as often as they have paths.
constexpr int LEAF_BLOCKS = 48;
constexpr u32 LEAF_RUN = 512;
template <bool WT, bool NOBULK>
__global__ __launch_bounds__(TPB) void k_leaves(Level f, const u64 *__restrict__ pm, const u64 *__restrict__ npm, u64 cap,
                                                u64 *__restrict__ counts) {
  using Sum = std::conditional_t<WT, u64, u32>;  // a run: 512 pairs of at most 740 moves
  const int lane = threadIdx.x & 63;
  const u64 m = *npm;
  if (m > cap) return;
  const u64 waves = (u64)gridDim.x * (TPB / 64), w = (u64)blockIdx.x * (TPB / 64) + (threadIdx.x >> 6);
  for (u64 r0 = w * LEAF_RUN; r0 < m; r0 += waves * LEAF_RUN) {
    const u32 n = m - r0 < LEAF_RUN ? (u32)(m - r0) : LEAF_RUN;
    Sum acc = 0;  // this lane's part of the sum of root cur
    u32 cur = 0;
    auto flush = [&] {
      u64 s;
      if constexpr (WT) {
        s = acc;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
      } else {
        s = (u64)(u32)__builtin_amdgcn_readlane(zw::wave_scan_add((int)acc), 63);
      }
      if (lane == 0 && s) atomicAdd((unsigned long long *)&counts[cur], (unsigned long long)s);
      acc = 0;
    };
    for (u32 j0 = 0; j0 < n; j0 += 64) {
      const bool on = j0 + lane < n;
      Sum v = 0;
      u32 root = 0;
      if (on) {
        const u64 e = pm[r0 + j0 + lane];
        const u32 pi = (u32)(e >> 32);
        const u32 meta = f.meta[pi];
        Pos p;
        p.b0 = f.b0[pi];
        p.b1 = f.b1[pi];
        p.b2 = f.b2[pi];
        p.b3 = f.b3[pi];
        p.cr = f.cr[pi];
        p.stm = meta & 1u;
        const Pos c = apply_v(p, (u32)e);
        Legal L;
        analyse(c, L);
        // nobulk: the reference visits every leaf: it generates the leaf's
        // (quiescence) moves and counts one node (src/zetaperft.cl:1316-1326)
        v = NOBULK ? 1u + (u32)(count_legal(c, L, true) > 4096) : (u32)count_legal(c, L, false);
        if constexpr (WT) v *= f.wt[pi];
        root = meta >> 1;
      }
      u64 pending = __ballot(on);
      while (pending) {
        const u32 rl = (u32)__builtin_amdgcn_readlane((int)root, __builtin_ctzll(pending));
        if (rl != cur) {
          flush();
          cur = rl;
        }
        const bool its = on && root == rl;
        acc += its ? v : 0;
        pending &= ~__ballot(its);
      }
    }
    flush();
  }
}

// ---- merging a stored level.  k_merge enters every node of `f` into a hash
// table (64-bit words: half of the hash, index + 1); a node that meets an equal
// one -- same root, planes and flags, compared in full -- gives it its paths
// and leaves.  k_compact writes those that stay to `g`.  Bound: the random
// accesses (16 us a level of 0.1 M nodes); a level keeps some 60 % of its nodes
// and everything below shrinks with it.
__device__ __forceinline__ u64 node_hash(const Pos &p, u32 meta) {
  u64 h = p.b0 * 0x9E3779B97F4A7C15ULL ^ (p.b1 + 0x7F4A7C15ULL) * 0xBF58476D1CE4E5B9ULL;
  h = (h ^ (h >> 32)) + p.b2 * 0x94D049BB133111EBULL;
  h = (h ^ (h >> 29)) * 0xD1B54A32D192ED03ULL + p.b3 * 0x9E3779B97F4A7C15ULL;
  h = (h ^ (h >> 32)) * 0xBF58476D1CE4E5B9ULL + (p.cr ^ ((u64)meta << 8)) * 0x94D049BB133111EBULL;
  return h ^ (h >> 31);
}
__global__ __launch_bounds__(TPB) void k_table_clear(u64 *__restrict__ tab, Level f, u64 tabcap) {
  // two slots a node, a power of two
  const u64 n = level_size(f);
  u64 slots = 1024;
  while (slots < 2 * n && slots < tabcap) slots *= 2;
  for (u64 i = (u64)blockIdx.x * TPB + threadIdx.x; i < slots; i += (u64)gridDim.x * TPB) tab[i] = 0;
}
__global__ __launch_bounds__(TPB) void k_merge(u64 *__restrict__ tab, Level f, u64 tabcap) {
  const u64 n = level_size(f);
  u64 slots = 1024;
  while (slots < 2 * n && slots < tabcap) slots *= 2;
  for (u64 i = (u64)blockIdx.x * TPB + threadIdx.x; i < n; i += (u64)gridDim.x * TPB) {
    const Pos p = level_pos(f, i);
    const u32 meta = f.meta[i];
    const u64 h = node_hash(p, meta);
    const u64 e = (h & 0xFFFFFFFF00000000ULL) | (i + 1);
    u64 s = h & (slots - 1);
    for (;;) {
      const u64 old = atomicCAS((unsigned long long *)&tab[s], 0ULL, (unsigned long long)e);
      if (old == 0) break;
      if ((old ^ e) >> 32 == 0) {
        const u64 j = (old & 0xFFFFFFFFULL) - 1;
        const Pos q = level_pos(f, j);
        if (q.b0 == p.b0 && q.b1 == p.b1 && q.b2 == p.b2 && q.b3 == p.b3 && q.cr == p.cr && f.meta[j] == meta) {
          // the one in the table keeps its place; this one's paths are its own
          // until here (only entered nodes receive any)
          atomicAdd((unsigned long long *)&f.wt[j], (unsigned long long)f.wt[i]);
          f.par[i] = ~0u;  // gone
          break;
        }
      }
      s = (s + 1) & (slots - 1);
    }
  }
}
__global__ __launch_bounds__(TPB) void k_compact(Level f, Level g) {
  __shared__ u32 part[TPB / 64];
  __shared__ u64 base;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const u64 n = level_size(f);
  for (u64 i0 = (u64)blockIdx.x * TPB; i0 < n; i0 += (u64)gridDim.x * TPB) {
    const u64 i = i0 + threadIdx.x;
    const bool stay = i < n && f.par[i] != ~0u;
    const u64 b = __ballot(stay);
    __syncthreads();
    if (lane == 0) part[w] = (u32)popc(b);
    __syncthreads();
    if (threadIdx.x == 0)
      base = atomicAdd((unsigned long long *)g.count, (unsigned long long)(part[0] + part[1] + part[2] + part[3]));
    __syncthreads();
    u64 o = base + (u64)popc(b & ((1ULL << lane) - 1));
    for (int k = 0; k < w; k++) o += part[k];
    if (stay && o < g.cap) level_store(g, o, level_pos(f, i), f.meta[i] >> 1, f.par[i], f.wt[i]);
  }
}
// the roots as level 0 (many roots)
__global__ __launch_bounds__(TPB) void k_load_roots(const u64 *__restrict__ in, int n, Level f, u64 *__restrict__ counts) {
  const int i = blockIdx.x * TPB + threadIdx.x;
  if (i >= n) return;
  if (i == 0) *f.count = (u64)n;
  level_store(f, i, root_pos(in, i), (u32)i, (u32)i, 1);
  counts[i] = 0;
}
// The end of a chain: the sizes of its levels to the host's words (and cleared
// for the next call), the counts to host memory where the call wants them.
// Words: level sizes [0, 14), the most pairs of a pass, the pairs of the
// current one, sizes before merging [16, 30), all pairs.
constexpr int CTL_WORDS = 32, CTL_MOST = 14, CTL_PAIRS = 15, CTL_ALL = 30;
// after a pass over the last level's parents
__global__ void k_pass(u64 *ctl) {
  const u64 n = ctl[CTL_PAIRS];
  if (n > ctl[CTL_MOST]) ctl[CTL_MOST] = n;
  ctl[CTL_ALL] += n;
  ctl[CTL_PAIRS] = 0;
}
__global__ __launch_bounds__(TPB) void k_end(u64 *ctl, u64 *host, const u64 *__restrict__ counts, u64 *hcounts, int n) {
  const int i = blockIdx.x * TPB + threadIdx.x;
  if (i < CTL_WORDS) {
    host[i] = ctl[i];
    ctl[i] = 0;
  }
  if (hcounts && i < n) hcounts[i] = counts[i];
}

__global__ void k_u32_to_u64(const u32 *a, u64 *b, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

__global__ void k_fill_u64(u64 *b, int n, u64 v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = v;
}

// ---- playouts (workload generator)
__device__ __forceinline__ Pos start_pos() {  // setboard of the standard FEN with KQkq
  Pos p;
  p.b0 = 0xFFFF000000000000ULL;
  p.b1 = 0x91FF00000000FF91ULL;
  p.b2 = 0x5A0000000000005AULL;
  p.b3 = 0xAD000000000000ADULL;
  p.cr = 0x6EFFFFFFFFFFFF6EULL;
  p.stm = 0;
  return p;
}
struct PlayRng {
  u64 st;
  __device__ __forceinline__ PlayRng(u64 seed, u32 i, u64 attempt)
      : st(seed ^ ((u64)i * 0x9E3779B97F4A7C15ULL) ^ (attempt * 0xD1B54A32D192ED03ULL)) {}
  __device__ __forceinline__ u64 next() {
    u64 z = (st += 0x9E3779B97F4A7C15ULL);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
  }
};
__device__ __forceinline__ void store_playout(u64 *q, const Pos &p, u32 hmc) {
  q[0] = p.b0;
  q[1] = p.b1;
  q[2] = p.b2;
  q[3] = p.b3;
  q[4] = p.cr;
  q[5] = hash_full(p);
  q[6] = hmc;
  q[7] = p.stm;
}

// One wavefront a position, lane = square.  A playout is a chain of plies:
// with a lane a position 4096 of them are 64 wavefronts on 1024 SIMDs, each as
// slow as its longest playout and its busiest lane (1.84 ms at 20-60 plies,
// 0.23 ms here).  Bound: instruction issue of one wavefront, about 650 a ply;
// the rays of the lane's square serve the attack map, the pins and the targets,
// and the x-rays through the king are left to the positions in check.
__global__ __launch_bounds__(TPB) void k_playout_wide(u64 seed, int n, int minply, int maxply, u64 *out, u32 *fails) {
  const int lane = threadIdx.x & 63;
  const int i = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (TPB / 64) + (threadIdx.x >> 6)));
  if (i >= n) return;
  const LaneSq me = lane_sq(lane);
  // the lane's legal targets; all of them, summed up to this lane: incl
  auto targets = [&](const Pos &p, int &incl) {
    const u64 occ = p.b1 | p.b2 | p.b3;
    const LaneRays y = lane_rays(me, occ);
    u64 A = __ballot(lane_attacked(p, me, y));
    const u64 own = p.stm ? p.b0 : p.b0 ^ occ;
    u64 t;
    if (A & own & p.b1 & p.b2 & ~p.b3) {  // in check
      Node0 B;
      node_basics(p, B);
      A = __ballot(attacked_nk(B, lane));
      t = (own >> lane) & 1 ? lane_targets(p, B, A, lane, false) : 0;
    } else {
      t = lane_free_targets(p, me, y, A, lane);
    }
    incl = zw::wave_scan_add(popc(t));
    return t;
  };
  for (u64 a = 0; a <= 1000; a++) {
    PlayRng rng(seed, (u32)i, a);
    const int plies = minply + (int)(rng.next() % (u64)(maxply - minply + 1));
    Pos p = start_pos();
    u32 hmc = 0;
    bool ok = true;
    for (int k = 0; k <= plies; k++) {
      int incl;
      const u64 t = targets(p, incl);
      const int nl = __builtin_amdgcn_readlane(incl, 63);
      if (nl == 0 || hmc >= 100) {
        ok = false;
        break;
      }
      if (k == plies) break;
      const int pick = (int)mod_small(rng.next(), (u32)nl);
      // the origin whose targets hold move `pick` (origins ascending, then targets)
      const int f = __builtin_ctzll(__ballot(incl > pick));
      const u64 tf = (u64)(u32)__builtin_amdgcn_readlane((int)(u32)t, f) |
                     (u64)(u32)__builtin_amdgcn_readlane((int)(u32)(t >> 32), f) << 32;
      const u32 m = make_code(p, f, nth_bit(tf, pick - __builtin_amdgcn_readlane(incl - popc(t), f)));
      hmc = next_hmc(hmc, m);
      p = apply(p, m, true);
    }
    if (ok) {
      if (lane == 0) store_playout(out + (size_t)i * 8, p, hmc);
      return;
    }
  }
  if (lane == 0) atomicAdd(fails, 1u);
}

// one lane a position: more of them than the wavefronts the chip holds
__global__ __launch_bounds__(TPB) void k_playout(u64 seed, int n, int minply, int maxply, u64 *out,
                                                 u32 *fails) {
  const int i = blockIdx.x * TPB + threadIdx.x;
  if (i >= n) return;
  for (u64 a = 0; a <= 1000; a++) {
    PlayRng rng(seed, (u32)i, a);
    const int plies = minply + (int)(rng.next() % (u64)(maxply - minply + 1));
    Pos p = start_pos();
    u32 hmc = 0;
    bool ok = true;
    for (int k = 0; k <= plies; k++) {
      Legal L;
      analyse(p, L);
      const int nl = count_legal(p, L, false);
      if (nl == 0 || hmc >= 100) {
        ok = false;
        break;
      }
      if (k == plies) break;
      const u32 m = nth_legal(p, L, (int)mod_small(rng.next(), (u32)nl));
      hmc = next_hmc(hmc, m);
      p = apply_v(p, m);
    }
    if (ok) {
      store_playout(out + (size_t)i * 8, p, hmc);
      return;
    }
  }
  atomicAdd(fails, 1u);
}

// ---- host driver
constexpr int MAXLEV = 16;

struct LevelBufs {
  zr::DevBuf b0, b1, b2, b3, cr, meta, cnt;  // SoA positions
  zr::DevBuf off, bsum;                      // scan
  zr::DevBuf pm;                             // (parent index << 32 | move) pairs of the next level
  size_t cap = 0, paircap = 0;
};

struct PerftState {
  LevelBufs lev[MAXLEV];
  zr::DevBuf total, roots, counts, fails, cuts;
};
PerftState g_ps;

// ---- the allocation-free entry point's scratch array: the frontier of a
// call to zeta_perft_batch_device_noalloc lives here instead of in buffers
// the library allocates.  One array per device (the whole code object is
// loaded per device), held until the process ends; every call on a device
// reuses it, so calls that overlap on one device race.
constexpr size_t SCRATCH_BYTES = 256ULL << 20;
static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];
constexpr int SCRATCH_MAX_DEVICES = 64;
unsigned char *g_scratch_dev[SCRATCH_MAX_DEVICES];  // hipGetSymbolAddress of scratch, per device
hipError_t g_scratch_err = hipSuccess;
constexpr int NCUT_FIXED = 511;  // chunk cuts a level can take in the scratch array

// The buffers one perft call works in: the library's growable ones, or views
// into the scratch array with fixed capacities (never grown, never freed).
struct PerftBufs {
  LevelBufs *lev;
  zr::DevBuf *total, *cuts;
  u64 budget;  // most pairs a chunk may hold
  bool fixed;
};
PerftBufs g_pb;
LevelBufs g_fixed_lev[MAXLEV];
zr::DevBuf g_fixed_total, g_fixed_cuts;

void use_growable_bufs() {
  g_pb.lev = g_ps.lev;
  g_pb.total = &g_ps.total;
  g_pb.cuts = &g_ps.cuts;
  g_pb.budget = zr::ctx().cfg.frontier_budget;
  g_pb.fixed = false;
}

int ensure_level(int L, size_t n) {
  LevelBufs &b = g_pb.lev[L];
  if (b.cap >= n && b.cap) return ZETA_OK;
  if (g_pb.fixed)
    return zr::fail(ZETA_ENOMEM, "perft scratch: level %d needs %zu positions, holds %zu", L, n, b.cap);
  size_t cap = n + n / 4 + 1024;
  int r;
  b.cap = 0;  // none until all are there: one that cannot grow is gone
  if ((r = zr::ensure(b.b0, cap * 8)) || (r = zr::ensure(b.b1, cap * 8)) || (r = zr::ensure(b.b2, cap * 8)) ||
      (r = zr::ensure(b.b3, cap * 8)) || (r = zr::ensure(b.cr, cap * 8)) || (r = zr::ensure(b.meta, cap * 4)) ||
      (r = zr::ensure(b.cnt, cap * 4)) || (r = zr::ensure(b.off, (cap + 1) * 8)) ||
      (r = zr::ensure(b.bsum, (cap / SCAN_TILE + 2) * 8)))
    return r;
  b.cap = cap;
  return ZETA_OK;
}

int ensure_pairs(int L, size_t m) {
  LevelBufs &b = g_pb.lev[L];
  if (b.paircap >= m && b.paircap) return ZETA_OK;
  if (g_pb.fixed)
    return zr::fail(ZETA_ENOMEM, "perft scratch: level %d needs %zu pairs, holds %zu", L, m, b.paircap);
  size_t cap = m + m / 8 + 1024;
  int r;
  b.paircap = 0;
  if ((r = zr::ensure(b.pm, cap * 8))) return r;
  b.paircap = cap;
  return ZETA_OK;
}

Front front_of(int L) {
  LevelBufs &b = g_pb.lev[L];
  return Front{(u64 *)b.b0.p, (u64 *)b.b1.p, (u64 *)b.b2.p, (u64 *)b.b3.p,
               (u64 *)b.cr.p, (u32 *)b.meta.p, (u32 *)b.cnt.p};
}

inline unsigned blocks(size_t n, int per) { return (unsigned)((n + per - 1) / per); }

// exclusive scan of level L's counts [i0, i1) into lev[L].off[0..n]; returns total
int scan_counts(int L, size_t i0, size_t i1, u64 *total) {
  LevelBufs &b = g_pb.lev[L];
  const size_t n = i1 - i0;
  const size_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
  const u32 *cnt = (const u32 *)b.cnt.p + i0;
  if (n == 0) {
    *total = 0;
    return ZETA_OK;
  }
  ZLAUNCH(zr::K_PERFT_SCAN, n, k_scan_reduce, (unsigned)nb, TPB, 0, cnt, n, (u64 *)b.bsum.p);
  ZLAUNCH(zr::K_PERFT_SCAN, n, k_scan_top, 1, TPB, 0, (u64 *)b.bsum.p, nb, (u64 *)g_pb.total->p);
  ZLAUNCH(zr::K_PERFT_SCAN, n, k_scan_down, (unsigned)nb, TPB, 0, cnt, n, (const u64 *)b.bsum.p, (u64 *)b.off.p);
  // into the pinned word zeta_init set aside for it
  ZCHECK(hipMemcpyAsync(zr::ctx().perft_total_host, g_pb.total->p, 8, hipMemcpyDeviceToHost, zr::ctx().stream));
  ZCHECK(hipEventRecord(zr::ctx().ev_total, zr::ctx().stream));
  *total = ~0ULL;  // known after wait_total()
  return ZETA_OK;
}

// the total copied by scan_counts (the stream may run on: only the copy is waited for)
int wait_total(u64 *total) {
  ZCHECK(hipEventSynchronize(zr::ctx().ev_total));
  *total = *zr::ctx().perft_total_host;
  return ZETA_OK;
}

int process(int L, size_t i0, size_t i1, int D, u64 *d_counts, int nobulk) {
  u64 total = 0;
  int r = scan_counts(L, i0, i1, &total);
  if (r) return r;
  if (i1 == i0) return ZETA_OK;
  const u64 budget = g_pb.budget;
  LevelBufs &lv = g_pb.lev[L];
  // the expansion is queued before the total is known and writes into the
  // current pair buffer when the total fits it (k_expand checks), so the
  // host's wait for the total overlaps the expansion instead of preceding it
  const u64 spec_cap = lv.paircap < budget ? lv.paircap : budget;
  if (spec_cap)
    ZLAUNCH(zr::K_PERFT_EXPAND, i1 - i0, k_expand, blocks(i1 - i0, XTPB), XTPB, 0, front_of(L), i0, i1,
            (const u64 *)lv.off.p - i0, (u64)0, (u64 *)lv.pm.p, (const u64 *)g_pb.total->p, spec_cap);
  if ((r = wait_total(&total))) return r;
  if (total == 0) return ZETA_OK;
  // a level with more pairs than the budget runs in chunks of parents, each
  // with at most `budget` pairs; the cuts come from the device (k_cuts) so the
  // host reads a few words, not the level's offsets
  if (total > budget) {
    if (budget < 512) return zr::fail(ZETA_EINVAL, "frontier budget %llu is below 512 moves", (unsigned long long)budget);
    const u64 bp = budget - 256;
    const u64 nb = total / bp + 1;
    const size_t n = i1 - i0;
    if (g_pb.fixed) {
      if (nb > (u64)NCUT_FIXED)
        return zr::fail(ZETA_ENOMEM, "perft scratch: level %d needs %llu chunks, holds %d", L,
                        (unsigned long long)nb, NCUT_FIXED);
    } else if ((r = zr::ensure(g_ps.cuts, (size_t)(nb + 1) * 16))) {
      return r;
    }
    u64 *d_idx = (u64 *)g_pb.cuts->p, *d_off = d_idx + nb + 1;
    ZLAUNCH(zr::K_PERFT_SCAN, n, k_cuts, blocks(n, TPB), TPB, 0, (const u64 *)lv.off.p, n, bp, nb, d_idx, d_off);
    // the cuts come back into a vector, or into a fixed array on the stack
    // when the call may not allocate
    std::vector<u64> cutv;
    u64 cutf[2 * (NCUT_FIXED + 1)];
    u64 *cut = cutf;
    if (!g_pb.fixed) {
      cutv.resize(2 * (nb + 1));
      cut = cutv.data();
    }
    ZCHECK(hipMemcpyAsync(cut, d_idx, 2 * (nb + 1) * 8, hipMemcpyDeviceToHost, zr::ctx().stream));
    ZCHECK(hipStreamSynchronize(zr::ctx().stream));
    const u64 *cidx = cut, *coff = cut + nb + 1;
    for (u64 c = 0; c < nb; c++) {
      const size_t a0 = (size_t)cidx[c], a1 = (size_t)cidx[c + 1];
      if (a1 <= a0) continue;
      const u64 m = coff[c + 1] - coff[c];
      if (m == 0) continue;
      if ((r = ensure_pairs(L, m))) return r;
      ZLAUNCH(zr::K_PERFT_EXPAND, a1 - a0, k_expand, blocks(a1 - a0, XTPB), XTPB, 0, front_of(L), i0 + a0, i0 + a1,
              (const u64 *)lv.off.p - i0, coff[c], (u64 *)lv.pm.p, (const u64 *)nullptr, (u64)0);
      if (L + 1 == D - 1) {
        ZLAUNCH(zr::K_PERFT_LEAF, m, k_leaf, blocks(m, TPB), TPB, 0, front_of(L), (const u64 *)lv.pm.p,
                (size_t)m, d_counts, nobulk);
      } else {
        if ((r = ensure_level(L + 1, m))) return r;
        ZLAUNCH(zr::K_PERFT_APPLY, m, k_apply, blocks(m, TPB), TPB, 0, front_of(L),
                (const u64 *)lv.pm.p, (size_t)m, front_of(L + 1));
        if ((r = process(L + 1, 0, m, D, d_counts, nobulk))) return r;
      }
    }
    return ZETA_OK;
  }
  if (!spec_cap || total > spec_cap) {
    if ((r = ensure_pairs(L, total))) return r;
    ZLAUNCH(zr::K_PERFT_EXPAND, i1 - i0, k_expand, blocks(i1 - i0, XTPB), XTPB, 0, front_of(L), i0, i1,
            (const u64 *)lv.off.p - i0, (u64)0, (u64 *)lv.pm.p, (const u64 *)nullptr, (u64)0);
  }
  if (L + 1 == D - 1) {
    ZLAUNCH(zr::K_PERFT_LEAF, total, k_leaf, blocks(total, TPB), TPB, 0, front_of(L), (const u64 *)lv.pm.p,
            (size_t)total, d_counts, nobulk);
    return ZETA_OK;
  }
  if ((r = ensure_level(L + 1, total))) return r;
  ZLAUNCH(zr::K_PERFT_APPLY, total, k_apply, blocks(total, TPB), TPB, 0, front_of(L), (const u64 *)lv.pm.p,
          (size_t)total, front_of(L + 1));
  return process(L + 1, 0, total, D, d_counts, nobulk);
}

int perft_device(const void *d_pos, int n, int depth, u64 *d_counts, int flags) {
  const int nobulk = (flags & ZETA_PERFT_NOBULK) ? 1 : 0;
  if (n < 0 || depth < 0) return zr::fail(ZETA_EINVAL, "perft: n=%d depth=%d", n, depth);
  if (n == 0) return ZETA_OK;
  const int D = nobulk ? depth + 1 : depth;
  if (D >= MAXLEV) return zr::fail(ZETA_EINVAL, "perft depth %d exceeds %d", depth, MAXLEV - 2);
  int r;
  if (!g_pb.fixed && (r = zr::ensure(g_ps.total, 64))) return r;
  if (depth == 0) {
    ZLAUNCH(zr::K_PERFT_ROOTS, n, k_fill_u64, blocks(n, TPB), TPB, 0, d_counts, n, (u64)1);
    return ZETA_OK;
  }
  if ((r = ensure_level(0, (size_t)n))) return r;
  ZLAUNCH(zr::K_PERFT_ROOTS, n, k_roots, blocks(n, TPB), TPB, 0, (const u64 *)d_pos, n, front_of(0));
  if (D == 1) {
    ZLAUNCH(zr::K_PERFT_ROOTS, n, k_u32_to_u64, blocks(n, TPB), TPB, 0, (const u32 *)g_pb.lev[0].cnt.p, d_counts,
            n);
    return ZETA_OK;
  }
  ZLAUNCH(zr::K_PERFT_ROOTS, n, k_fill_u64, blocks(n, TPB), TPB, 0, d_counts, n, (u64)0);
  return process(0, 0, (size_t)n, D, d_counts, nobulk);
}

// ---- host side of the fast path
// Expected parents (32 moves a position) up to which a wavefront takes each.
// Two plies from n positions, a wavefront each against a lane each: n = 1 18
// and 29 us, 4096 33 and 73, 8192 51 and 71, 16384 85 and 72, 32768 145 and 86.
constexpr u64 WIDE_PARENTS = 16384;
// Playouts up to which a wavefront takes each.  Kernel time at 20-60 plies, a
// wavefront each against a lane each: n = 1 51 and 181 us, 4096 230 and 1802,
// 32768 1139 and 1588, 65536 2129 and 1613; at 8-40 plies 32768 748 and 918,
// 65536 1392 and 959.
constexpr int WIDE_PLAYOUTS = 40960;
constexpr int MERGE_LEVEL = 3;  // the first level with transpositions: x, y, z and z, y, x

struct LevelMem {
  zr::DevBuf b0, b1, b2, b3, cr, wt, meta, mv, par;
  u64 cap = 0;
};
struct FastState {
  LevelMem lev[MAXLEV], cand;  // cand: a level before it is merged
  zr::DevBuf ctl, table, pairs;
  u64 tabcap = 0;
  bool ctl_clean = false;
};
FastState g_fs;

void release_level(LevelMem &m) {
  for (zr::DevBuf *b : {&m.b0, &m.b1, &m.b2, &m.b3, &m.cr, &m.wt, &m.meta, &m.mv, &m.par}) zr::release(*b);
  m.cap = 0;
}
int ensure_fast(LevelMem &m, u64 n) {
  if (m.cap >= n) return ZETA_OK;
  m.cap = 0;
  int r;
  for (zr::DevBuf *b : {&m.b0, &m.b1, &m.b2, &m.b3, &m.cr, &m.wt})
    if ((r = zr::ensure(*b, n * 8))) return r;
  for (zr::DevBuf *b : {&m.meta, &m.mv, &m.par})
    if ((r = zr::ensure(*b, n * 4))) return r;
  m.cap = n;
  return ZETA_OK;
}
Level level_of(LevelMem &m, int word, u64 cap) {
  return Level{(u64 *)m.b0.p,   (u64 *)m.b1.p, (u64 *)m.b2.p,  (u64 *)m.b3.p, (u64 *)m.cr.p,
               (u64 *)m.wt.p,   (u32 *)m.meta.p, (u32 *)m.mv.p, (u32 *)m.par.p, (u64 *)g_fs.ctl.p + word, cap};
}

// One call's shape, and its buffers' capacities (a level's, and before merging).
struct Chain {
  const u64 *pos;  // device-visible
  int n, D;
  bool nobulk;
  u64 *counts, *hcounts;  // device; where the host reads them, or null
  u64 caps[MAXLEV], ccaps[MAXLEV], paircap;
  double expect(int L) const {  // parents at level L
    double e = n;
    for (int k = 0; k < L; k++) e *= 32;
    return e;
  }
  bool wide(int L) const { return expect(L) <= (double)WIDE_PARENTS; }
  bool merged(int L) const { return !nobulk && L >= MERGE_LEVEL; }
};

unsigned wide_blocks(double e) { return (unsigned)(e < 8 * 2048 ? (e + 7) / 8 : 2048); }
unsigned grid_blocks(double e, int per, int most) {
  const double b = e / per + 1, cap = (double)most * zr::ctx().cu_count;
  return (unsigned)(b < cap ? b : cap);
}
Level chain_level(const Chain &q, int L) { return level_of(g_fs.lev[L], L, q.caps[L]); }

// levels 1 .. D - 2
int launch_levels(const Chain &q) {
  for (int L = 0; L < q.D - 2; L++) {
    const bool merge = q.merged(L + 1);
    const Level out = merge ? level_of(g_fs.cand, 16 + L + 1, q.ccaps[L + 1]) : chain_level(q, L + 1);
    const double e = q.expect(L);
    if (q.wide(L)) {
      ZLAUNCH(zr::K_PERFT_EXPAND, 0, k_wide, wide_blocks(e), WIDE_TPB, 0, L ? (const u64 *)nullptr : q.pos, q.n,
              chain_level(q, L), out, q.counts);
    } else {
      if (L == 0)
        ZLAUNCH(zr::K_PERFT_ROOTS, q.n, k_load_roots, blocks(q.n, TPB), TPB, 0, q.pos, q.n, chain_level(q, 0), q.counts);
      ZLAUNCH(zr::K_PERFT_EXPAND, 0, k_spread<false>, grid_blocks(e, XTPB, 6), XTPB, 0, chain_level(q, L), (u64)0,
              ~(u64)0, out, (u64 *)nullptr);
    }
    if (merge) {
      const unsigned nb = grid_blocks(e * 32, TPB, 8);
      ZLAUNCH(zr::K_PERFT_APPLY, 0, k_table_clear, nb, TPB, 0, (u64 *)g_fs.table.p, out, g_fs.tabcap);
      ZLAUNCH(zr::K_PERFT_APPLY, 0, k_merge, nb, TPB, 0, (u64 *)g_fs.table.p, out, g_fs.tabcap);
      ZLAUNCH(zr::K_PERFT_APPLY, 0, k_compact, nb, TPB, 0, out, chain_level(q, L + 1));
    }
  }
  return ZETA_OK;
}

int launch_end(const Chain &q) {
  ZLAUNCH(zr::K_PERFT_SCAN, 0, k_end, q.hcounts ? blocks(q.n, TPB) : 1, TPB, 0, (u64 *)g_fs.ctl.p,
          (u64 *)zr::ctx().perft_ctl_dev, q.counts, q.hcounts, q.n);
  return ZETA_OK;
}

// the last level, below the parents of level D - 2: a wavefront a parent, or
// passes over [0, size) of `step` parents each
int launch_leaves(const Chain &q, u64 size, u64 step) {
  const int L = q.D - 2;
  const double e = q.expect(L);
  if (q.wide(L)) {
    // (a root's children: nothing is summed over blocks)
    ZLAUNCH(zr::K_PERFT_LEAF, 0, k_wide_leaf, wide_blocks(e), WIDE_TPB, 0, L ? (const u64 *)nullptr : q.pos, q.n,
            chain_level(q, L), L == 0 && q.hcounts ? q.hcounts : q.counts, q.nobulk ? 1 : 0);
    return ZETA_OK;
  }
  if (L == 0) ZLAUNCH(zr::K_PERFT_ROOTS, q.n, k_load_roots, blocks(q.n, TPB), TPB, 0, q.pos, q.n, chain_level(q, 0), q.counts);
  const Level pairs = level_of(g_fs.cand, CTL_PAIRS, q.paircap);
  const auto leaves = q.nobulk ? k_leaves<false, true> : L >= MERGE_LEVEL ? k_leaves<true, false> : k_leaves<false, false>;
  for (u64 i = 0; i < size; i += step) {
    const double here = e < (double)step ? e : (double)step;
    ZLAUNCH(zr::K_PERFT_EXPAND, 0, k_spread<true>, grid_blocks(here, XTPB, 6), XTPB, 0, chain_level(q, L), i, i + step,
            pairs, (u64 *)g_fs.pairs.p);
    ZLAUNCH(zr::K_PERFT_LEAF, 0, leaves, grid_blocks(here * 32, TPB, LEAF_BLOCKS), TPB, 0, chain_level(q, L),
            (const u64 *)g_fs.pairs.p, (const u64 *)pairs.count, q.paircap, q.counts);
    ZLAUNCH(zr::K_PERFT_SCAN, 0, k_pass, 1, 1, 0, (u64 *)g_fs.ctl.p);
  }
  return ZETA_OK;
}

void fast_release() {
  for (auto &l : g_fs.lev) release_level(l);
  release_level(g_fs.cand);
  zr::release(g_fs.ctl);
  zr::release(g_fs.table);
  zr::release(g_fs.pairs);
  g_fs.tabcap = 0;
  g_fs.ctl_clean = false;
}
// the device is full: the chunked path, which needs less, takes the call
int no_room() {
  (void)hipGetLastError();
  fast_release();
  return ZETA_OK;
}

// depth 1, queued only: the caller waits, behind the copy of the counts if it
// takes one (two waits: 300 positions 45 us, one 33)
int count_roots(const u64 *pos, int n, u64 *counts) {
  ZLAUNCH(zr::K_PERFT_ROOTS, n, k_count_roots, blocks(n, 64), 64, 0, pos, n, counts);
  return ZETA_OK;
}

// The whole call, depth 2 or more; *done = false: a level is beyond the frontier budget (or the
// call is one the fast path does not take) and nothing has been counted.
int fast_perft(const u64 *pos, int n, int depth, u64 *counts, u64 *hcounts, int flags, bool *done) {
  zr::Ctx &c = zr::ctx();
  *done = false;
  const bool nobulk = (flags & ZETA_PERFT_NOBULK) != 0;
  const int D = nobulk ? depth + 1 : depth;
  const u64 budget = c.cfg.frontier_budget;
  if (D < 2 || D >= MAXLEV || budget < 512 || (u64)n > budget || !c.perft_ctl_dev) return ZETA_OK;
  int r;
  if ((r = zr::ensure(g_fs.ctl, CTL_WORDS * 8))) return r;
  if (!g_fs.ctl_clean) {
    ZCHECK(hipMemsetAsync(g_fs.ctl.p, 0, CTL_WORDS * 8, c.stream));
    g_fs.ctl_clean = true;
  }
  Chain q = {pos, n, D, nobulk, counts, hcounts, {0}, {0}, 0};
  const u64 *const want = c.perft_ctl_host;
  // waits for the chain; the sizes it reports are in `want`
  auto finish = [&](int rc) {
    const hipError_t e = hipStreamSynchronize(c.stream);
    if (rc || e != hipSuccess) g_fs.ctl_clean = false;
    return rc ? rc : e != hipSuccess ? zr::hip_fail(e, "perft sync", __FILE__, __LINE__) : ZETA_OK;
  };
  auto clear_words = [&] { memset(c.perft_ctl_host, 0, CTL_WORDS * 8); };
  const int last = D - 2;
  // pairs a pass may hold and parents whose pairs they are: 64 moves a parent
  // at first, in the end as many as a parent can have
  u64 moves = 64;
  for (int tries = 0; tries < 3 * MAXLEV; tries++) {
    // room for every level: at first 40 moves a position up to 16 M nodes,
    // later what the levels have asked for
    double e = n;
    u64 cand = 0;
    for (int L = 0; L <= last; L++, e *= 40) {
      const double first = e < 65536 ? 65536 : (e > (double)(1 << 24) ? (double)(1 << 24) : e);
      u64 room = (u64)first > g_fs.lev[L].cap ? (u64)first : g_fs.lev[L].cap;
      if (L == 0) room = (u64)n;
      if (room > budget) room = budget;
      if (ensure_fast(g_fs.lev[L], room)) return no_room();
      q.caps[L] = g_fs.lev[L].cap < budget ? g_fs.lev[L].cap : budget;
      if (q.merged(L) && room > cand) cand = room;
    }
    if (cand) {
      if (ensure_fast(g_fs.cand, cand)) return no_room();
      for (int L = 0; L <= last; L++) q.ccaps[L] = g_fs.cand.cap < budget ? g_fs.cand.cap : budget;
      u64 t = 1024;
      while (t < 2 * g_fs.cand.cap) t *= 2;
      if (t > g_fs.tabcap) {
        g_fs.tabcap = 0;
        if (zr::ensure(g_fs.table, t * 8)) return no_room();
        g_fs.tabcap = t;
      }
    }
    const bool wide = q.wide(last);
    u64 step = ~(u64)0 >> 1;
    if (!wide) {
      u64 pairs = q.caps[last] > (u64)(1 << 27) / moves ? (u64)(1 << 27) : q.caps[last] * moves;
      if (pairs > budget) pairs = budget;
      if (pairs < (u64)MAXMOVES) return ZETA_OK;
      if (zr::ensure(g_fs.pairs, pairs * 8)) return no_room();
      q.paircap = pairs;
      step = pairs / moves;
    }
    // one chain where one pass holds every parent there can be, else the
    // level's size is read first
    const bool whole = wide || q.caps[last] <= step;
    clear_words();
    r = launch_levels(q);
    if (!r && whole) r = launch_leaves(q, 1, step);
    if (!r && !(wide && last == 0)) r = launch_end(q);
    if ((r = finish(r))) return r;
    bool again = false;
    for (int L = 1; L <= last && !again; L++) {
      if (q.merged(L) && want[16 + L] > q.ccaps[L]) {
        if (want[16 + L] > budget) return ZETA_OK;
        if (ensure_fast(g_fs.cand, want[16 + L] + want[16 + L] / 4)) return no_room();
        again = true;
      } else if (want[L] > q.caps[L]) {
        if (want[L] > budget) return ZETA_OK;
        if (ensure_fast(g_fs.lev[L], want[L] + want[L] / 4)) return no_room();
        again = true;
      }
    }
    if (again) continue;
    if (!whole) {
      // the level's count is a word the end has cleared: give it back
      const u64 size = last ? want[last] : (u64)n;
      ZLAUNCH(zr::K_PERFT_SCAN, 0, k_fill_u64, 1, 1, 0, (u64 *)g_fs.ctl.p + last, 1, size);
      r = launch_leaves(q, size, step);
      if (!r) r = launch_end(q);
      if ((r = finish(r))) return r;
    }
    if (!wide && want[CTL_MOST] > q.paircap) {
      moves = moves == 64 ? 256 : (u64)MAXMOVES;
      continue;
    }
    if (c.timing) c.kstat[zr::K_PERFT_LEAF].items += want[CTL_ALL];
    *done = true;
    return ZETA_OK;
  }
  return zr::fail(ZETA_ENOMEM, "perft: the levels keep growing");
}

}  // namespace

void perft_release() {
  for (auto &l : g_ps.lev) {
    zr::release(l.b0); zr::release(l.b1); zr::release(l.b2); zr::release(l.b3);
    zr::release(l.cr); zr::release(l.meta); zr::release(l.cnt); zr::release(l.off);
    zr::release(l.bsum); zr::release(l.pm);
    l.cap = l.paircap = 0;
  }
  zr::release(g_ps.total);
  zr::release(g_ps.roots);
  zr::release(g_ps.counts);
  zr::release(g_ps.fails);
  zr::release(g_ps.cuts);
  fast_release();
}

extern "C" int zeta_perft_batch_device(const void *d_pos, int n, int depth, void *d_counts, int flags) {
  int r = zr::require_up();
  if (r) return r;
  if ((!d_pos || !d_counts) && n > 0) return zr::fail(ZETA_EINVAL, "perft: null pointer");
  bool done = false;
  if (n > 0 && depth == 1 && !(flags & ZETA_PERFT_NOBULK)) {
    if (!(r = count_roots((const u64 *)d_pos, n, (u64 *)d_counts))) ZCHECK(hipStreamSynchronize(zr::ctx().stream));
    zr::time_collect();
    return r;
  }
  if (n > 0 && depth > 0) {
    r = fast_perft((const u64 *)d_pos, n, depth, (u64 *)d_counts, nullptr, flags, &done);
    if (r || done) {
      zr::time_collect();
      return r;
    }
  }
  use_growable_bufs();
  r = perft_device(d_pos, n, depth, (u64 *)d_counts, flags);
  hipError_t e = hipStreamSynchronize(zr::ctx().stream);
  zr::time_collect();
  if (r) return r;
  if (e != hipSuccess) return zr::hip_fail(e, "perft sync", __FILE__, __LINE__);
  return ZETA_OK;
}

// zeta_init, with the device current: where this device holds the scratch
// array (the array's name in host code is only a stand-in for it)
int perft_setup() {
  const int dev = zr::ctx().device;
  if (dev < 0 || dev >= SCRATCH_MAX_DEVICES) return zr::fail(ZETA_ENODEV, "perft: device %d beyond %d", dev,
                                                             SCRATCH_MAX_DEVICES);
  if (g_scratch_dev[dev]) return ZETA_OK;
  void *ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr) {
    // the other entry points do not need the array: the allocation-free one
    // reports this error when it is called
    (void)hipGetLastError();
    g_scratch_err = e != hipSuccess ? e : hipErrorInvalidSymbol;
    return ZETA_OK;
  }
  g_scratch_dev[dev] = (unsigned char *)ptr;
  return ZETA_OK;
}

// Views of the scratch array for a call of D - 1 frontier levels: every level
// holds up to C positions (5 x u64 planes, meta, count, offset, scan sums)
// and C pairs; C is the largest that fits, and it is the chunk budget, so no
// level and no chunk ever needs more.  Returns C, 0 when it is below what
// the roots need.
size_t fixed_layout(unsigned char *base, int D, size_t n) {
  const int nl = D - 1 > 1 ? D - 1 : 1;
  const size_t align = 256, head = 2 * align + 2 * (NCUT_FIXED + 1) * 8;
  // per level: 9 arrays, each rounded up to the alignment
  const size_t slack = 9 * align + 8 * 3;
  const size_t per_pos = 5 * 8 + 4 + 4 + 8 + 8;  // planes, meta, cnt, off, pairs
  size_t C = (SCRATCH_BYTES - head) / nl;
  C = C > slack ? (C - slack) / per_pos : 0;
  C -= C / (SCAN_TILE / 8) + 2;  // room for the scan sums (8 B per SCAN_TILE positions)
  if (C < 1024 || C < n) return 0;
  size_t o = 0;
  auto take = [&](size_t bytes) {
    void *p = base + o;
    o += (bytes + align - 1) / align * align;
    return p;
  };
  g_fixed_total.p = take(64);
  g_fixed_total.bytes = 64;
  g_fixed_cuts.p = take(2 * (NCUT_FIXED + 1) * 8);
  g_fixed_cuts.bytes = 2 * (NCUT_FIXED + 1) * 8;
  for (int L = 0; L < MAXLEV; L++) {
    LevelBufs &b = g_fixed_lev[L];
    b = LevelBufs();
    if (L >= nl) continue;
    zr::DevBuf *planes[5] = {&b.b0, &b.b1, &b.b2, &b.b3, &b.cr};
    for (auto *q : planes) {
      q->p = take(C * 8);
      q->bytes = C * 8;
    }
    b.meta.p = take(C * 4);
    b.meta.bytes = C * 4;
    b.cnt.p = take(C * 4);
    b.cnt.bytes = C * 4;
    b.off.p = take((C + 1) * 8);
    b.off.bytes = (C + 1) * 8;
    b.bsum.p = take((C / SCAN_TILE + 2) * 8);
    b.bsum.bytes = (C / SCAN_TILE + 2) * 8;
    b.pm.p = take(C * 8);
    b.pm.bytes = C * 8;
    b.cap = C;
    b.paircap = C;
  }
  if (o > SCRATCH_BYTES) return 0;
  return C;
}

extern "C" int zeta_perft_batch_device_noalloc(const void *d_pos, int n, int depth, void *d_counts, int flags) {
  int r = zr::require_up();
  if (r) return r;
  if ((!d_pos || !d_counts) && n > 0) return zr::fail(ZETA_EINVAL, "perft (no-alloc): null pointer");
  if (n < 0 || n > ZETA_NOALLOC_MAX_ROOTS)
    return zr::fail(ZETA_EINVAL, "perft (no-alloc): %d roots, at most %d", n, ZETA_NOALLOC_MAX_ROOTS);
  if (depth < 0 || depth > ZETA_NOALLOC_MAX_DEPTH)
    return zr::fail(ZETA_EINVAL, "perft (no-alloc): depth %d, at most %d", depth, ZETA_NOALLOC_MAX_DEPTH);
  const int dev = zr::ctx().device;
  unsigned char *base = (dev >= 0 && dev < SCRATCH_MAX_DEVICES) ? g_scratch_dev[dev] : nullptr;
  if (!base)
    return zr::fail(ZETA_ENODEV, "perft (no-alloc): no scratch array on device %d (hipGetSymbolAddress: %s)", dev,
                    hipGetErrorString(g_scratch_err));
  const int D = (flags & ZETA_PERFT_NOBULK) ? depth + 1 : depth;
  const size_t C = fixed_layout(base, D, (size_t)n);
  if (!C) return zr::fail(ZETA_EINVAL, "perft (no-alloc): %d roots at depth %d do not fit the scratch array", n, depth);
  g_pb.lev = g_fixed_lev;
  g_pb.total = &g_fixed_total;
  g_pb.cuts = &g_fixed_cuts;
  g_pb.budget = C;
  g_pb.fixed = true;
  // no kernel timing here: its events come from a pool that may grow
  const bool timing = zr::ctx().timing;
  zr::ctx().timing = false;
  r = perft_device(d_pos, n, depth, (u64 *)d_counts, flags);
  zr::ctx().timing = timing;
  use_growable_bufs();
  const hipError_t e = hipStreamSynchronize(zr::ctx().stream);
  if (r) return r;
  if (e != hipSuccess) return zr::hip_fail(e, "perft (no-alloc) sync", __FILE__, __LINE__);
  return ZETA_OK;
}

extern "C" int zeta_perft_batch(const zeta_pos *pos, int n, int depth, uint64_t *counts) {
  int r = zr::require_up();
  if (r) return r;
  if (n < 0 || (n > 0 && (!pos || !counts))) return zr::fail(ZETA_EINVAL, "perft: bad arguments");
  if (n == 0) return ZETA_OK;
  if ((r = zr::ensure(g_ps.roots, (size_t)n * sizeof(zeta_pos))) || (r = zr::ensure(g_ps.counts, (size_t)n * 8)))
    return r;
  zr::Ctx &c = zr::ctx();
  // few positions go through pinned host memory, which the kernels read and
  // write themselves: two copies less in the chain
  const bool pinned = n <= zr::PERFT_STAGE;
  if (pinned) memcpy(c.perft_stage_host, pos, (size_t)n * sizeof(zeta_pos));
  else ZCHECK(hipMemcpyAsync(g_ps.roots.p, pos, (size_t)n * sizeof(zeta_pos), hipMemcpyHostToDevice, c.stream));
  if (depth > 0) {
    bool done = depth == 1;
    const u64 *const in = pinned ? (const u64 *)c.perft_stage_dev : (const u64 *)g_ps.roots.p;
    u64 *const out = (u64 *)g_ps.counts.p, *const hout = pinned ? (u64 *)c.perft_counts_dev : nullptr;
    r = depth == 1 ? count_roots(in, n, pinned ? hout : out) : fast_perft(in, n, depth, out, hout, 0, &done);
    if (r) {
      zr::time_collect();
      return r;
    }
    if (done) {
      if (!pinned) ZCHECK(hipMemcpyAsync(counts, out, (size_t)n * 8, hipMemcpyDeviceToHost, c.stream));
      if (!pinned || depth == 1) ZCHECK(hipStreamSynchronize(c.stream));
      if (pinned) memcpy(counts, c.perft_counts_host, (size_t)n * 8);
      zr::time_collect();
      return ZETA_OK;
    }
  }
  if (pinned) ZCHECK(hipMemcpyAsync(g_ps.roots.p, pos, (size_t)n * sizeof(zeta_pos), hipMemcpyHostToDevice, c.stream));
  use_growable_bufs();
  r = perft_device(g_ps.roots.p, n, depth, (u64 *)g_ps.counts.p, 0);
  if (r) {
    (void)hipStreamSynchronize(zr::ctx().stream);
    zr::time_collect();
    return r;
  }
  ZCHECK(hipMemcpyAsync(counts, g_ps.counts.p, (size_t)n * 8, hipMemcpyDeviceToHost, zr::ctx().stream));
  ZCHECK(hipStreamSynchronize(zr::ctx().stream));
  zr::time_collect();
  return ZETA_OK;
}

extern "C" int zeta_playouts(uint64_t seed, int n, int minply, int maxply, zeta_pos *out) {
  int r = zr::require_up();
  if (r) return r;
  if (n < 0 || minply < 0 || maxply < minply || (n > 0 && !out))
    return zr::fail(ZETA_EINVAL, "playouts: bad arguments");
  if (n == 0) return ZETA_OK;
  if ((r = zr::ensure(g_ps.roots, (size_t)n * sizeof(zeta_pos))) || (r = zr::ensure(g_ps.fails, 4))) return r;
  ZCHECK(hipMemsetAsync(g_ps.fails.p, 0, 4, zr::ctx().stream));
  const bool wide = n <= WIDE_PLAYOUTS;
  ZLAUNCH(zr::K_PLAYOUT, n, wide ? k_playout_wide : k_playout, blocks(n, wide ? TPB / 64 : TPB), TPB, 0, seed, n, minply,
          maxply, (u64 *)g_ps.roots.p, (u32 *)g_ps.fails.p);
  u32 fails = 0;
  ZCHECK(hipMemcpyAsync(out, g_ps.roots.p, (size_t)n * sizeof(zeta_pos), hipMemcpyDeviceToHost, zr::ctx().stream));
  ZCHECK(hipMemcpyAsync(&fails, g_ps.fails.p, 4, hipMemcpyDeviceToHost, zr::ctx().stream));
  ZCHECK(hipStreamSynchronize(zr::ctx().stream));
  zr::time_collect();
  if (fails) return zr::fail(ZETA_EINVAL, "playouts: %u positions found no acceptable playout", fails);
  return ZETA_OK;
}
