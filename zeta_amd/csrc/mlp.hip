// mlp.hip -- training of the learned move-ordering network on gfx950:
// BF16 MFMA forward and backward GEMMs with FP32 accumulation, pairwise
// ranking loss, Adam with FP32 master weights.  No reference counterpart
// (the reference orders moves with fixed scores, src/zeta.cl:2059-2104).
//
// Training examples are pairs logged by the search at cut nodes: the move
// that caused the beta cutoff and another move of the node.  A step takes P
// pairs = B = 2P examples (row 2p the cutoff move of pair p, row 2p+1 the
// other) and minimises
//   L = mean_p softplus(s(neg_p) - s(pos_p) + o_p / PLAIN_PER_LOGIT),
// o_p the plain ordering's score difference of the pair: the search ranks
// by plain score + PLAIN_PER_LOGIT x s, so s learns a correction of it.
// One step is two launches.  k_rows takes 32 rows a block from the records to
// the gradient at the first layer's output, k_weights forms the weight
// gradients and applies Adam to them in place.  The products, on
// v_mfma_f32_32x32x16_bf16 tiles (BF16 operands, FP32 accumulation):
//   z1   [B][256]   = X     [B][928]  . W1t  [256][928]  -> h1 = relu(z1 + b1)
//   z2   [B][32]    = H1    [B][256]  . W2t  [32][256]   -> scores, loss, dz2
//   dH1  [B][256]   = dZ2   [B][32]   . W2   [256][32]   -> dz1, b1 gradient
//   gW2t [32][256]  = dZ2t  [32][B]   . H1t  [256][B]
//   gW1t [256][928] = dZ1t  [256][B]  . Xt   [928][B]
#include <math.h>
#include <string.h>

#include <vector>

#include "mlp.h"
#include "runtime.h"

using namespace zm;
using zc::u32;
using zc::u8;
using zc::u64;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// internal FP32 layout (master weights, gradients, Adam moments)
constexpr int I_W1T = 0;                      // [256][928]
constexpr int I_B1 = I_W1T + NH1 * NINP;      // [256]
constexpr int I_W2T = I_B1 + NH1;             // [32][256]
constexpr int I_B2 = I_W2T + NH2 * NH1;       // [32]
constexpr int I_W3 = I_B2 + NH2;              // [32]
constexpr int I_B3 = I_W3 + NH2;              // [1]
constexpr int NINT = I_B3 + 1;

struct PairRec {  // one logged training pair (48 B)
  u64 b0, b1, b2, b3;
  u32 stm, mpos, mneg, depth;
};

constexpr u16 BF_ONE = 0x3F80;

// ---- examples of a batch: pair p gives rows 2p (its cutoff move) and 2p+1
// (the other move), so every 32-row tile of a product holds 16 whole pairs
// and the loss is an epilogue of the layer-2 product.

// record index of pair i of a training step: splitmix64 of (seed, i) mod nrec
__device__ __forceinline__ u32 sample_index(u64 seed, int i, u64 nrec) {
  u64 z = seed + (u64)(i + 1) * 0x9E3779B97F4A7C15ULL;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  z ^= z >> 31;
  return (u32)(z % nrec);
}

__device__ __forceinline__ uint2 pack4(const u16 *v) {
  return make_uint2((u32)v[0] | ((u32)v[1] << 16), (u32)v[2] | ((u32)v[3] << 16));
}
__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// C row of register i in lane half h
__device__ __forceinline__ int c_row(int i, int h) { return 8 * (i >> 2) + 4 * h + (i & 3); }

// A one-hot operand is eight feature bits of a row, or eight row bits of a
// feature: a byte, turned into eight BF16 by a 4-KB table in LDS.
struct OneHot {
  bf16x8 v[256];
};
__device__ __forceinline__ void one_hot_table(OneHot &t, int tid) {
  if (tid < 256) {
    u32 w[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
      w[j] = (((tid >> (2 * j)) & 1) ? (u32)BF_ONE : 0u) | (((tid >> (2 * j + 1)) & 1) ? (u32)BF_ONE << 16 : 0u);
    *(uint4 *)&t.v[tid] = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// The 16-bit operands of the products lie in memory as the matrix unit takes
// them: the 32x16 block (tile t, step s) is 1 KB, 16 bytes a lane -- index
// c = t * 32 + (lane & 31), k = s * 16 + 8 * (lane >> 5) + 0..7 -- so that a
// wavefront's operand is one contiguous load.  (Row by row, a load touched 64
// lines a power of two apart: the weight gradients of 16384 pairs took 130 us.)
__device__ __forceinline__ size_t frag(int t, int s, int steps) { return ((size_t)t * steps + s) * 512; }
// element (c, k) of it
__device__ __forceinline__ size_t frag_at(int c, int k, int steps) {
  return frag(c >> 5, k >> 4, steps) + (((k >> 3) & 1) * 32 + (c & 31)) * 8 + (k & 7);
}

// A barrier for data in LDS: loads from and stores to device memory stay in
// flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

constexpr int TPB = 512;       // eight wavefronts
constexpr int NW = TPB / 64;
constexpr int HS = NH1 + 8;    // LDS row strides that spread the banks
constexpr int DS = NH2 + 8;

// Gradients of the biases and the head, and the loss: each block of k_rows
// leaves its part of every sum, [sum][block]; k_weights adds them up in 64
// bits, always in the same order.
constexpr int S_B1 = 0, S_B2 = NH1, S_W3 = S_B2 + NH2, S_B3 = S_W3 + NH2, S_LOSS = S_B3 + 1, NSUM = S_LOSS + 1;

// Forward and backward of 32 rows (16 pairs) a block, from the records to
// dz1, all of it on chip: the rows' features as bits, h1 = relu(z1 + b1) with a
// 32-column tile a wavefront, kept in registers for relu' and as BF16 in LDS
// for layer 2, then z2, the scores, the loss and dz2, then dz1.  What the
// weight gradients need goes out as BF16 operands (h1, dz1, dz2) and as the
// one-hot rows' bits, 1/16 of their BF16 size.  nrec > 0: the step's pairs are
// drawn here (sample_index); nrec = 0: pair p is record p.
// Bound: latency.  The phases follow one another -- record, features, the W1
// operand (464 KB a block), a chain of products, the head -- and 0.4 of the
// wavefronts' cycles wait for memory, 0.35 for an issue slot; the L1 gives
// 0.36 of its 64 bytes a cycle, the matrix units are busy 0.12 of the time, and
// at 2048 pairs half of the CUs have no block.  A third of the W1 operand is
// asked for before the records are looked at, a third while the features are
// taken apart.
// At 2048 pairs 14.3 us, where features, layer 1, head and layer-1 backward as
// launches of their own took 39 us; 50 us at 16384 pairs.
__global__ __launch_bounds__(TPB) void k_rows(const PairRec *__restrict__ recs, int B, u64 nrec, u64 seed,
                                              const float *__restrict__ prm, const u16 *__restrict__ w1x,
                                              const u16 *__restrict__ w2t, const u16 *__restrict__ w2,
                                              u32 *__restrict__ bits, u16 *__restrict__ h1x, u16 *__restrict__ dz2x,
                                              u16 *__restrict__ dz1x, float *__restrict__ sums) {
  __shared__ OneHot hot;
  __shared__ u32 mask[NINP];       // feature -> rows
  __shared__ u32 rowbits[32][NINP / 32];  // row -> features
  __shared__ u32 depth[16];
  __shared__ __align__(16) u16 h1s[32 * HS];
  __shared__ __align__(16) u16 d2s[32 * DS];
  __shared__ float red[4][16][64];
  __shared__ float hs[4][2 * NH2 + 2];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, half = lane >> 5;
  const int e0 = blockIdx.x * 32;
  // operands that depend on nothing: layer 2 and its backward
  const int c1 = 32 * w + r;  // this lane's hidden unit
  constexpr int KS = NINP / 16, AHEAD = 20;  // layer-1 steps of 16 features; a third of them, loaded together
  bf16x8 bw2[4], bw2t[2], bw1[AHEAD];
  // sixteen threads per row, half a rank of the board each (the first one also
  // the move's features)
  const int row = tid >> 4, part = tid & 15, e = e0 + row;
  const PairRec rc = recs[nrec ? sample_index(seed, e >> 1, nrec) : (u32)(e >> 1)];
  const u16 *pb = w1x + frag(w, 0, KS) + lane * 8;
  const int units = B / 16;
#pragma unroll
  for (int j = 0; j < AHEAD; j++) bw1[j] = *(const bf16x8 *)(pb + 512 * j);
#pragma unroll
  for (int j = 0; j < 4; j++) bw2[j] = *(const bf16x8 *)(w2t + (size_t)r * NH1 + (4 * (w & 3) + j) * 16 + 8 * half);
#pragma unroll
  for (int j = 0; j < 2; j++) bw2t[j] = *(const bf16x8 *)(w2 + (size_t)c1 * NH2 + 16 * j + 8 * half);
  const float b1c = prm[I_B1 + c1], b2o = prm[I_B2 + r], w3o = prm[I_W3 + r], b3 = prm[I_B3];
  one_hot_table(hot, tid);
  for (int f = tid; f < NINP; f += TPB) {
    mask[f] = 0;
    ((u32 *)rowbits)[f] = 0;
  }
  lds_barrier();
  bf16x8 next[AHEAD];
#pragma unroll
  for (int j = 0; j < AHEAD; j++) next[j] = *(const bf16x8 *)(pb + 512 * (AHEAD + j));
  {
    zc::Pos p;
    p.b0 = rc.b0; p.b1 = rc.b1; p.b2 = rc.b2; p.b3 = rc.b3; p.cr = 0; p.stm = rc.stm & 1u;
    const u32 bit = 1u << row;
    auto add = [&](int f) {
      atomicOr(&mask[f], bit);
      atomicOr(&rowbits[row][f >> 5], 1u << (f & 31));
    };
    u64 occ = (p.b1 | p.b2 | p.b3) & (0xFull << (4 * part));
    while (occ) {
      const int sq = zc::lsb(occ);
      occ &= occ - 1;
      add(feat_ps(zc::piece_at(p, sq), sq, p.stm));
    }
    if (part == 0) {
      const u32 m = (e & 1) ? rc.mneg : rc.mpos;
      add(feat_from(m, p.stm));
      add(feat_to(m, p.stm));
      add(feat_piece(m));
      const int fc = feat_capt(m);
      if (fc >= 0) add(fc);
      if (!(row & 1)) depth[row >> 1] = rc.depth;
    }
  }
  lds_barrier();
  for (int f = tid; f < NINP; f += TPB) bits[(size_t)blockIdx.x * NINP + f] = mask[f];

  // z1 = X . W1t^T
  f32x16 acc = {};
  {
    auto row_operand = [&](int k) { return hot.v[(rowbits[r][k >> 1] >> (16 * (k & 1) + 8 * half)) & 0xFFu]; };
    bf16x8 a[4];
#pragma unroll
    for (int j = 0; j < 4; j++) a[j] = row_operand(j);
#pragma unroll
    for (int k = 0; k < KS; k++) {
      const int g = k / AHEAD, i = k % AHEAD;
      acc = mfma(a[k & 3], g == 1 ? next[i] : bw1[i], acc);
      if (k + 4 < KS) a[k & 3] = row_operand(k + 4);
      if (g == 0 && 2 * AHEAD + i < KS) bw1[i] = *(const bf16x8 *)(pb + 512 * (2 * AHEAD + i));
    }
  }
  float h[16];
  {
#pragma unroll
    for (int g = 0; g < 4; g++) {
      u16 hb[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const float x = acc[4 * g + j] + b1c;
        h[4 * g + j] = x > 0.f ? x : 0.f;
        hb[j] = f2bf(h[4 * g + j]);
        h1s[c_row(4 * g + j, half) * HS + c1] = hb[j];
      }
      *(uint2 *)(h1x + frag_at(c1, e0 + c_row(4 * g, half), units)) = pack4(hb);
    }
  }
  lds_barrier();

  // z2 = H1 . W2t^T on the first four wavefronts, a quarter of the hidden
  // units each; the partial tiles are summed in LDS and wavefront w takes the
  // rows of registers 4w .. 4w+3: h2 = relu(z2 + b2), s = w3.h2 + b3 (sum over
  // the 32 lanes of a half), and for its 2 pairs per half the loss
  // softplus(s_neg - s_pos + o/PLAIN_PER_LOGIT), dz2 and the b2, W3, b3
  // gradients and the loss
  if (w < 4) {
    f32x16 z = {};
#pragma unroll
    for (int j = 0; j < 4; j++) z = mfma(*(const bf16x8 *)(h1s + r * HS + (4 * w + j) * 16 + 8 * half), bw2[j], z);
#pragma unroll
    for (int i = 0; i < 16; i++) red[w][i][lane] = z[i];
  }
  lds_barrier();
  if (w < 4) {
    float h2[4], sc[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int i = 4 * w + j;
      const float z = red[0][i][lane] + red[1][i][lane] + red[2][i][lane] + red[3][i][lane] + b2o;
      h2[j] = z > 0.f ? z : 0.f;
      float t = w3o * h2[j];
#pragma unroll
      for (int x = 16; x > 0; x >>= 1) t += __shfl_xor(t, x, 64);
      sc[j] = t + b3;
    }
    const float invP = 1.f / (float)(B / 2);
    float gb2 = 0.f, gw3 = 0.f, gb3 = 0.f, gl = 0.f;
    u16 dzb[4];
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const int j = 2 * q;  // rows j, j+1 of this lane's group: an even row (cutoff move) and its pair
      const u32 dw = depth[(c_row(4 * w, half) + j) >> 1];
      const float d = sc[j + 1] - sc[j] + (float)pair_offset(dw) / (float)PLAIN_PER_LOGIT;
      const float sig = 1.f / (1.f + expf(-d));
      const float l = d > 0.f ? d + log1pf(expf(-d)) : log1pf(expf(d));
      const float ds0 = -sig * invP, ds1 = sig * invP;
      const float dz0 = h2[j] > 0.f ? ds0 * w3o : 0.f, dz1 = h2[j + 1] > 0.f ? ds1 * w3o : 0.f;
      dzb[j] = f2bf(dz0);
      dzb[j + 1] = f2bf(dz1);
      gb2 += dz0 + dz1;
      gw3 += ds0 * h2[j] + ds1 * h2[j + 1];
      if (r == 0) {
        gb3 += ds0 + ds1;
        gl += l * invP;
      }
    }
    const int row0 = c_row(4 * w, half);
#pragma unroll
    for (int j = 0; j < 4; j++) d2s[(row0 + j) * DS + r] = dzb[j];
    *(uint2 *)(dz2x + frag_at(r, e0 + row0, units)) = pack4(dzb);
    gb2 += __shfl_xor(gb2, 32, 64);
    gw3 += __shfl_xor(gw3, 32, 64);
    gb3 += __shfl_xor(gb3, 32, 64);
    gl += __shfl_xor(gl, 32, 64);
    if (lane < 32) {
      hs[w][r] = gb2;
      hs[w][NH2 + r] = gw3;
    }
    if (lane == 0) {
      hs[w][2 * NH2] = gb3;
      hs[w][2 * NH2 + 1] = gl;
    }
  }
  lds_barrier();
  if (tid < 2 * NH2 + 2)
    sums[(size_t)(S_B2 + tid) * gridDim.x + blockIdx.x] = hs[0][tid] + hs[1][tid] + hs[2][tid] + hs[3][tid];

  // dh1 = dZ2 . W2^T -> dz1 = dh1 * relu'(h1); b1 gradient
  f32x16 dh = {};
#pragma unroll
  for (int j = 0; j < 2; j++) dh = mfma(*(const bf16x8 *)(d2s + r * DS + 16 * j + 8 * half), bw2t[j], dh);
  float cs = 0.f;
#pragma unroll
  for (int g = 0; g < 4; g++) {
    u16 db[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float dz = h[4 * g + j] > 0.f ? dh[4 * g + j] : 0.f;
      cs += dz;
      db[j] = f2bf(dz);
    }
    *(uint2 *)(dz1x + frag_at(c1, e0 + c_row(4 * g, half), units)) = pack4(db);
  }
  cs += __shfl_xor(cs, 32, 64);
  if (lane < 32) sums[(size_t)(S_B1 + c1) * gridDim.x + blockIdx.x] = cs;
}

// ---- weight gradients, and the use made of them in the same pass
struct Adam {
  float lr, b1, b2, eps, c1, c2;
  float *prm, *m, *v;
  u16 *w1x, *w1f, *w2t, *w2;  // BF16 working copies of the weights
};
struct AdamState {
  float p, m, v;
};
__device__ __forceinline__ AdamState adam_load(const Adam &a, int i) { return AdamState{a.prm[i], a.m[i], a.v[i]}; }
__device__ __forceinline__ float adam_step(const Adam &a, int i, const AdamState &s, float g) {
  const float mi = a.b1 * s.m + (1.f - a.b1) * g;
  const float vi = a.b2 * s.v + (1.f - a.b2) * g * g;
  a.m[i] = mi;
  a.v[i] = vi;
  const float p = s.p - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
  a.prm[i] = p;
  return p;
}

__device__ __forceinline__ int w2_slices(int B) {
  int n = 4;
  while (n < 128 && B / (2 * n) >= 128) n *= 2;
  return n;
}

constexpr int W1_TILES = (NH1 / 32) * (NINP / 32), W2_TILES = NH1 / 32;
constexpr int SUM_BLOCKS = (NSUM + 31) / 32;  // 32 sums a block

// gW1t [256][928] = dZ1t . X and gW2t [32][256] = dZ2t . H1: one 32x32 tile a
// block, the batch split over its eight wavefronts and summed in LDS, so that
// the block holds the whole gradient of its weights.  UPDATE: Adam on them
// and their BF16 copies here (no gradient goes to memory and no pass of its
// own updates the weights); else the gradient in the ABI's layout.  The last
// blocks do the same for the biases and the head, whose sums k_rows left.
// X comes from its bits (a byte is one operand).
// At 2048 pairs 9.3 us, where the two products (22 us) and the update (6.6 us)
// were passes of their own; 48 us at 16384 pairs.  Bound: latency, of operands
// that another chiplet's kernel has just written, and of the table lookups (a
// tenth of the cycles are bank conflicts) ahead of one chain of products: 0.4 of
// the cycles wait for memory, the L1 gives 0.36 of its 64 bytes a cycle, the
// matrix units are busy 0.14 of the time.
template <bool UPDATE>
__global__ __launch_bounds__(TPB) void k_weights(int B, const u32 *__restrict__ bits, const u16 *__restrict__ h1x,
                                                 const u16 *__restrict__ dz2x, const u16 *__restrict__ dz1x, const float *__restrict__ sums,
                                                 Adam ad, float *__restrict__ gout, float *__restrict__ loss) {
  __shared__ OneHot hot;
  __shared__ float red[NW][16][64];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, half = lane >> 5;
  if (blockIdx.x >= W1_TILES + W2_TILES) {
    const int nblk = B / 32;
    for (int q = w; q < 32; q += NW) {
      const int t = (blockIdx.x - (W1_TILES + W2_TILES)) * 32 + q;
      if (t >= NSUM) break;
      double d = 0.;
      for (int k = lane; k < nblk; k += 64) d += (double)sums[(size_t)t * nblk + k];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) d += __shfl_xor(d, o, 64);
      if (lane == 0) {
        const float g = (float)d;
        const int i = t < S_B2 ? I_B1 + t : (t < S_W3 ? I_B2 + t - S_B2 : I_W3 + t - S_W3);
        if (t == S_LOSS) *loss = g;
        else if (UPDATE) (void)adam_step(ad, i, adam_load(ad, i), g);
        else gout[t < S_B2 ? P_B1 + t : P_B2 + t - S_B2] = g;
      }
    }
    return;
  }
  const bool second = blockIdx.x >= W1_TILES;
  const int tile = second ? blockIdx.x - W1_TILES : blockIdx.x;
  const int tm = second ? 0 : tile % (NH1 / 32), tn = second ? tile : tile / (NH1 / 32);
  // The batch is cut into slices of whole 16-row products, each with an
  // accumulator of its own, and the slices are added four at a time: eight
  // slices (four below 1024 rows) for W1, one a wavefront; up to 128 of at
  // least 128 rows for W2, groups of four a wavefront.  Training follows the
  // rounding of these sums: a BF16 rounding or a ReLU decision that flips is, by
  // Adam, part of a step of a rarely used weight.  With the head's and W2's sums
  // added by FP32 atomics, two runs of 100 steps of 2048 pairs differed by more
  // than 8e-4 in some weight in 56 % of 3600 cases (median of the largest
  // difference 1.3e-3); these sums, nearer to the exact ones, differ from such a
  // run by that in 52 % (9.4e-4), and FP32 sums in ascending order in 58 %.
  const int units = B / 16;
  const int nslice = second ? w2_slices(B) : (B >= 1024 ? 8 : 4);
  const int per = (units + nslice - 1) / nslice;
  // the weights' own state, asked for before the products
  AdamState own[2];
  if (UPDATE) {
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const int e = tid + q * TPB, row = e >> 5, col = e & 31;
      own[q] = adam_load(ad, second ? I_W2T + row * NH1 + 32 * tn + col : I_W1T + (32 * tm + row) * NINP + 32 * tn + col);
    }
  }
  auto slice_end = [&](int u0) { return u0 + per < units ? u0 + per : units; };
  f32x16 acc = {};
  // two sets of eight products' operands take turns: one is loaded while the
  // other is used (16 KB a wavefront in flight; the scheduler would sink the
  // loads to their uses)
  constexpr int SET = 8;
  auto pipeline = [&](int u0, int u1, auto &&load, auto &&use) {
    if (u0 >= u1) return;
    load(0, u0);
    for (int u = u0; u < u1; u += 2 * SET) {
      load(1, u + SET);
      __builtin_amdgcn_sched_barrier(0);
      use(0, u);
      load(0, u + 2 * SET);
      __builtin_amdgcn_sched_barrier(0);
      use(1, u + SET);
    }
  };
  if (second) {
    const u16 *pa = dz2x + lane * 8, *pb = h1x + frag(tn, 0, units) + lane * 8;
    for (int g = w; g < nslice / 4; g += NW) {
      f32x16 group = {};
      for (int q = 0; q < 4; q++) {
        const int u0 = (4 * g + q) * per, u1 = slice_end(u0);
        f32x16 part = {};
        for (int u = u0; u < u1; u += SET) {
          bf16x8 a[SET], b[SET];
#pragma unroll
          for (int j = 0; j < SET; j++) {
            const int t = u + j < u1 ? u + j : u1 - 1;
            a[j] = *(const bf16x8 *)(pa + (size_t)512 * t);
            b[j] = *(const bf16x8 *)(pb + (size_t)512 * t);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int j = 0; j < SET; j++) part = mfma(u + j < u1 ? a[j] : bf16x8{}, b[j], part);
        }
        group += part;
      }
      acc += group;
    }
  } else {
    one_hot_table(hot, tid);
    lds_barrier();
    const u16 *pa = dz1x + frag(tm, 0, units) + lane * 8;
    const u32 *px = bits + 32 * tn + r;
    const int u0 = w * per, u1 = w < nslice ? slice_end(u0) : u0;
    bf16x8 a[2][SET];
    u32 x[2][SET];
    pipeline(
        u0, u1,
        [&](int k, int u) {
#pragma unroll
          for (int j = 0; j < SET; j++) {
            const int t = u + j < u1 ? u + j : u1 - 1;
            a[k][j] = *(const bf16x8 *)(pa + (size_t)512 * t);
            x[k][j] = px[(size_t)(t >> 1) * NINP];
          }
        },
        [&](int k, int u) {
#pragma unroll
          for (int j = 0; j < SET; j++)
            acc = mfma(a[k][j], hot.v[u + j < u1 ? (x[k][j] >> (16 * ((u + j) & 1) + 8 * half)) & 0xFFu : 0u], acc);
        });
  }
#pragma unroll
  for (int i = 0; i < 16; i++) red[w][i][lane] = acc[i];
  lds_barrier();
  // two elements a thread; the row (internal layout) or the column (ABI) runs
  // over the threads' low bits, as their arrays lie in memory
  __shared__ u16 copy[32][34];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const int e = tid + q * TPB;
    const int row = UPDATE ? e >> 5 : e & 31, col = UPDATE ? e & 31 : e >> 5;
    const int i = 4 * (row >> 3) + (row & 3), l = 32 * ((row >> 2) & 1) + col;
    // (the W2 sum, whose order is free, in 64 bits)
    float g = second ? (float)((double)red[0][i][l] + red[1][i][l] + red[2][i][l] + red[3][i][l] + red[4][i][l] +
                               red[5][i][l] + red[6][i][l] + red[7][i][l])
                     : (red[0][i][l] + red[1][i][l] + red[2][i][l] + red[3][i][l]) +
                           (red[4][i][l] + red[5][i][l] + red[6][i][l] + red[7][i][l]);
    if (second) {
      const int o = row, u = 32 * tn + col;
      if (UPDATE) {
        const u16 b = f2bf(adam_step(ad, I_W2T + o * NH1 + u, own[q], g));
        ad.w2t[o * NH1 + u] = b;
        ad.w2[u * NH2 + o] = b;
      } else {
        gout[P_W2 + u * NH2 + o] = g;
      }
    } else {
      const int u = 32 * tm + row, f = 32 * tn + col;
      if (UPDATE) {
        u16 b = 0;  // padded inputs keep zero weights
        if (f < NIN) b = f2bf(adam_step(ad, I_W1T + u * NINP + f, own[q], g));
        ad.w1x[frag_at(u, f, NINP / 16)] = b;
        copy[col][row] = b;
      } else if (f < NIN) {
        gout[P_W1 + f * NH1 + u] = g;
      }
    }
  }
  if (UPDATE && !second) {
    lds_barrier();
    const int col = tid >> 4, row = 2 * (tid & 15);
    *(u32 *)(ad.w1f + (size_t)(32 * tn + col) * NH1 + 32 * tm + row) = *(const u32 *)&copy[col][row];
  }
}

// ABI layout -> master weights and their BF16 copies; master weights -> ABI
__global__ void k_set(const float *__restrict__ in, float *prm, u16 *w1x, u16 *w1f, u16 *w2t, u16 *w2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= NINT) return;
  float p;
  if (i < I_B1) {
    const int u = i / NINP, f = i % NINP;
    p = f < NIN ? in[P_W1 + f * NH1 + u] : 0.f;
    const u16 b = f2bf(p);
    w1x[frag_at(u, f, NINP / 16)] = b;
    w1f[f * NH1 + u] = b;
  } else if (i < I_W2T) {
    p = in[P_B1 + i - I_B1];
  } else if (i < I_B2) {
    const int j = i - I_W2T, o = j / NH1, u = j % NH1;
    p = in[P_W2 + u * NH2 + o];
    const u16 b = f2bf(p);
    w2t[j] = b;
    w2[u * NH2 + o] = b;
  } else {
    p = in[P_B2 + i - I_B2];
  }
  prm[i] = p;
}
__global__ void k_get(const float *__restrict__ prm, float *__restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= NPARAMS) return;
  float p;
  if (i < P_B1) p = prm[I_W1T + (i % NH1) * NINP + i / NH1];
  else if (i < P_W2) p = prm[I_B1 + i - P_B1];
  else if (i < P_B2) p = prm[I_W2T + ((i - P_W2) % NH2) * NH1 + (i - P_W2) / NH2];
  else p = prm[I_B2 + i - P_B2];
  out[i] = p;
}

// BF16 working copies of the master weights
__global__ void k_refresh(const float *__restrict__ prm, u16 *w1x, u16 *w1f, u16 *w2t, u16 *w2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < NH1 * NINP) {
    const u16 b = f2bf(prm[I_W1T + i]);
    const int u = i / NINP, f = i % NINP;
    w1x[frag_at(u, f, NINP / 16)] = b;
    w1f[f * NH1 + u] = b;
  }
  if (i < NH2 * NH1) {
    const u16 b = f2bf(prm[I_W2T + i]);
    w2t[i] = b;
    const int o = i / NH1, u = i % NH1;
    w2[u * NH2 + o] = b;
  }
}

// deterministic initialisation (He-uniform), splitmix64 stream per element
__device__ __forceinline__ float unif(u64 seed, u64 i) {
  u64 z = seed + (i + 1) * 0x9E3779B97F4A7C15ULL;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  z ^= z >> 31;
  return (float)((z >> 40) * (1.0 / 16777216.0)) * 2.f - 1.f;
}
__global__ void k_init(float *prm, u64 seed) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= NINT) return;
  float v = 0.f;
  if (i < I_B1) v = ((i % NINP) < NIN) ? unif(seed, i) * sqrtf(6.f / 40.f) : 0.f;  // ~40 active inputs
  else if (i >= I_W2T && i < I_B2) v = unif(seed, i) * sqrtf(6.f / NH1);
  else if (i >= I_W3 && i < I_B3) v = unif(seed, i) * sqrtf(6.f / NH2);
  prm[i] = v;
}

struct MlpState {
  zr::DevBuf prm, grad, m, v, w1x, w1f, w2t, w2;     // weights
  zr::DevBuf bits, h1x, dz2x, dz1x, sums, loss, recs_scratch;  // a batch
  int cap_pairs = 0;
  bool ready = false;
  int step = 0;
};
MlpState g_ms;

int ensure_weights() {
  int r;
  if ((r = zr::ensure(g_ms.prm, NINT * 4)) || (r = zr::ensure(g_ms.grad, NINT * 4)) ||
      (r = zr::ensure(g_ms.m, NINT * 4)) || (r = zr::ensure(g_ms.v, NINT * 4)) ||
      (r = zr::ensure(g_ms.w1x, NH1 * NINP * 2)) || (r = zr::ensure(g_ms.w1f, NH1 * NINP * 2)) ||
      (r = zr::ensure(g_ms.w2t, NH2 * NH1 * 2)) ||
      (r = zr::ensure(g_ms.w2, NH2 * NH1 * 2)))
    return r;
  return ZETA_OK;
}

int ensure_batch(int P) {
  int r;
  if ((r = zr::ensure(g_ms.loss, 64))) return r;  // (training grows it by itself)
  if (g_ms.cap_pairs >= P) return ZETA_OK;
  const size_t B = 2 * (size_t)P;
  // none until all are there: one that cannot grow is gone
  g_ms.cap_pairs = 0;
  if ((r = zr::ensure(g_ms.h1x, B * NH1 * 2)) || (r = zr::ensure(g_ms.dz1x, B * NH1 * 2)) ||
      (r = zr::ensure(g_ms.bits, B / 32 * NINP * 4)) || (r = zr::ensure(g_ms.dz2x, B * NH2 * 2)) ||
      (r = zr::ensure(g_ms.sums, B / 32 * NSUM * 4)))
    return r;
  g_ms.cap_pairs = P;
  return ZETA_OK;
}

inline unsigned nb(size_t n, int t) { return (unsigned)((n + t - 1) / t); }

// forward and backward of one batch of P pairs (nrec = 0: the first P records;
// nrec > 0: drawn from nrec records with seed); `ad` given: Adam with the
// gradients, else the gradients into gout in the ABI's layout.  The mean loss
// goes to *loss.
int step(const PairRec *recs, int P, u64 nrec, u64 seed, const Adam *ad, float *gout, float *loss) {
  const int B = 2 * P;
  const unsigned tiles = W1_TILES + W2_TILES + SUM_BLOCKS;
  ZLAUNCH(zr::K_MLP_FWD, B, k_rows, B / 32, TPB, 0, recs, B, nrec, seed, (const float *)g_ms.prm.p,
          (const u16 *)g_ms.w1x.p, (const u16 *)g_ms.w2t.p, (const u16 *)g_ms.w2.p, (u32 *)g_ms.bits.p,
          (u16 *)g_ms.h1x.p, (u16 *)g_ms.dz2x.p, (u16 *)g_ms.dz1x.p, (float *)g_ms.sums.p);
  if (ad)
    ZLAUNCH(zr::K_MLP_BWD, B, k_weights<true>, tiles, TPB, 0, B, (const u32 *)g_ms.bits.p, (const u16 *)g_ms.h1x.p,
            (const u16 *)g_ms.dz2x.p, (const u16 *)g_ms.dz1x.p, (const float *)g_ms.sums.p, *ad, (float *)nullptr, loss);
  else
    ZLAUNCH(zr::K_MLP_BWD, B, k_weights<false>, tiles, TPB, 0, B, (const u32 *)g_ms.bits.p, (const u16 *)g_ms.h1x.p,
            (const u16 *)g_ms.dz2x.p, (const u16 *)g_ms.dz1x.p, (const float *)g_ms.sums.p, Adam{}, gout, loss);
  return ZETA_OK;
}

int refresh() {
  ZLAUNCH(zr::K_MLP_ADAM, NH1 * NINP, k_refresh, nb((size_t)NH1 * NINP, 256), 256, 0, (const float *)g_ms.prm.p,
          (u16 *)g_ms.w1x.p, (u16 *)g_ms.w1f.p, (u16 *)g_ms.w2t.p, (u16 *)g_ms.w2.p);
  return ZETA_OK;
}

}  // namespace

// ---- records (training pairs) shared with the search kernel
namespace zrec {
zr::DevBuf g_recs, g_count;
u64 g_cap = 0;
int ensure(u64 cap) {
  int r;
  if ((r = zr::ensure(g_count, 64))) return r;
  if (g_cap >= cap && g_recs.p) return ZETA_OK;
  // keep already logged pairs when growing
  u64 n = 0;
  if (g_recs.p) {
    ZCHECK(hipMemcpyAsync(&n, g_count.p, 8, hipMemcpyDeviceToHost, zr::ctx().stream));
    ZCHECK(hipStreamSynchronize(zr::ctx().stream));
  }
  zr::DevBuf nb2;
  if ((r = zr::ensure(nb2, cap * sizeof(PairRec)))) return r;
  if (g_recs.p && n) {
    // the count runs on past the capacity (the search counts the pairs it
    // could not store): keep what the old buffer holds, and count that
    u64 keep = n < g_cap ? n : g_cap;
    if (keep > cap) keep = cap;
    ZCHECK(hipMemcpyAsync(nb2.p, g_recs.p, keep * sizeof(PairRec), hipMemcpyDeviceToDevice, zr::ctx().stream));
    ZCHECK(hipMemcpyAsync(g_count.p, &keep, 8, hipMemcpyHostToDevice, zr::ctx().stream));
    ZCHECK(hipStreamSynchronize(zr::ctx().stream));
  } else {
    ZCHECK(hipMemsetAsync(g_count.p, 0, 8, zr::ctx().stream));
  }
  zr::release(g_recs);
  g_recs = nb2;
  g_cap = cap;
  return ZETA_OK;
}
}  // namespace zrec

void *records_buffer(u64 *cap, u64 **count) {
  *cap = zrec::g_cap;
  *count = (u64 *)zrec::g_count.p;
  return zrec::g_recs.p;
}

const zm::Weights *mlp_weights() {
  static zm::Weights w;
  if (!g_ms.ready) return nullptr;
  const float *prm = (const float *)g_ms.prm.p;
  w.w1f = (const u16 *)g_ms.w1f.p;
  w.w2t = (const u16 *)g_ms.w2t.p;
  w.b1 = prm + I_B1;
  w.b2 = prm + I_B2;
  w.w3 = prm + I_W3;
  w.b3 = prm + I_B3;
  return &w;
}

void mlp_release() {
  zr::DevBuf *bufs[] = {&g_ms.prm,  &g_ms.grad, &g_ms.m,    &g_ms.v,    &g_ms.w1x,  &g_ms.w1f,  &g_ms.w2t,         &g_ms.w2,
                        &g_ms.bits, &g_ms.h1x,  &g_ms.dz2x, &g_ms.dz1x, &g_ms.sums, &g_ms.loss, &g_ms.recs_scratch};
  for (auto *b : bufs) zr::release(*b);
  g_ms.cap_pairs = 0;
  g_ms.ready = false;
  zr::release(zrec::g_recs);
  zr::release(zrec::g_count);
  zrec::g_cap = 0;
}

extern "C" int zeta_mlp_init(uint64_t seed) {
  int r = zr::require_up();
  if (r) return r;
  if ((r = ensure_weights())) return r;
  hipStream_t st = zr::ctx().stream;
  ZLAUNCH(zr::K_MLP_ADAM, NINT, k_init, nb(NINT, 256), 256, 0, (float *)g_ms.prm.p, (u64)seed);
  ZCHECK(hipMemsetAsync(g_ms.m.p, 0, NINT * 4, st));
  ZCHECK(hipMemsetAsync(g_ms.v.p, 0, NINT * 4, st));
  if ((r = refresh())) return r;
  ZCHECK(hipStreamSynchronize(st));
  zr::time_collect();
  g_ms.step = 0;
  g_ms.ready = true;
  return ZETA_OK;
}

extern "C" int zeta_mlp_set(const float *params, size_t n) {
  int r = zr::require_up();
  if (r) return r;
  if (!params || n != (size_t)NPARAMS) return zr::fail(ZETA_EINVAL, "zeta_mlp_set: expected %d floats", NPARAMS);
  if ((r = ensure_weights())) return r;
  hipStream_t st = zr::ctx().stream;
  ZCHECK(hipMemcpyAsync(g_ms.grad.p, params, (size_t)NPARAMS * 4, hipMemcpyHostToDevice, st));
  ZLAUNCH(zr::K_MLP_ADAM, NINT, k_set, nb(NINT, 256), 256, 0, (const float *)g_ms.grad.p, (float *)g_ms.prm.p,
          (u16 *)g_ms.w1x.p, (u16 *)g_ms.w1f.p, (u16 *)g_ms.w2t.p, (u16 *)g_ms.w2.p);
  ZCHECK(hipMemsetAsync(g_ms.m.p, 0, NINT * 4, st));
  ZCHECK(hipMemsetAsync(g_ms.v.p, 0, NINT * 4, st));
  ZCHECK(hipStreamSynchronize(st));
  zr::time_collect();
  g_ms.step = 0;
  g_ms.ready = true;
  return ZETA_OK;
}

extern "C" int zeta_mlp_get(float *params, size_t n) {
  int r = zr::require_up();
  if (r) return r;
  if (!g_ms.ready) return zr::fail(ZETA_ESTATE, "zeta_mlp_get: no network (zeta_mlp_init / zeta_mlp_set first)");
  if (!params || n != (size_t)NPARAMS) return zr::fail(ZETA_EINVAL, "zeta_mlp_get: expected %d floats", NPARAMS);
  ZLAUNCH(zr::K_MLP_ADAM, NPARAMS, k_get, nb(NPARAMS, 256), 256, 0, (const float *)g_ms.prm.p, (float *)g_ms.grad.p);
  ZCHECK(hipMemcpyAsync(params, g_ms.grad.p, (size_t)NPARAMS * 4, hipMemcpyDeviceToHost, zr::ctx().stream));
  ZCHECK(hipStreamSynchronize(zr::ctx().stream));
  zr::time_collect();
  return ZETA_OK;
}

// gradient of one batch without an update (ABI layout), for gradient checks
extern "C" int zeta_mlp_grad(const void *pairs, int npairs, float *loss, float *grads, size_t n) {
  int r = zr::require_up();
  if (r) return r;
  if (!g_ms.ready) return zr::fail(ZETA_ESTATE, "zeta_mlp_grad: no network");
  if (!pairs || npairs <= 0 || npairs % 16 != 0 || !grads || n != (size_t)NPARAMS)
    return zr::fail(ZETA_EINVAL, "zeta_mlp_grad: npairs must be a positive multiple of 16");
  if ((r = ensure_batch(npairs)) || (r = zr::ensure(g_ms.recs_scratch, (size_t)npairs * sizeof(PairRec))))
    return r;
  hipStream_t st = zr::ctx().stream;
  ZCHECK(hipMemcpyAsync(g_ms.recs_scratch.p, pairs, (size_t)npairs * sizeof(PairRec), hipMemcpyHostToDevice, st));
  if ((r = step((const PairRec *)g_ms.recs_scratch.p, npairs, 0, 0, nullptr, (float *)g_ms.grad.p, (float *)g_ms.loss.p)))
    return r;
  float l = 0.f;
  ZCHECK(hipMemcpyAsync(grads, g_ms.grad.p, (size_t)NPARAMS * 4, hipMemcpyDeviceToHost, st));
  ZCHECK(hipMemcpyAsync(&l, g_ms.loss.p, 4, hipMemcpyDeviceToHost, st));
  ZCHECK(hipStreamSynchronize(st));
  zr::time_collect();
  if (loss) *loss = l;
  return ZETA_OK;
}

// Adam training on the logged pairs; losses[i] = mean loss of step i
extern "C" int zeta_mlp_train(int steps, int pairs_per_step, float lr, uint64_t seed, float *losses) {
  int r = zr::require_up();
  if (r) return r;
  if (!g_ms.ready) return zr::fail(ZETA_ESTATE, "zeta_mlp_train: no network (zeta_mlp_init first)");
  if (steps < 0 || pairs_per_step <= 0 || pairs_per_step % 16 != 0)
    return zr::fail(ZETA_EINVAL, "zeta_mlp_train: pairs_per_step must be a positive multiple of 16");
  u64 nrec = 0;
  if (zrec::g_count.p) {
    ZCHECK(hipMemcpyAsync(&nrec, zrec::g_count.p, 8, hipMemcpyDeviceToHost, zr::ctx().stream));
    ZCHECK(hipStreamSynchronize(zr::ctx().stream));
  }
  if (nrec > zrec::g_cap) nrec = zrec::g_cap;
  if (nrec == 0) return zr::fail(ZETA_ESTATE, "zeta_mlp_train: no logged training pairs");
  if ((r = ensure_batch(pairs_per_step)) || (r = zr::ensure(g_ms.loss, (size_t)steps * 4))) return r;
  hipStream_t st = zr::ctx().stream;
  Adam ad;
  ad.lr = lr;
  ad.b1 = 0.9f;
  ad.b2 = 0.999f;
  ad.eps = 1e-8f;
  ad.prm = (float *)g_ms.prm.p;
  ad.m = (float *)g_ms.m.p;
  ad.v = (float *)g_ms.v.p;
  ad.w1x = (u16 *)g_ms.w1x.p;
  ad.w1f = (u16 *)g_ms.w1f.p;
  ad.w2t = (u16 *)g_ms.w2t.p;
  ad.w2 = (u16 *)g_ms.w2.p;
  for (int s = 0; s < steps; s++) {
    g_ms.step++;
    ad.c1 = 1.f - powf(ad.b1, (float)g_ms.step);
    ad.c2 = 1.f - powf(ad.b2, (float)g_ms.step);
    if ((r = step((const PairRec *)zrec::g_recs.p, pairs_per_step, nrec, (u64)seed + (u64)s * 0xD1B54A32D192ED03ULL, &ad,
                  nullptr, (float *)g_ms.loss.p + s)))
      return r;
  }
  if (losses && steps) ZCHECK(hipMemcpyAsync(losses, g_ms.loss.p, (size_t)steps * 4, hipMemcpyDeviceToHost, st));
  ZCHECK(hipStreamSynchronize(st));
  zr::time_collect();
  return ZETA_OK;
}

extern "C" int zeta_records_reserve(uint64_t capacity) {
  int r = zr::require_up();
  if (r) return r;
  if (capacity == 0) return zr::fail(ZETA_EINVAL, "zeta_records_reserve: capacity 0");
  return zrec::ensure(capacity);
}

extern "C" int zeta_records_count(uint64_t *n) {
  int r = zr::require_up();
  if (r) return r;
  if (!n) return ZETA_EINVAL;
  *n = 0;
  if (!zrec::g_count.p) return ZETA_OK;
  ZCHECK(hipMemcpyAsync(n, zrec::g_count.p, 8, hipMemcpyDeviceToHost, zr::ctx().stream));
  ZCHECK(hipStreamSynchronize(zr::ctx().stream));
  if (*n > zrec::g_cap) *n = zrec::g_cap;
  return ZETA_OK;
}

extern "C" int zeta_records_clear(void) {
  int r = zr::require_up();
  if (r) return r;
  if (!zrec::g_count.p) return ZETA_OK;
  ZCHECK(hipMemsetAsync(zrec::g_count.p, 0, 8, zr::ctx().stream));
  ZCHECK(hipStreamSynchronize(zr::ctx().stream));
  return ZETA_OK;
}

extern "C" int zeta_records_get(void *out, uint64_t max, uint64_t *n) {
  int r = zr::require_up();
  if (r) return r;
  u64 have = 0;
  if ((r = zeta_records_count(&have))) return r;
  const u64 k = have < max ? have : max;
  if (n) *n = k;
  if (k && !out) return ZETA_EINVAL;
  if (k) {
    ZCHECK(hipMemcpyAsync(out, zrec::g_recs.p, k * sizeof(PairRec), hipMemcpyDeviceToHost, zr::ctx().stream));
    ZCHECK(hipStreamSynchronize(zr::ctx().stream));
  }
  return ZETA_OK;
}

extern "C" int zeta_records_put(const void *in, uint64_t n) {
  int r = zr::require_up();
  if (r) return r;
  if (n && !in) return ZETA_EINVAL;
  if ((r = zrec::ensure(n ? n : 1))) return r;
  if (n) ZCHECK(hipMemcpyAsync(zrec::g_recs.p, in, n * sizeof(PairRec), hipMemcpyHostToDevice, zr::ctx().stream));
  ZCHECK(hipMemcpyAsync(zrec::g_count.p, &n, 8, hipMemcpyHostToDevice, zr::ctx().stream));
  ZCHECK(hipStreamSynchronize(zr::ctx().stream));
  return ZETA_OK;
}
