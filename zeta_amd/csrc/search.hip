// search.hip -- batched fixed-depth alpha-beta + quiescence on gfx950.
//
// Replaces alphabeta_gpu (src/zeta.cl:852-2512) and its host driver
// rootsearch (src/search.c:35-223), for many root positions per launch.
//
// Execution model: one wavefront = one worker; a persistent grid of workers
// takes root positions from a queue and, once the queue is empty, joins
// unfinished roots as ABDADA helpers (busy siblings deferred to a second pass,
// src/zeta.cl:1648-1717).  The first worker to finish a root's last
// iteration publishes its score; the others abandon that root.
// Per worker, the depth-first stack lives in LDS: one Ply record per ply and a
// move stack.  Node control is wave-uniform (every lane holds the same
// values); lanes split the per-node work:
//   * move generation: lane = square, each lane enumerates its piece's legal
//     targets; a wave prefix sum compacts them into the LDS move stack;
//   * move selection: wave arg-max over the node's remaining moves
//     (score, then lowest slot, so runs are deterministic per worker);
//   * evaluation: lane = square (src/zeta.cl:1482-1531), wave sum.
//
// Node semantics follow alphabeta_gpu with null move, LMR and IID off:
// check / queen-promotion extension (src/zeta.cl:1330-1345), quiescence at
// depth <= 0 with captures + e.p. only and stand pat when not in check,
// mate = -INF+ply only outside quiescence, stalemate 0, in-path repetition,
// fifty-move and bare-king draws below the root, MAXPLY cut, fail-hard
// window propagation, root score = PV[0] semantics.
//
// Transposition table (2^k entries x 16 B in HBM, lockless: word0 =
// key ^ word1): every entry supplies the move ordering's TT move; its score
// is used only when it cannot change the root value: at the same depth, with
// the exact castle squares in the key, and where neither the storing nor the
// probing path can repeat a position above the node (path_free).
#include <string.h>

#include "bounds.h"
#include "chess.h"
#include "evaltab.h"
#include "mlp.h"
#include "runtime.h"
#include "wave.h"

using namespace zc;

namespace {

constexpr int MAXPLY = 64;  // src/types.h:76
constexpr s32 INF = 32000;
constexpr s32 MATESCORE = 30000;
constexpr int MSTACK = 1024;  // move-stack slots per worker (LDS)
// Slots past them for moves not yet tested for legality: a list whose legal moves
// fit must fit before the test too.  No position of a game has 256 moves, legal or
// not; eight workers a CU have room for them.
constexpr int MPAD = 256;
// A move-list entry is a move code and a key: the ordering score + 32768 in the
// upper half (0: the move was searched), in the lower half what is known of
// the child, if it is a quiescence node: KEY_CHECK, KEY_OPEN, or its static
// evaluation for the side to move + 32768.
constexpr u32 KEY_CHECK = 0;  // in check
constexpr u32 KEY_OPEN = 1;   // nothing known
__device__ __forceinline__ u32 move_key(s32 score, u32 child) { return ((u32)(score + 32768) << 16) | child; }
constexpr s32 TTMOVE_SCORE = 32000;  // above every other score (src/zeta.cl:2101)
constexpr s32 HINT_SCORE = 32100;    // the hint table's move, above the TT move
// the killer (one per ply) and the counter move (indexed by the previous
// move's squares), quiet moves only: src/zeta.cl:2073-2082
constexpr s32 KILLER_SCORE = 1400;
constexpr s32 COUNTER_SCORE = 1300;
// counter-move table entries per worker: in device memory (its 8 KB would take
// two of eight workers' room in LDS), read once a node, ahead of its use
constexpr int NCOUNTER = 64 * 64;
constexpr u32 DEFERRED = 0x80000000u;  // move-stack flag: deferred by ABDADA (move codes use bits 0-29)
constexpr u32 MOVE_BITS = 0x3FFFFFFFu;
// Default split depth (zeta_search_opts.split_depth), by workers per root: from
// 16 on, workers meet at the nodes next to quiescence often enough that marking
// those pays too (16 positions, depth 4: 229 ms with 1, 290 with 2 at 32
// workers; one position, depth 5, 128 workers: 206, 229, and 278 with 3).  Up
// to 8, single positions take 2-4 % longer with 1 (batches 10 % less), and a
// root's nodes spread over its workers, so that per-worker node budgets end a
// search later than they did.
inline int default_split(int workers) { return workers >= 16 ? 1 : 2; }
constexpr int POLL_EVERY = 64;

typedef u32 u32x4 __attribute__((ext_vector_type(4)));  // one 16-byte TT entry

// The quiescence table.  A quiescence node's value is a function of its pieces
// and side to move alone (captures only, no repetition, no castling), so the
// captures of a position in another order, the other workers of a root and its
// next iteration meet it again: three quarters of a search's time went into
// quiescence trees, and trees of 10^5 nodes below one node kept a worker busy
// after all others had ended.  An entry is 8 bytes, read and written whole: the
// key's bits above QT_BITS (those below are in the index, of at least QT_BITS
// bits, so that no two keys share an entry), the kind of bound (Q_LOWER ..
// Q_EXACT), the value.
// It starts empty in every call.  1024 positions, depth 4, 128 workers each:
// 373 -> 151 ms (1057 -> 251 ms for a batch with one root of 89 M nodes); one
// position, depth 5: 52 -> 45 ms.
constexpr int QT_BITS = 18;
constexpr u64 QT_MIN = 1ULL << QT_BITS, QT_MAX = 1ULL << 22, QT_WORKER = 4096;  // entries: least, most, per worker

// ---- serving (zeta_serve_*): the host publishes requests in coherent pinned
// host memory; a persistent grid of workers claims them in ticket order,
// helps running ones (ABDADA) when idle, and writes results back there.
struct ServeReq {  // 80 B
  u64 pos[8];      // zeta_pos
  s32 depth;
  s32 flags;       // bit 0: learned ordering
  s32 workers;     // at most this many workers on the request
  s32 pad;
};
struct ServeSlot {  // 128 B, pinned host memory
  ServeReq req;     // written by the host before the ticket is published
  s32 score;        // results, written by the device
  u32 bestmove;
  u64 nodes;
  u64 ticket;       // ticket + 1 of the result
  s32 depth_done;
  s32 status;       // SV_DONE / SV_FAILED / SV_CANCELLED
  u32 state;        // 0 -> 1 when the result is complete (device store, host clears)
  u32 pad[3];
};
struct ServeHost {  // pinned host memory header, then u64 queue[qcap], ack[qcap], cancel[nslots]
  u64 submitted;    // tickets published; ticket t names slot queue[t % qcap]
  u64 heartbeat;    // bumped by every host call (watchdog)
  u32 shutdown;
  u32 cancel_gen;   // bumped when cancel[] changes
  u32 pad[10];
};
struct ServeDev {  // device memory; mirrors of the host words, written by the scheduler wavefront
  u64 claimed;     // tickets claimed by workers
  u64 sub;         // mirror of ServeHost::submitted
  u32 shut;        // 1 shutdown, 2 watchdog, 3 protocol error
  u32 exit_xcc;    // diagnostics of a watchdog / protocol exit
  u64 exit_now;
  u64 exit_arg;
};
// slot word (device): ticket+1 << 24 | max workers << 16 | workers << 2 | status
enum { SV_RUN = 0, SV_DONE = 1, SV_FAILED = 2, SV_CANCELLED = 3 };

// batch counters (device, summed per worker at the end of each root)
struct SearchArgs {
  const u64 *roots;  // zeta_pos[n]
  int nroots;
  int depth;
  int workers;       // at most this many workers on one root
  int split_depth;   // ABDADA deferral / busy marking at depth - 1 >= split_depth
  u64 *tt;           // 2 words per entry
  u64 ttmask;        // entries - 1 (0 = no TT)
  u64 *qtt;          // quiescence table, 8 bytes an entry (qt_store), where there is a TT
  u64 qmask;         // its entries - 1
  const u64 *hint;   // read-only table in the TT's format whose moves go first (null = none)
  u64 *rbound;       // per root (slot): best root score so far, ticket << 32 | iteration << 16 | score + 32768
  u32 *busy;
  u32 busymask;
  u16 *ctab;          // counter moves, NCOUNTER per worker (block)
  int *queue;
  u32 *done;
  int *nworkers;
  s32 *score;
  u32 *bestmove;
  u64 *nodes;
  s32 *depth_done;
  u32 *err;
  const u32 *habort;  // abort word in coherent pinned host memory (zeta_search_abort)
  u64 max_nodes;  // per worker and root (0 = none)
  u64 *ctr;       // batch counters, see zeta_search_counters
  // learned ordering
  int use_mlp;
  int mlp_min_depth;
  zm::Weights w;
  // training-pair log (cut nodes): PairRec[cap], counter
  u64 *recs;
  u64 *rec_count;
  u64 rec_cap;
  u32 rec_mask;  // a cut node is logged when (hash >> 40) & rec_mask == 0
  // game history before each root, newest first (ZETA_HISTORY per root)
  const u64 *hist;
  const s32 *hlen;
  // serving mode (slots != nullptr)
  ServeHost *sh;
  const u64 *squeue;  // host: slot of ticket t at [t % qcap]
  u64 *sack;          // host: ticket + 1 once claimed
  const u64 *scancel; // host: ticket + 1 to cancel, per slot
  ServeSlot *slots;   // host
  int nslots;
  int qcap;
  ServeDev *sv;       // device
  u64 *sw;            // device slot words
  ServeReq *dreq;     // device copies of the claimed requests
  u64 *dres;          // per slot: score | best move << 32 of the worker that completed the request
  u64 *dcancel;       // device mirror of scancel
  u64 watchdog_ticks; // wall-clock ticks without a heartbeat before the grid exits (0 = never)
};

// The kernel's arguments, read from the kernarg segment where they are used:
// held in registers through the search they take 120 of the 102 scalar
// registers a wavefront has, and the compiler then keeps them in vector lanes
// (270 spilled registers in k_search, a v_readlane at every use).  The empty
// asm hides where the pointer comes from, so that a load stays behind it.
typedef const __attribute__((address_space(4))) SearchArgs *Args;
__device__ __forceinline__ Args args() {
  Args p = (Args)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}

// a pointer read from the arguments, known to point to device memory (an
// address the compiler cannot place costs the slower flat access)
template <class T>
__device__ __forceinline__ T *glob(T *p) {
  return (T *)(__attribute__((address_space(1))) T *)p;
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Entries of the tables are written and read at agent scope: the chiplets' L2s do
// not see each other's lines, and with plain accesses workers on different
// chiplets shared next to nothing. (One position, depth 5: four workers made 3.7
// times the nodes of one and were 5 % faster, now 1.6 times and 2.3 times as
// fast; six positions with 128 workers 182 -> 113 ms.)
// A search with a node budget per worker shares less: plain accesses, no
// quiescence table, no entries by path, full windows.  Its workers make about
// the nodes they made before all that, so that the same budgets stop the same
// searches (with it, a root of 30000 nodes over 8 workers ends within 2000 each).
// The engine's moves, whose clock is a node budget, run this one.
enum { T_NONE = 0, T_SHARED, T_BUDGET };  // a search's tables
__device__ __forceinline__ u64 shared_load(const u64 *p) {
  return __hip_atomic_load(glob(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void shared_store(u64 *p, u64 v) {
  __hip_atomic_store(glob(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <int TABLE>
__device__ __forceinline__ u32x4 tt_load(const u64 *p) {
  if (TABLE == T_BUDGET) return *glob((const u32x4 *)p);
  const u64 a = shared_load(p), b = shared_load(p + 1);
  return u32x4{(u32)a, (u32)(a >> 32), (u32)b, (u32)(b >> 32)};
}

enum { C_TT_PROBE = 0, C_TT_HIT, C_TT_CUT, C_TT_STORE, C_DEFER, C_MAXPLY, C_MLP_NODES, C_RECORDS, C_NODES, C_NCTR = 16 };

__device__ __forceinline__ void wsync() { __syncthreads(); }  // one wave per block

// Wave-uniform values: readfirstlane puts them in SGPRs, so the node logic
// (position analysis, window and TT bookkeeping) runs on the scalar unit.
__device__ __forceinline__ u32 uf(u32 v) { return (u32)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ s32 uf(s32 v) { return (s32)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ u64 uf(u64 v) { return ((u64)uf((u32)(v >> 32)) << 32) | (u64)uf((u32)v); }

// add v to statistics counter k, held in lane k of a vector register
__device__ __forceinline__ void lcount(u32 &cvec, int k, u32 v) { cvec += (threadIdx.x == (unsigned)k) ? v : 0u; }
__device__ __forceinline__ s32 wave_sum_i(s32 v) {
  return (s32)__builtin_amdgcn_readlane(zw::wave_scan_add(v), 63);
}
__device__ __forceinline__ u32 wave_max_u32(u32 v) {
  return (u32)__builtin_amdgcn_readlane((int)zw::wave_scan_max(v), 63);
}

// TT / busy-table key: the reference hash plus the exact castle squares
// (a1 e1 h1 a8 e8 h8, bits 0 4 7 56 60 63 of the moved-flags word), folded
// into 16 bits and spread by one multiplication by an odd constant (17
// fewer scalar instructions per node than a full 64-bit mix, about 1 % of a
// node's time)
__device__ __forceinline__ u64 tt_key(u64 hash, u64 cr) {
  const u64 c = cr & 0x9100000000000091ULL;
  const u32 x = (u32)c | (u32)(c >> 48);
  return hash ^ ((u64)x * 0x9E3779B97F4A7C15ULL);
}

__device__ __forceinline__ bool is_mate(s32 v) { return (v > MATESCORE && v < INF) || (v < -MATESCORE && v > -INF); }

__device__ __forceinline__ bool is_promo(u32 m) {
  return m && ((mv_pfrom(m) >> 1) & 7) == PAWN && ((mv_pto(m) >> 1) & 7) == QUEEN;
}

struct Node {  // the current full-width node (wave-uniform)
  Pos p;
  u64 hash, phash;
  s32 alpha, beta, depth;
  u32 move, best, ttm;
  int mbeg, mcnt;
  u64 left;         // moves not searched yet (lists of up to 64)
  u32 hmc;
  bool kic, pass2;  // in check; second pass (deferred moves)
  int ndefer, searched;
  bool busy;
  u32 reach;        // see path_free
  bool scout;       // the move being searched has a window of one above `floor`
  s32 floor;
  u32 child;        // what its key says of the child
};

// child hash of the alpha-beta move-up (src/zeta.cl:2297-2359), incremental
__device__ __forceinline__ void child_hash(const Node &n, u32 m, const Pos &c, u64 &hash, u64 &phash) {
  const int f = (int)mv_from(m), t = (int)mv_to(m), x = (int)mv_cpt(m);
  const u32 pf = mv_pfrom(m), pt = mv_pto(m), pc = mv_pcpt(m);
  u64 ph = n.phash ^ piece_key(pf, f) ^ piece_key(pt, t);
  if (((pc >> 1) & 7) != PNONE) ph ^= piece_key(pc, x);
  if (((pf >> 1) & 7) == KING && (f - t == 2 || t - f == 2)) {
    const u32 rook = (ROOK << 1) | (pf & 1);
    const int rf = (f - t == 2) ? f - 4 : f + 3, rt = (f - t == 2) ? t + 1 : t - 1;
    ph ^= piece_key(rook, rf) ^ piece_key(rook, rt);
  }
  u64 h = ph;
  const u32 col = pf & 1;
  const int rfr = col ? ((f >> 3) ^ 7) : (f >> 3), rto = col ? ((t >> 3) ^ 7) : (t >> 3);
  if (((pf >> 1) & 7) == PAWN && rto - rfr == 2) h ^= rotl(ZOBRIST[16], t & 7);
  if (c.stm) h ^= 1ULL;
  h ^= hash_castle(c.cr);
  hash = h;
  phash = ph;
}

__device__ __forceinline__ u32 child_hmc(u32 hmc, u32 m) {
  // src/zeta.cl:2362-2373 (8-bit counter)
  const u32 pf = mv_pfrom(m);
  const int f = (int)mv_from(m), t = (int)mv_to(m);
  if (((pf >> 1) & 7) == PAWN || ((mv_pcpt(m) >> 1) & 7) != PNONE) return 0;
  if (((pf >> 1) & 7) == KING && (f - t == 2 || t - f == 2)) return 0;
  return (hmc + 1) & 0xFF;
}

// least depth of nodes that are looked up under their path too (below, most
// bounds hold on any path)
constexpr int PATH_DEPTH = 2;

enum { S_ENTER = 0, S_NEXT, S_RETURN, S_QS };

// The value a move of the node has to exceed.  At the root that is the best of
// all workers less one (ra - 1), not this worker's own: a worker that starts on
// a root move with no score of its own would look at every reply to it (six
// batches of 1024 positions, depth 4: 770 -> 698 ms).
__device__ __forceinline__ s32 floor_of(const Node &n, int sd, s32 ra) {
  return sd == 1 && ra - 1 > n.alpha ? ra - 1 : n.alpha;
}

// A counter move is a quiet move, which its from- and to-square and its
// piece determine (sqcpt = to, no captured piece, pto = pfrom or the queen a
// pawn on the last rank becomes): 16 bits hold it, and a quiet candidate
// equals the stored move exactly when its 16 bits do (a capture never does,
// as in the reference's full-code comparison, src/zeta.cl:2072)
__device__ __forceinline__ u16 counter_code(u32 m) { return (u16)((m & 0xFFFu) | (mv_pfrom(m) << 12)); }
__device__ __forceinline__ int counter_index(u32 prev) { return (int)(mv_from(prev) * 64 + mv_to(prev)); }

__device__ __forceinline__ void busy_release(Args a, u64 hash, u64 cr, int lane) {
  const u32 bidx = (u32)(tt_key(hash, cr) >> 40) & a->busymask;
  if (lane == 0) atomicSub(&a->busy[bidx], 1u);
}

// next root for this worker: the queue first, then the unfinished root with
// the fewest workers (ABDADA helper), at most a->workers per root
// A worker takes the next unstarted root; once all have started it joins,
// as an ABDADA helper below the per-root limit, the unfinished root with the
// fewest completed iterations (the most work left: an iteration costs
// several times the one before it), then the fewest workers.  The wave's
// lanes scan the roots together and agree on the minimum.
__device__ int pick_root(Args a, int hstart, int lane) {
  int r = 0;
  if (lane == 0) r = atomicAdd(a->queue, 1);
  r = uf(r);
  if (r < a->nroots) {
    if (lane == 0) atomicAdd(&a->nworkers[r], 1);
    return r;
  }
  if (a->workers <= 1) return -1;
  for (int attempt = 0; attempt < 8; attempt++) {
    u64 best = ~0ULL;  // (iterations done << 48) | (workers << 32) | root
    for (int k = lane; k < a->nroots; k += 64) {
      const int rr = (hstart + k) % a->nroots;
      if (__atomic_load_n(&a->done[rr], __ATOMIC_RELAXED)) continue;
      const int w = __atomic_load_n(&a->nworkers[rr], __ATOMIC_RELAXED);
      if (w >= a->workers) continue;
      const int dd = __atomic_load_n(&a->depth_done[rr], __ATOMIC_RELAXED);
      const u64 key = ((u64)(dd < 0 ? 0 : (dd > 255 ? 255 : dd)) << 48) | ((u64)(u32)w << 32) | (u32)rr;
      best = key < best ? key : best;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const u64 other = ((u64)(u32)__shfl_xor((int)(u32)(best >> 32), o, 64) << 32) |
                        (u32)__shfl_xor((int)(u32)best, o, 64);
      best = other < best ? other : best;
    }
    best = uf(best);
    if (best == ~0ULL) return -1;
    const int pick = (int)(u32)best;
    int got = 0;
    if (lane == 0) {
      got = atomicAdd(&a->nworkers[pick], 1) < a->workers ? 1 : 0;
      if (!got) atomicSub(&a->nworkers[pick], 1);
    }
    if (uf(got)) return pick;
  }
  return -1;
}

__device__ __forceinline__ void add_row(float x[8], const u16 *row) {
  const uint4 q = *(const uint4 *)row;  // 8 BF16
  const u32 v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
  for (int j = 0; j < 4; j++) {
    x[2 * j] += zm::bf2f((u16)(v[j] & 0xFFFF));
    x[2 * j + 1] += zm::bf2f((u16)(v[j] >> 16));
  }
}

// Learned ordering: network score of every move of the node (moves
// [mbeg, mbeg+total) in LDS) given to out(slot, score), once each.  Layer 1's position part is
// accumulated once (lane = 4 hidden units); each chunk of 32 moves then runs
// layer 2 as 16 MFMA steps whose A operand (move x 8 hidden units, BF16) is
// built in registers from the position part plus the move's 3-4 feature rows.
template <class Out>
__device__ void mlp_score_moves(Args a, const Pos &p, int mbeg, int total, int lane, float *hpos,
                                const u32 *mmove, Out &&out) {
  const u16 *const w1f = a->w.w1f, *const w2t = a->w.w2t;
  const float *const wb1 = a->w.b1;
  float h4[4];
#pragma unroll
  for (int j = 0; j < 4; j++) h4[j] = wb1[lane * 4 + j];
  u64 occ = p.b1 | p.b2 | p.b3;
  while (occ) {
    const int sq = lsb(occ);
    occ &= occ - 1;
    const int f = zm::feat_ps(piece_at(p, sq), sq, p.stm);
    const uint2 q = *(const uint2 *)(w1f + (size_t)f * zm::NH1 + lane * 4);
    h4[0] += zm::bf2f((u16)(q.x & 0xFFFF));
    h4[1] += zm::bf2f((u16)(q.x >> 16));
    h4[2] += zm::bf2f((u16)(q.y & 0xFFFF));
    h4[3] += zm::bf2f((u16)(q.y >> 16));
  }
#pragma unroll
  for (int j = 0; j < 4; j++) hpos[lane * 4 + j] = h4[j];
  wsync();
  const int col = lane & 31, half = lane >> 5;
  const float b2o = a->w.b2[col], w3o = a->w.w3[col], b3 = a->w.b3[0];
  for (int c0 = 0; c0 < total; c0 += 32) {
    const int mi = c0 + col;
    const u32 m = mi < total ? mmove[mbeg + mi] : 0u;
    const int ff = m ? zm::feat_from(m, p.stm) : 0, ft = m ? zm::feat_to(m, p.stm) : 0;
    const int fp = m ? zm::feat_piece(m) : 0, fc = m ? zm::feat_capt(m) : -1;
    f32x16 acc = {};
    for (int ks = 0; ks < zm::NH1 / 16; ks++) {
      const int kb = ks * 16 + half * 8;
      float x[8];
#pragma unroll
      for (int j = 0; j < 8; j++) x[j] = hpos[kb + j];
      if (m) {
        add_row(x, w1f + (size_t)ff * zm::NH1 + kb);
        add_row(x, w1f + (size_t)ft * zm::NH1 + kb);
        add_row(x, w1f + (size_t)fp * zm::NH1 + kb);
        if (fc >= 0) add_row(x, w1f + (size_t)fc * zm::NH1 + kb);
      }
      bf16x8 av;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const u16 hb = zm::f2bf(x[j] > 0.f ? x[j] : 0.f);
        av[j] = __builtin_bit_cast(__bf16, hb);
      }
      const bf16x8 bv = *(const bf16x8 *)(w2t + (size_t)col * zm::NH1 + kb);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc, 0, 0, 0);
    }
    // layer 3: register i of lane l holds z2[move 8*(i/4)+4*half+i%4][unit col]
    float t[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const float z = acc[i] + b2o;
      t[i] = z > 0.f ? w3o * z : 0.f;
    }
#pragma unroll
    for (int o = 16; o > 0; o >>= 1)
#pragma unroll
      for (int i = 0; i < 16; i++) t[i] += __shfl_xor(t[i], o, 64);
    if (col == 0) {
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int row = 8 * (i >> 2) + 4 * half + (i & 3);
        if (c0 + row < total) {
          float sc = (t[i] + b3) * 256.f;
          sc = sc > 31000.f ? 31000.f : (sc < -31000.f ? -31000.f : sc);
          out(mbeg + c0 + row, __float2int_rn(sc));
        }
      }
    }
  }
  wsync();
}

// the plain ordering's score of a move (src/zeta.cl:2059-2082): MVV-LVA or
// the piece-square delta, the killer's 1400 and the counter move's 1300
template <class T>
__device__ __forceinline__ s32 plain_score(const T *tab, u32 stm, u32 m, u32 killer, u32 counter) {
  s32 sc = order_score(tab, stm, m);
  sc = sc > 31999 ? 31999 : (sc < -31999 ? -31999 : sc);
  if (((mv_pcpt(m) >> 1) & 7) == PNONE) {
    if (m == killer) sc = KILLER_SCORE;
    else if (counter_code(m) == counter) sc = COUNTER_SCORE;
  }
  return sc;
}

// Training pairs at a cut node of the full-width search whose cutoff move is
// not the TT move (the TT move goes first whatever the network says): the
// cutoff move against every other move of the node -- those searched before
// it, which failed, and those never searched, which the
// plain ordering ranked below it.  Each pair carries the plain ordering's
// score difference (negative minus positive), which the ranking loss adds to
// the network's, so that the network learns what to add to the plain
// ordering.  Wave-compacted.
__device__ void log_pairs(Args a, const Node &n, int lane, const u32 *mmove, const int16_t *tab, u32 ttm, u32 killer, u32 counter, u32 &nrec) {
  if (n.move == ttm) return;
  const s32 ppos = plain_score(tab, n.p.stm, n.move, killer, counter);
  for (int c0 = 0; c0 < n.mcnt; c0 += 64) {
    const int k = c0 + lane;
    bool neg = false;
    u32 m = 0;
    if (k < n.mcnt) {
      m = mmove[n.mbeg + k] & MOVE_BITS;
      neg = m != n.move && m != ttm;
    }
    const u64 mask = __ballot(neg);
    if (!mask) continue;
    const u32 cnt = (u32)popc(mask);
    u64 base = 0;
    if (lane == 0) base = atomicAdd((unsigned long long *)a->rec_count, (unsigned long long)cnt);
    base = uf(base);
    if (neg) {
      const u64 slot = base + (u64)popc(mask & ((1ULL << lane) - 1));
      if (slot < a->rec_cap) {
        s32 dp = plain_score(tab, n.p.stm, m, killer, counter) - ppos;
        dp = dp > zm::PAIR_OFFSET_MAX ? zm::PAIR_OFFSET_MAX : (dp < -zm::PAIR_OFFSET_MAX ? -zm::PAIR_OFFSET_MAX : dp);
        u64 *rp = a->recs + slot * 6;
        rp[0] = n.p.b0;
        rp[1] = n.p.b1;
        rp[2] = n.p.b2;
        rp[3] = n.p.b3;
        rp[4] = (u64)n.p.stm | ((u64)n.move << 32);
        rp[5] = (u64)m | ((u64)zm::pair_depth_word(n.depth, dp) << 32);
      }
    }
    nrec += cnt;
  }
}

// Serving synchronisation polls with relaxed atomics only: on this chip an
// acquire or release at agent scope costs an L2 invalidate / write-back (the
// L2 is per XCD), which, issued by polling workers, evicts every other
// worker's transposition-table and weight lines.  Relaxed agent- and
// system-scope atomics are coherent without cache maintenance.  Ordering is
// paid only where data is handed over, once per request or join: the release
// that opens a claimed request, the acquire of a helper's join, and the
// release that publishes a finished result to the host.
__device__ __forceinline__ u64 sys_load64(const u64 *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ u32 sys_load32(const u32 *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
template <class T> __device__ __forceinline__ T ag_load(const T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T> __device__ __forceinline__ void ag_store(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T> __device__ __forceinline__ bool ag_cas(T *p, T expect, T v) {
  return __hip_atomic_compare_exchange_strong(p, &expect, v, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT);
}
template <class T> __device__ __forceinline__ void sys_store(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ u64 sw_tk(u64 v) { return v >> 24; }
__device__ __forceinline__ int sw_max(u64 v) { return (int)((v >> 16) & 0xFF); }
__device__ __forceinline__ int sw_w(u64 v) { return (int)((v >> 2) & 0x3FFF); }
__device__ __forceinline__ int sw_st(u64 v) { return (int)(v & 3); }

// Serving: a slot's node count and deepest iteration carry the low 16 bits of
// their request's ticket (count: tag << 48 | nodes; depth: tag << 16 |
// iteration), and a worker adds to them only while the tag is its request's,
// in one compare-and-swap: a late helper of an earlier request can neither
// write into the slot's next request nor see its own numbers mixed with it.
__device__ __forceinline__ u64 slot_tag(u64 tk) { return tk & 0xFFFFULL; }
__device__ __forceinline__ void slot_add_nodes(u64 *p, u64 tk, u64 add) {
  u64 v = ag_load(p);
  while ((v >> 48) == slot_tag(tk)) {
    const u64 nv = (v & ~0xFFFFFFFFFFFFULL) | (((v & 0xFFFFFFFFFFFFULL) + add) & 0xFFFFFFFFFFFFULL);
    u64 e = v;
    if (__hip_atomic_compare_exchange_strong(p, &e, nv, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      return;
    v = e;
  }
}
__device__ __forceinline__ void slot_max_depth(s32 *p, u64 tk, s32 id) {
  s32 v = ag_load(p);
  while ((u64)((u32)v >> 16) == slot_tag(tk) && (v & 0xFFFF) < id) {
    s32 e = v;
    const s32 nv = (s32)((u32)(slot_tag(tk) << 16) | (u32)id);
    if (__hip_atomic_compare_exchange_strong(p, &e, nv, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      return;
    v = e;
  }
}

__device__ __forceinline__ u32 xcc_id() {
  // HW_REG_XCC_ID (hwreg 20), bits [3:0]
  return (u32)__builtin_amdgcn_s_getreg((20) | (0 << 6) | ((4 - 1) << 11)) & 15u;
}

// The scheduler wavefront (the grid's last block) never searches: every few
// microseconds it mirrors the host words (ticket count, shutdown, cancel
// generation) into device memory, so that the workers poll device memory
// only, and it runs the watchdog on its own clock.
__device__ void serve_scheduler(Args a, int lane) {
  ServeDev *v = a->sv;
  u64 hb_seen = 0, hb_time = 0;
  u32 cg_seen = 0;
  for (;;) {
    u32 shut = 0, cg = 0;
    if (lane == 0) {
      const u64 now = wall_clock64();
      const u64 sub = sys_load64(&a->sh->submitted);
      const u64 hb = sys_load64(&a->sh->heartbeat);
      shut = sys_load32(&a->sh->shutdown) ? 1u : 0u;
      cg = sys_load32(&a->sh->cancel_gen);
      if (hb != hb_seen || hb_time == 0) {
        hb_seen = hb;
        hb_time = now;
      } else if (a->watchdog_ticks && now - hb_time > a->watchdog_ticks) {
        shut = 2;
        ag_store(&v->exit_now, now);
        ag_store(&v->exit_arg, hb_time);
        ag_store(&v->exit_xcc, xcc_id());
      }
      ag_store(&v->sub, sub);
    }
    cg = uf(cg);
    if (cg != cg_seen) {
      for (int s = lane; s < a->nslots; s += 64) ag_store(&a->dcancel[s], sys_load64(&a->scancel[s]));
      cg_seen = cg;
    }
    shut = uf(shut);
    if (shut) {
      if (lane == 0) ag_store(&v->shut, shut);
      return;
    }
    __builtin_amdgcn_s_sleep(127);
  }
}

// serving: claim the next published ticket, else join the running request
// with the fewest workers; returns its slot and ticket+1, or -1 on shutdown
__device__ int serve_pick(Args a, int lane, u64 &tk_out) {
  int backoff = 1;
  for (;;) {
    int res = -2;
    u64 tk = 0;
    if (lane == 0) {
      if (ag_load(&a->sv->shut)) {
        res = -1;
      } else {
        const u64 c = ag_load(&a->sv->claimed);
        if (c < ag_load(&a->sv->sub) && ag_cas(&a->sv->claimed, c, c + 1)) {
          const int qi = (int)(c % (u64)a->qcap);
          const u64 s = sys_load64(&a->squeue[qi]);
          if (s >= (u64)a->nslots) {
            ag_store(&a->sv->exit_now, c);
            ag_store(&a->sv->exit_arg, s);
            ag_store(&a->sv->shut, 3u);  // the host broke the protocol: stop serving
            res = -1;
          } else {
            ServeReq &d = a->dreq[s];
            const ServeReq &h = a->slots[s].req;
            for (int k = 0; k < 8; k++) ag_store(&d.pos[k], sys_load64(&h.pos[k]));
            const s32 hw = (s32)sys_load32((const u32 *)&h.workers);
            ag_store(&d.depth, (s32)sys_load32((const u32 *)&h.depth));
            ag_store(&d.flags, (s32)sys_load32((const u32 *)&h.flags));
            ag_store(&d.workers, hw);
            sys_store(&a->sack[qi], c + 1);
            ag_store(&a->nodes[s], slot_tag(c + 1) << 48);
            ag_store(&a->depth_done[s], (s32)(u32)(slot_tag(c + 1) << 16));
            const u64 wmax = (u64)(hw < 1 ? 1 : (hw > 255 ? 255 : hw));
            // release: the request copy above is visible to every helper
            // that joins through this word (one write-back per request)
            __hip_atomic_store(&a->sw[s], (u64)(((c + 1) << 24) | (wmax << 16) | (u64)4 | (u64)SV_RUN),
                               __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            res = (int)s;
            tk = c + 1;
          }
        }
      }
    }
    res = uf(res);
    if (res != -2) {
      tk_out = uf(tk);
      return res;
    }
    // no new request: the running request with the fewest workers below its maximum
    u32 bestkey = 0;
    for (int base = 0; base < a->nslots; base += 64) {
      const int s = base + lane;
      if (s < a->nslots) {
        const u64 v = ag_load(&a->sw[s]);
        const int w = sw_w(v);
        // a cancelled request takes no new helpers: its workers drain and the
        // last one publishes the cancellation
        if (sw_tk(v) && sw_st(v) == SV_RUN && w >= 1 && w < sw_max(v) && ag_load(&a->dcancel[s]) != sw_tk(v))
          bestkey = max(bestkey, ((u32)(255 - w) << 16) | (u32)(0xFFFF - s));
      }
    }
    bestkey = wave_max_u32(bestkey);
    if (bestkey) {
      const int s = 0xFFFF - (int)(bestkey & 0xFFFF);
      int got = -1;
      if (lane == 0) {
        const u64 v = ag_load(&a->sw[s]);
        u64 e = v;
        if (sw_tk(v) && sw_st(v) == SV_RUN && sw_w(v) >= 1 && sw_w(v) < sw_max(v) &&
            ag_load(&a->dcancel[s]) != sw_tk(v) &&
            __hip_atomic_compare_exchange_strong(&a->sw[s], &e, v + 4, __ATOMIC_ACQUIRE, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT)) {  // acquire: once per join
          got = s;
          tk = sw_tk(v);
        }
      }
      got = uf(got);
      if (got >= 0) {
        tk_out = uf(tk);
        return got;
      }
    } else {
      // nothing to do: back off (up to ~50 us) so idle workers stay off the
      // memory system the searching ones use
      for (int i = 0; i < backoff; i++) __builtin_amdgcn_s_sleep(127);
      backoff = backoff < 16 ? 2 * backoff : 16;
    }
  }
}

// serving: leave the request.  The worker that completes it (or fails it)
// records the result in device memory and sets the status in the slot word,
// which sends the others away at their next poll; the last worker to leave
// publishes the result to the host slot -- DONE or FAILED as set, or
// CANCELLED when every worker left a running request -- so the published
// node count includes every worker's nodes.
__device__ void serve_leave(Args a, int r, u64 tk, bool aborted, bool failed, s32 score, u32 move) {
  if (!aborted && !failed) ag_store(&a->dres[r], (u64)(u32)score | ((u64)move << 32));
  for (;;) {
    const u64 v = ag_load(&a->sw[r]);
    if (sw_tk(v) != tk) return;  // the slot has moved on
    int st = sw_st(v);
    if (st == SV_RUN) {
      if (failed) st = SV_FAILED;
      else if (!aborted) st = SV_DONE;
    }
    const bool last = sw_w(v) == 1;
    const u64 nv = ((v - 4) & ~3ULL) | (u64)st;
    // release: the result recorded above before the status that announces
    // it; acquire: the last worker sees the result the completing one wrote
    u64 e = v;
    if (!__hip_atomic_compare_exchange_strong(&a->sw[r], &e, nv, __ATOMIC_ACQ_REL, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT))
      continue;
    if (last) {
      const int pub = st == SV_RUN ? SV_CANCELLED : st;
      const u64 res = pub == SV_DONE ? ag_load(&a->dres[r]) : 0ULL;
      ServeSlot &sl = a->slots[r];
      sys_store(&sl.score, (s32)(u32)res);
      sys_store(&sl.bestmove, (u32)(res >> 32));
      sys_store(&sl.nodes, (u64)(ag_load(&a->nodes[r]) & 0xFFFFFFFFFFFFULL));
      sys_store(&sl.ticket, tk);
      sys_store(&sl.depth_done, (s32)(ag_load(&a->depth_done[r]) & 0xFFFF));
      sys_store(&sl.status, (s32)pub);
      // the one ordering point: the result fields before the done flag
      __hip_atomic_store(&sl.state, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    return;
  }
}

constexpr u64 OUTER_RANKS = 0xFF000000000000FFULL;

// One ply of a worker's stack: a node as 32-bit words, stored and loaded with
// one word a lane in one LDS access (field by field, and with the parent's
// board taken back from the child's by undoing the move, a visit spent 1100
// instructions on it).
constexpr int NWORDS = 24;
enum { W_PLANES = 0, W_CR = 8, W_HASH = 10, W_PHASH = 12, W_LEFT = 14, W_WINDOW = 16, W_MOVE, W_BEST, W_LIST, W_COUNTS, W_FLAGS, W_TTM, W_FLOOR };
struct Ply {
  u32 w[24];
};

struct Lds {  // one worker's memory: eight workers a CU
  __align__(16) u64 lines[64][4];  // rank, file, diagonal, anti-diagonal through a square, without it
  Ply ply[MAXPLY + 2];
  u32 mmove[MSTACK + MPAD];
  u32 mkey[MSTACK];
  u32 killers[MAXPLY + 2];
  union {
    float hpos[zm::NH1];  // the learned scorer's hidden vector
    u8 mstart[64];        // move-list start marks (lane + 1 at its offset)
  };
  int16_t tab[7 * 64];    // EVAL_SQ
  // the root in progress: its ticket (serving), index and depth, the iteration,
  // its best move so far, and the result of the last completed one
  u64 ticket;
  int root, depth, iteration;
  int hlen;  // positions of the game before the root
  u64 hsalt;  // of their hashes, see path_key
  s32 best_score, final_score;
  u32 best_move, final_move;
};

// v_writelane_b32: x with lane k (a constant) set to v
extern "C" __device__ int write_lane(int v, int k, int x) __asm("llvm.amdgcn.writelane.i32");
__device__ __forceinline__ int put32(int w, int k, u32 v) { return write_lane((int)v, k, w); }
__device__ __forceinline__ int put64(int w, int k, u64 v) { return put32(put32(w, k, (u32)v), k + 1, (u32)(v >> 32)); }
__device__ __forceinline__ u32 get32(int w, int k) { return (u32)__builtin_amdgcn_readlane(w, k); }
__device__ __forceinline__ u64 get64(int w, int k) { return ((u64)get32(w, k + 1) << 32) | get32(w, k); }
__device__ __forceinline__ int put_planes(int w, const Pos &p) {
  return put64(put64(put64(put64(w, W_PLANES, p.b0), W_PLANES + 2, p.b1), W_PLANES + 4, p.b2), W_PLANES + 6, p.b3);
}
__device__ __forceinline__ void get_planes(int w, Pos &p) {
  p.b0 = get64(w, W_PLANES);
  p.b1 = get64(w, W_PLANES + 2);
  p.b2 = get64(w, W_PLANES + 4);
  p.b3 = get64(w, W_PLANES + 6);
}
__device__ __forceinline__ u32 window(s32 alpha, s32 beta) { return ((u32)alpha & 0xFFFFu) | ((u32)beta << 16); }

enum { F_STM = 1, F_CHECK = 2, F_PASS2 = 4, F_BUSY = 8, F_REACH = 16, F_SCOUT = 64, F_CHILD = 1 << 16 };  // F_REACH: two bits, F_CHILD: 16

__device__ __forceinline__ void save(Ply &y, const Node &n, int lane) {
  int w = put_planes(0, n.p);
  w = put64(w, W_CR, n.p.cr);
  w = put64(w, W_HASH, n.hash);
  w = put64(w, W_PHASH, n.phash);
  w = put64(w, W_LEFT, n.left);
  w = put32(w, W_WINDOW, window(n.alpha, n.beta));
  w = put32(w, W_MOVE, n.move);
  w = put32(w, W_BEST, n.best);
  w = put32(w, W_LIST, (u32)n.mbeg | ((u32)n.mcnt << 16));
  w = put32(w, W_COUNTS, (u32)n.depth | (n.hmc << 8) | ((u32)n.searched << 16) | ((u32)n.ndefer << 24));
  w = put32(w, W_FLAGS, (n.p.stm ? F_STM : 0) | (n.kic ? F_CHECK : 0) | (n.pass2 ? F_PASS2 : 0) | (n.busy ? F_BUSY : 0) |
                         n.reach * F_REACH | (n.scout ? F_SCOUT : 0) | n.child * F_CHILD);
  w = put32(w, W_TTM, n.ttm);
  w = put32(w, W_FLOOR, (u32)n.floor);
  if (lane < NWORDS) y.w[lane] = (u32)w;
}
__device__ __forceinline__ void restore(const Ply &y, Node &n, int lane) {
  const int w = (int)y.w[lane < NWORDS ? lane : 0];
  get_planes(w, n.p);
  n.p.cr = get64(w, W_CR);
  n.hash = get64(w, W_HASH);
  n.phash = get64(w, W_PHASH);
  n.left = get64(w, W_LEFT);
  const u32 win = get32(w, W_WINDOW), list = get32(w, W_LIST), cnt = get32(w, W_COUNTS), fl = get32(w, W_FLAGS);
  n.alpha = (s32)(int16_t)(u16)win;
  n.beta = (s32)win >> 16;
  n.move = get32(w, W_MOVE);
  n.best = get32(w, W_BEST);
  n.mbeg = (int)(list & 0xFFFFu);
  n.mcnt = (int)(list >> 16);
  n.depth = (s32)(cnt & 0xFFu);
  n.hmc = (cnt >> 8) & 0xFFu;
  n.searched = (int)((cnt >> 16) & 0xFFu);
  n.ndefer = (int)(cnt >> 24);
  n.p.stm = fl & F_STM ? 1u : 0u;
  n.kic = (fl & F_CHECK) != 0;
  n.pass2 = (fl & F_PASS2) != 0;
  n.busy = (fl & F_BUSY) != 0;
  n.reach = (fl / F_REACH) & 3u;
  n.scout = (fl & F_SCOUT) != 0;
  n.child = fl / F_CHILD;
  n.ttm = get32(w, W_TTM);
  n.floor = (s32)get32(w, W_FLOOR);
}
// x of lane k (wave-uniform)
__device__ __forceinline__ u64 lane64(u64 x, int k) {
  return ((u64)(u32)__builtin_amdgcn_readlane((int)(x >> 32), k) << 32) | (u32)__builtin_amdgcn_readlane((int)x, k);
}
// the move that led to the node at ply sd, 0 at the root
__device__ __forceinline__ u32 last_move(const Lds &L, int sd) { return sd > 1 ? uf(L.ply[sd - 1].w[W_MOVE]) : 0u; }

// Whether what a search below the node at ply sd found holds on any path to it.
// Only positions searched in full width are tested for repetition.  `reach` is
// how far below the node the search (or a table entry it used) tested one that
// reversible moves lead to: 3 for 3 or more.  hr plies above the node are
// reversibly connected to it.  A position k plies below repeats one above only
// if they are 4, 6, .. plies apart: none while reach + hr <= 3.  One ply below,
// 4 plies apart, the two moves of the side that moved last are both on the path
// and have to take each other back.  The half-move clock has to stay clear of
// 100 as well.  With a clock of 0 nothing above can be met again.
// Most nodes have one ply left, no checking move and so reach 0: their bounds
// serve every order of the moves that lead to them: 1.0 M of 4.1 M probes of a
// 1024-position depth-4 batch end the node (before, with a clock of 0 on both
// sides required, moves in another order were searched again), and the probe
// comes ahead of the generation.
__device__ __forceinline__ bool path_free(const Lds &L, const Node &n, u32 reach, int sd) {
  if (n.hmc == 0) return true;
  if (reach >= 3 || n.hmc >= 90) return false;
  if (reach == 0) return true;
  const int above = sd - 1 + uf(L.hlen), hr = (int)n.hmc < above ? (int)n.hmc : above;
  if ((int)reach + hr <= 3) return true;
  if (reach != 1 || hr > 4 || sd < 4) return false;
  const u32 m = uf(L.ply[sd - 1].w[W_MOVE]), o = uf(L.ply[sd - 3].w[W_MOVE]);
  return mv_from(m) != mv_to(o) || mv_to(m) != mv_from(o);
}

// The positions above the node at ply sd that a search below it can repeat, as
// one word: those of the path since the last irreversible move, the game's if
// that lies before the root, and the half-move clock.  A bound that holds on
// this path only is stored under the position's key and this one.  The workers
// of a root share its nodes high in the tree through it, whose bounds depend on
// the path (six positions, depth 5, 128 workers: 113 -> 107 ms).
__device__ __forceinline__ u64 hash_mix(u64 x) {
  x ^= x >> 32;
  x *= 0x9E3779B97F4A7C15ULL;
  return x ^ (x >> 29);
}
__device__ __forceinline__ u32 wave_xor(u32 x) {
  x ^= (u32)zw::dpp0<0x111, 0xF>((int)x);
  x ^= (u32)zw::dpp0<0x112, 0xF>((int)x);
  x ^= (u32)zw::dpp0<0x114, 0xF>((int)x);
  x ^= (u32)zw::dpp0<0x118, 0xF>((int)x);
  x ^= (u32)zw::dpp0<0x142, 0xA>((int)x);
  x ^= (u32)zw::dpp0<0x143, 0xC>((int)x);
  return (u32)__builtin_amdgcn_readlane((int)x, 63);
}
__device__ __forceinline__ u64 wave_xor(u64 x) { return ((u64)wave_xor((u32)(x >> 32)) << 32) | wave_xor((u32)x); }
__device__ __forceinline__ u64 path_key(const Lds &L, const Node &n, int sd, int lane) {
  u64 v = 0;
  const int k = sd - 1 - lane;  // the node's ancestors are at plies 1 .. sd - 1
  if (k >= 1 && lane < (int)n.hmc) {
    const u32 *const w = L.ply[k].w;
    v = hash_mix(((u64)w[W_HASH + 1] << 32) | w[W_HASH]);
  }
  u64 x = wave_xor(v) + (u64)(n.hmc + 1) * 0xD1B54A32D192ED03ULL;
  if ((int)n.hmc >= sd) x += uf(L.hsalt);
  return hash_mix(x);
}
template <int TABLE>
__device__ __forceinline__ void tt_write(Args a, u64 ttmask, u64 key, u64 w1, int lane) {
  if (lane == 0) {
    const u64 w0 = key ^ w1;
    u64 *const e = a->tt + 2 * (key & ttmask);
    if (TABLE == T_BUDGET) {
      *glob((u32x4 *)e) = u32x4{(u32)w0, (u32)(w0 >> 32), (u32)w1, (u32)(w1 >> 32)};
    } else {
      shared_store(e, w0);
      shared_store(e + 1, w1);
    }
  }
}

// TT store when a full-width node returns: with a move that raised alpha, a
// lower bound of the node's value and that move; with none (every move
// failed low), an upper bound (bit 58) and the move that the table had before,
// which the next iteration would otherwise lose (six batches of 1024 positions,
// depth 4: 714 -> 645 ms).  The score is kept as
// distance-to-mate from this node.  Bit 56: the bound does not depend on the
// path above the node, or the entry is under this path's key; bits 59-60: the
// node's reach (path_free).  Nothing is stored where the root's bound may have
// made the value (bound_holds).  Returns how many values were.
template <int TABLE>
__device__ __forceinline__ u32 tt_store(Args a, u64 ttmask, const Lds &L, const Node &n, int sd, s32 ra, int lane) {
  if (!bound_holds(sd, ra, n.best != 0, n.alpha)) return 0;
  s32 s = n.alpha;
  const int plyn = sd - 1;
  if (is_mate(s) && s > 0) s += plyn;
  if (is_mate(s) && s < 0) s -= plyn;
  const u64 key = tt_key(n.hash, n.p.cr);
  const bool any = path_free(L, n, n.reach, sd);
  const u64 w1 = (u64)(n.best ? n.best : n.ttm) | ((u64)(u16)(int16_t)s << 32) | ((u64)(n.depth & 0xFF) << 48) |
                 (1ULL << 57) | ((u64)(n.best ? 0 : 1) << 58) | ((u64)n.reach << 59);
  tt_write<TABLE>(a, ttmask, key, w1 | ((u64)(any ? 1 : 0) << 56), lane);
  if (TABLE == T_SHARED && !any && n.depth >= PATH_DEPTH)
    tt_write<TABLE>(a, ttmask, key ^ path_key(L, n, sd, lane), w1 | (1ULL << 56), lane);
  return 1;
}

// the lines of a wave-uniform square, in vector registers (24 scalar ones for
// the two kings are more than the search has to spare)
__device__ __forceinline__ SqLines lds_lines(const Lds &L, int k) {
  const u64 b = bit(k);
  const u64 *q = L.lines[k];
  return SqLines{b, bit(63 - k), q[0], q[1], q[2], q[3]};
}

// the static evaluation for the side to move: lane = square
__device__ __forceinline__ s32 static_eval(const Pos &p, int lane) {
  // the square is hidden from the compiler, which would keep a 64-bit mask of
  // lanes for every condition on it through the whole search
  asm volatile("" : "+v"(lane));
  const s32 e = wave_sum_i(eval_square(p, lane)) + eval_bishop_pair(p);
  return p.stm ? -e : e;
}

// The periodic test (every POLL_EVERY nodes) looks at words that were loaded at
// the test before it: the abort word lies in host memory, a read of 2 us.  So
// what the host or another worker sets is seen at the second test after it, up
// to 2 * POLL_EVERY nodes later; a node budget at the first.
struct Poll {
  int count;      // nodes since the last test
  u64 nodes;      // nodes made at this root
  u64 state;      // done (batch) or the slot word (serving)
  u64 cancel;     // abort word, or the slot's cancelled ticket
  u32 shut;       // serving: the grid shuts down
  u64 rbound;     // the root bound published by the root's workers
};
__device__ __forceinline__ void poll_load(Args a, int r, int lane, Poll &q) {
  if (lane == 0) {
    if (a->slots) {
      q.state = ag_load(glob(&a->sw[r]));
      q.cancel = ag_load(glob(&a->dcancel[r]));
      q.shut = ag_load(&glob(a->sv)->shut);
    } else {
      q.state = ag_load(glob(&a->done[r]));
      q.cancel = sys_load32(glob(a->habort));
    }
    q.rbound = ag_load(glob(&a->rbound[r]));
  }
}
// true when the worker has to leave the root; renews the root bound `ra`
__device__ __forceinline__ bool poll_root(Args a, const Lds &L, int lane, Poll &q, s32 &ra) {
  q.count = 0;
  const int r = uf(L.root);
  bool d;
  if (a->slots) {
    d = sw_tk(q.state) != L.ticket || sw_st(q.state) != SV_RUN || q.cancel == L.ticket || q.shut != 0;
  } else {
    // stop when the root is finished or given up, or the host aborts
    d = q.state != 0 || q.cancel != 0;
    if (!d && a->max_nodes && q.nodes > a->max_nodes) {
      // over the node budget: give the root up, so that no worker picks it
      // again (a fresh budget on the same iteration could repeat forever);
      // its result is this worker's deepest completed iteration
      if (lane == 0 && atomicCAS(&a->done[r], 0u, 3u) == 0u) {
        a->score[r] = L.final_score;
        a->bestmove[r] = L.final_move;
      }
      d = true;
    }
  }
  if (uf((u32)d)) return true;
  // (the word may be older than the bound that the iteration started with)
  const u64 rb = uf(q.rbound);
  const s32 b = (s32)(rb & 0xFFFF) - 32768;
  if ((rb >> 32) == (uf(L.ticket) & 0xFFFFFFFFULL) && (int)((rb >> 16) & 0xFFFF) == uf(L.iteration) && b > ra) ra = b;
  poll_load(a, r, lane, q);
  return false;
}

// A node's move list while it is the current one: lane j holds move j and its
// key (of lists of up to 64 moves; longer ones are read from the move stack,
// where every list is kept).
struct List {
  u32 move, key;
};
__device__ __forceinline__ List load_list(const Lds &L, int lane, int mbeg) {
  // lanes past the list's end read other slots of the worker's memory
  const int k = mbeg + lane < MSTACK ? mbeg + lane : 0;
  return List{L.mmove[k], L.mkey[k]};
}

// The next move of a node's list: the highest score, the lowest slot among
// equals (wave arg-max); takes it out of the list and gives its slot, code and
// key, or -1.  Moves whose child is known to stand pat at or above `limit` (the
// child's beta; 2 * INF: no such test) return at once in a visit and change
// nothing at the node but the node count, for a limit that only falls while
// the node is searched: those ahead of the next move are counted here (more
// than half of all nodes), up to the periodic poll, whose turn comes in the
// visit of the child it falls on.
// defer: the list holds deferred moves, which pass 2 takes and pass 1 skips.
__device__ __forceinline__ int pick_move(Lds &L, int lane, int mbeg, int mcnt, const List &li, u64 &left, s32 limit,
                                         bool defer, bool pass2, Poll &q, int &searched, u32 &m, u32 &mk) {
  u32 lim = (u32)(limit + 32768);
  lim = lim > KEY_OPEN ? lim : KEY_OPEN + 1;
  if (mcnt <= 64) {
    const u32 sk = (li.key | 0xFFFFu) - (u32)lane;
    const u64 refuted = __ballot((li.key & 0xFFFFu) >= lim);
    u64 avail = left;
    if (defer) {
      const u64 d = __ballot((L.mmove[mbeg + lane < MSTACK ? mbeg + lane : 0] & DEFERRED) != 0u);
      avail &= pass2 ? d : ~d;
    }
    for (;;) {
      u32 best = wave_max_u32(__builtin_amdgcn_inverse_ballot_w64(avail & ~refuted) ? sk : 0u);
      u64 ahead = avail & refuted & __ballot(sk > best);
      if (ahead) {
        int c = popc(ahead);
        bool one = false;
        if (q.count + c >= POLL_EVERY) {
          // a poll falls among them: one at a time up to it
          const u32 top = wave_max_u32(__builtin_amdgcn_inverse_ballot_w64(ahead) ? sk : 0u);
          one = q.count + 1 < POLL_EVERY;
          if (one) ahead = 1ULL << (0xFFFFu - (top & 0xFFFFu));
          else best = top;
          c = one ? 1 : 0;
        }
        if (c) {
          left &= ~ahead;
          avail &= ~ahead;
          q.count += c;
          q.nodes += (u64)c;
          if (!pass2) searched += c;
          if (one) continue;
        }
      }
      if (best == 0) return -1;
      const int k = (int)(0xFFFFu - (best & 0xFFFFu));
      left &= ~(1ULL << k);
      m = get32((int)li.move, k) & MOVE_BITS;
      mk = get32((int)li.key, k);
      return k;
    }
  }
  // a longer list: its searched moves lose the score in their keys
  auto sort_key = [&](int k) {
    if (k >= mcnt) return 0u;
    const u32 key = L.mkey[mbeg + k];
    u32 sk = key >> 16 ? (key | 0xFFFFu) - (u32)k : 0u;
    if (defer && ((L.mmove[mbeg + k] & DEFERRED) != 0u) != pass2) sk = 0;
    return sk;
  };
  auto refuted = [&](int k) { return k < mcnt && (L.mkey[mbeg + k] & 0xFFFFu) >= lim; };
  for (;;) {
    u32 best = 0, top = 0;
    for (int k = lane; k < mcnt; k += 64) {
      const u32 sk = sort_key(k);
      if (refuted(k)) top = sk > top ? sk : top;
      else best = sk > best ? sk : best;
    }
    best = wave_max_u32(best);
    top = wave_max_u32(top);
    if (top > best) {
      // one refuted move at a time, and a visit where the poll falls
      best = top;
      if (q.count + 1 < POLL_EVERY) {
        const int k = (int)(0xFFFFu - (best & 0xFFFFu));
        if (lane == 0) L.mkey[mbeg + k] &= 0xFFFFu;
        q.count++;
        q.nodes++;
        if (!pass2) searched++;
        wsync();
        continue;
      }
    }
    if (best == 0) return -1;
    const int k = (int)(0xFFFFu - (best & 0xFFFFu));
    m = uf(L.mmove[mbeg + k]) & MOVE_BITS;
    mk = uf(L.mkey[mbeg + k]);
    wsync();
    if (lane == 0) L.mkey[mbeg + k] = mk & 0xFFFFu;
    wsync();
    return k;
  }
}

// The legal moves of a node -- QS: its captures, e.p. included -- in the order
// of origin, then target, with their keys; returns how many, or -1 when they
// do not fit the move stack.  Lane = square gives the targets of its piece;
// then lane = move makes the child, tests its legality (own king not attacked;
// only when the king is in check or a slider is lined up with it, king moves
// by the attack map instead, e.p. on its own) and finds what the key says of
// the child: in check, and, where the children are quiescence nodes
// (leafward), the evaluation: the parent's piece-square sum by the move's
// change of it, the pawn terms set by set.
// ep = the bit of the pawn that may be taken en passant, or 0.
template <bool QS>
__device__ __forceinline__ int gen_moves(Lds &L, const LaneSq &me, int lane, const Pos &p, u64 ep, bool kic, u32 hmc,
                                         int mbeg, bool leafward, u32 killer, u32 counter, List &li) {
  const u64 occ = p.b1 | p.b2 | p.b3;
  const u64 white = p.b0 ^ occ;
  const u64 own = p.stm ? p.b0 : white, opp = p.stm ? white : p.b0;
  const u64 rq = p.b3 & (p.b1 ^ p.b2), bq = p.b3 & ~p.b1;
  const u64 kings = p.b1 & p.b2 & ~p.b3, kbb = own & kings, okb = opp & kings;
  const u32 pc = piece_at(p, lane);
  const u32 type = pc >> 1;
  const bool mine = type != PNONE && (pc & 1u) == p.stm;
  const u64 patt = p.stm ? me.bpawn : me.wpawn;
  // the pawn sums want no pawn on the outer ranks
  const bool keyed = leafward && !(p.b1 & ~p.b2 & ~p.b3 & OUTER_RANKS);
  const s32 psq = keyed ? eval_piece(L.tab, pc, lane) : 0;
  u64 t = sel(type == ROOK || type == QUEEN, rook_sq(me.q, occ)) | sel(type == BISHOP || type == QUEEN, bishop_sq(me.q, occ));
  t = type == KNIGHT ? me.knight : t;
  t = type == KING ? me.king : t;
  t &= QS ? opp : ~own;
  if (QS) {
    t = type == PAWN ? patt & opp : t;
  } else {
    const u64 s1 = (p.stm ? me.q.b >> 8 : me.q.b << 8) & ~occ;
    const u64 s2 = (p.stm ? (s1 & RANK6) >> 8 : (s1 & RANK3) << 8) & ~occ;
    t = type == PAWN ? (patt & opp) | s1 | s2 : t;
  }
  t = mine ? t : 0;
  const bool rights = !QS && (p.cr & SMCRALL);
  if (rights || __ballot(type == KING && t != 0)) {
    // squares the king may not step to: attacked with the king off the board
    const u64 o2 = occ ^ kbb;
    u64 at = (rook_sq(me.q, o2) & rq) | (bishop_sq(me.q, o2) & bq);
    at |= me.knight & ~p.b1 & p.b2 & ~p.b3;
    at |= me.king & kings;
    at |= patt & p.b1 & ~p.b2 & ~p.b3;
    const u64 A = __ballot((at & opp) != 0);
    if (type == KING) t &= ~A;
    if (rights && type == KING && mine) t |= castle_squares(p, own & rq & ~p.b2, occ, A, lane);
  }
  const int ksq = kbb ? lsb(kbb) : 0;
  if (ep) {
    const int sqep = lsb(ep);
    const bool cand = mine && type == PAWN && (((p.stm ? RANK4 : RANK5) & (bit(sqep + 1) | bit(sqep - 1))) >> lane) & 1;
    if (__ballot(cand)) {
      Node0 B;
      B.own = own;
      B.opp = opp;
      B.occ = occ;
      B.kbb = kbb;
      B.pawns = p.b1 & ~p.b2 & ~p.b3;
      B.knights = ~p.b1 & p.b2 & ~p.b3;
      B.kings = kings;
      B.rq = rq;
      B.bq = bq;
      B.ksq = ksq;
      B.stm = p.stm;
      const int to = (p.stm ? sqep - 8 : sqep + 8) & 63;
      if (cand && ep_legal0(B, lane, to, sqep)) t |= bit(to);
    }
  }
  // one scan for the slots (below 1024) and the piece-square sum
  const s32 scan = zw::wave_scan_add(popc(t) + psq * 1024), last = (s32)__builtin_amdgcn_readlane(scan, 63);
  const int total = last & 1023;
  if (total == 0) return 0;
  const int off = (scan & 1023) - popc(t);
  const s32 base = last >> 10;
  int from = 0, to = 0;  // of the lane's move
  const bool small = !QS && total <= 64;
  if (small) {
    // lane j takes move j of the list: its origin is the last lane with
    // targets whose offset is <= j (a prefix max over start marks), its target
    // the (j - offset)-th bit of that lane's set -- one pass instead of as
    // many loop trips as the busiest lane has targets
    L.mstart[lane] = 0;
    wsync();
    if (t) L.mstart[off] = (u8)(lane + 1);
    wsync();
    const int own1 = (int)zw::wave_scan_max(lane < total ? (u32)L.mstart[lane] : 0u);
    from = (own1 > 0 ? own1 : 1) - 1;
    const int k = lane - __shfl(off, from, 64);
    const u64 ts = ((u64)(u32)__shfl((int)(u32)(t >> 32), from, 64) << 32) | (u32)__shfl((int)(u32)t, from, 64);
    to = lane < total ? nth_bit(ts, k) : 0;
  } else {
    if (mbeg + total > MSTACK + MPAD) return -1;
    u32 *out = L.mmove + mbeg + off;
    while (t) {
      *out++ = (u32)lane | ((u32)lsb(t) << 6);
      t &= t - 1;
    }
    wsync();
  }
  const SqLines kq = lds_lines(L, ksq);
  const bool test = kbb && (kic || __ballot(((((kq.rank | kq.file) & rq) | ((kq.diag | kq.anti) & bq)) & opp) != 0));
  const int osq = okb ? lsb(okb) : 0;
  const SqLines oq = lds_lines(L, osq);
  // what attacks the kings' squares: the lanes of those squares hold it (made
  // from the square it took 130 of a visit's 860 instructions, with the constants
  // spilled; six batches of 1024 positions, depth 4: 635 -> 592 ms)
  const u64 kknight = lane64(me.knight, ksq), kpawn = lane64(patt, ksq);
  const u64 oknight = lane64(me.knight, osq), opawn = lane64(p.stm ? me.wpawn : me.bpawn, osq);
  int kept = 0;
  for (int c0 = 0; c0 < total; c0 += 64) {
    const bool act = c0 + lane < total;
    if (!small) {
      const u32 raw = act ? L.mmove[mbeg + c0 + lane] : 0u;
      from = (int)(raw & 63u);
      to = (int)(raw >> 6);
    }
    const u32 pf = (u32)__shfl((int)pc, from, 64);
    u32 cap = (u32)__shfl((int)pc, to, 64);
    const bool pawn = (pf >> 1) == PAWN;
    bool isep = false;
    int x = to;
    if (ep) {  // wave-uniform
      isep = pawn && cap == 0 && ((from ^ to) & 7);
      x = isep ? (p.stm ? to + 8 : to - 8) & 63 : to;
      cap = (u32)__shfl((int)pc, x, 64);
    }
    const u32 pt = pawn && (p.stm ? to < 8 : to >= 56) ? ((QUEEN << 1) | p.stm) : pf;
    const u32 m = mv_make((u32)from, (u32)to, (u32)x, pf, pt, cap);
    const Pos c = QS ? apply_capture(p, m) : apply(p, m, false);
    bool legal = act;
    if (test) legal = act && ((pf >> 1) == KING || isep || !king_attacked(c, kq, true, kknight, kpawn, p.stm ^ 1u));
    u32 key = KEY_OPEN;
    if (keyed) {
      const u64 cocc = c.b1 | c.b2 | c.b3;
      const s32 e = base + (QS ? eval_move_delta<false>(L.tab, p.stm, m) : eval_move_delta<true>(L.tab, p.stm, m)) +
                    pawn_terms(c.b1 & ~c.b2 & ~c.b3, c.b0 ^ cocc, c.b0) + eval_bishop_pair(c);
      // a draw or a sum beyond 16 bits is left to the visit, so are
      // promotions (extended) and full half-move clocks
      bool known = popc(cocc) > 2 && (u32)(e + 31000) <= 62000u;
      if (!QS) known = known && !is_promo(m) && child_hmc(hmc, m) < 100;
      if (known) key = (u32)((p.stm ? e : -e) + 32768);
    }
    // (a captured king is in no check)
    if (king_attacked(c, oq, okb != 0 && (cap >> 1) != KING, oknight, opawn, p.stm)) key = KEY_CHECK;
    const s32 sc = QS ? piece_value(cap >> 1) * 16 - piece_value(pt >> 1) : plain_score(L.tab, p.stm, m, killer, counter);
    const u64 lm = __ballot(legal);
    const int slot = mbeg + kept + popc(lm & ((1ULL << lane) - 1));
    kept += popc(lm);
    if (mbeg + kept > MSTACK) return -1;
    wsync();
    li = List{m, move_key(sc, key)};
    if (legal) {
      L.mmove[slot] = m;
      L.mkey[slot] = li.key;
    }
  }
  wsync();
  // illegal moves left out: the list's lanes close up
  if (kept != total) li = load_list(L, lane, mbeg);
  return kept;
}
// the slots of a list of n moves
__device__ __forceinline__ u64 all_moves(int n) { return n < 64 ? (1ULL << n) - 1 : ~0ULL; }

enum { QS_DONE = 0, QS_ABORTED, QS_FAILED };

__device__ __forceinline__ void qt_store(const Pos &p, u64 phash, s32 v, u32 kind, int lane) {
  if (lane != 0 || kind == Q_NONE || v != (s32)(int16_t)(u16)v) return;
  const Args a = args();
  const u64 key = phash ^ (u64)p.stm;
  shared_store(a->qtt + (key & a->qmask), (key >> QT_BITS << QT_BITS) | (kind << 16) | ((u32)v & 0xFFFFu));
}

// A quiescence node and everything below it, which is quiescence too: captures
// only, stand pat when not in check, no table, no hash, no extension, no
// deferral.  Apart from the full-width loop it keeps a few scalars a ply: the
// four planes, the window and the list.  ev / known: the evaluation, if the
// parent has it; kic: in check; polled: the visit has been counted to the poll.
template <bool TABLE>
__device__ __forceinline__ int qsearch(Lds &L, const LaneSq &me, int lane, Pos p, s32 alpha, s32 beta, u32 hmc,
                                       const int sd0, int mbeg, s32 ev, bool known, bool kic, bool polled, u64 phash,
                                       Poll &q, s32 &ra, u32 &cvec, s32 &vout) {
  int sd = sd0, mcnt = 0, unused = 0;
  // the node's value goes into the table; a move or the stand pat raised alpha
  bool store = false, raised = false;
  u64 qe = 0;
  u64 ep = ~p.cr & RANKS45;  // captures leave none behind
  u64 left = 0;
  List li = {};
  s32 v = 0;
  bool arrive = true;  // at a new node; else back at a parent, with moves to go on with
  for (;;) {
    bool leaf = false;  // the node's value is v
    if (arrive) {
      if (!polled && ++q.count >= POLL_EVERY && poll_root(args(), L, lane, q, ra)) return QS_ABORTED;
      polled = false;
      if (floor_lifts(sd, ra, alpha, beta)) alpha = ra - 1;
      store = raised = false;
      const bool draw = hmc >= 100 || popc(p.b1 | p.b2 | p.b3) <= 2;
      // stand pat before any move generation: the reference returns the static
      // evaluation both on a stand-pat cutoff and when no capture exists
      // (src/zeta.cl:1597-1605)
      if (!kic) {
        if (!known && !draw) ev = static_eval(p, lane);
        if (draw) ev = 0;
        leaf = draw || ev >= beta || sd >= MAXPLY;
        if (!draw && sd >= MAXPLY) lcount(cvec, C_MAXPLY, 1);
        v = ev;
      }
      if (TABLE && !leaf && !ep && !draw && any_ply(sd, popc(p.b1 | p.b2 | p.b3), MAXPLY)) {
        const u64 key = phash ^ (u64)p.stm;
        if (sd == sd0) qe = shared_load(args()->qtt + (key & args()->qmask));
        const u64 e = uf(qe);
        store = true;
        if ((e >> QT_BITS) == (key >> QT_BITS)) {
          const u32 kind = (u32)(e >> 16) & 3u;
          const s32 ts = (s32)(int16_t)(u16)e;
          leaf = kind == Q_EXACT || (kind == Q_LOWER && ts >= beta) || (kind == Q_UPPER && ts <= alpha);
          if (leaf) {
            v = ts;
            store = false;
          } else if (kind == Q_LOWER && ts > alpha) {
            alpha = ts;
            raised = true;
          }
        }
      }
      if (!leaf) {
        mcnt = gen_moves<true>(L, me, lane, p, ep, kic, 0, mbeg, true, 0, 0, li);
        left = all_moves(mcnt);
        if (mcnt < 0) {
          if (lane == 0) atomicOr(args()->err, 1u);
          return QS_FAILED;
        }
        if (draw) {
          v = 0;
          leaf = true;
        } else if (mcnt == 0 || sd >= MAXPLY) {
          if (sd >= MAXPLY) lcount(cvec, C_MAXPLY, 1);
          if (kic) v = static_eval(p, lane);
          leaf = true;
          if (TABLE && store) qt_store(p, phash, v, Q_EXACT, lane);
        } else if (!kic && ev > alpha) {
          alpha = ev;
          raised = true;
        }
      }
      ep = 0;
      hmc = 0;
    }
    if (!leaf) {
      u32 m, mk;
      if (pick_move(L, lane, mbeg, mcnt, li, left, sd + 1 < MAXPLY ? -alpha : 2 * INF, false, false, q, unused, m, mk) >= 0) {
        int w = put_planes(0, p);
        w = put32(w, 8, window(alpha, beta));
        w = put32(w, 9, (u32)mbeg | ((u32)mcnt << 16));
        w = put64(w, 10, left);
        if (TABLE) {
          w = put64(w, 12, phash);
          w = put32(w, 14, (store ? 1u : 0u) | (raised ? 2u : 0u));
        }
        if (lane < 15) L.ply[sd].w[lane] = (u32)w;
        q.nodes++;
        if (TABLE) {
          // the child's entry is on its way while the child is made
          phash ^= piece_key(mv_pfrom(m), (int)mv_from(m)) ^ piece_key(mv_pto(m), (int)mv_to(m)) ^
                   piece_key(mv_pcpt(m), (int)mv_cpt(m));
          qe = shared_load(args()->qtt + ((phash ^ (u64)(p.stm ^ 1u)) & args()->qmask));
        }
        p = apply_capture(p, m);
        const s32 t = alpha;
        alpha = -beta;
        beta = -t;
        mbeg += mcnt;
        kic = (mk & 0xFFFFu) == KEY_CHECK;
        known = (mk & 0xFFFFu) > KEY_OPEN;
        ev = (s32)(mk & 0xFFFFu) - 32768;
        sd++;
        arrive = true;
        continue;
      }
      v = alpha;
      if (TABLE && store) qt_store(p, phash, v, bound_kind(sd, ra, raised, v), lane);
    }
    // return v to the parent, and on while the parents fail high
    do {
      if (sd == sd0) {
        vout = v;
        return QS_DONE;
      }
      sd--;
      wsync();
      const int w = (int)L.ply[sd].w[lane < 15 ? lane : 0];
      get_planes(w, p);
      if (TABLE) {
        phash = get64(w, 12);
        store = get32(w, 14) & 1u;
        raised = get32(w, 14) & 2u;
      }
      p.stm ^= 1u;
      const u32 win = get32(w, 8), list = get32(w, 9);
      left = get64(w, 10);
      alpha = (s32)(int16_t)(u16)win;
      beta = (s32)win >> 16;
      mbeg = (int)(list & 0xFFFFu);
      mcnt = (int)(list >> 16);
      v = -v;
      if (floor_lifts(sd, ra, alpha, beta)) {
        alpha = ra - 1;
        raised = false;
      }
      if (v > alpha) {
        alpha = v;
        raised = true;
      }
      v = alpha;
      if (TABLE && store && alpha >= beta && bound_holds(sd, ra, true, v)) qt_store(p, phash, v, Q_LOWER, lane);
    } while (alpha >= beta);
    li = load_list(L, lane, mbeg);
    arrive = false;
  }
}

// The TT (or hint) move of a list goes first: its key takes the score, in the
// move stack and in the lanes.
__device__ __forceinline__ void first_move(Lds &L, int lane, const Node &n, List &li, u32 m, s32 score) {
  for (int k = lane; k < n.mcnt; k += 64)
    if (L.mmove[n.mbeg + k] == m) L.mkey[n.mbeg + k] = move_key(score, L.mkey[n.mbeg + k] & 0xFFFFu);
  wsync();
  li = load_list(L, lane, n.mbeg);
}

// What the search asks of its arguments at every node, in one scalar register:
// flags, the split depth (bits 8-15), the network's least depth (16-23) and
// the logarithm of the table's size (24-31, 0 = no table).
enum { CF_MLP = 1, CF_HINT = 2, CF_RECORDS = 4, CF_ABDADA = 8, CF_SERVING = 16 };
__device__ __forceinline__ u32 search_config(Args a) {
  const s32 least = a->mlp_min_depth;
  return (a->use_mlp ? CF_MLP : 0) | (a->hint ? CF_HINT : 0) | (a->recs ? CF_RECORDS : 0) | (a->workers > 1 ? CF_ABDADA : 0) |
         (a->slots ? CF_SERVING : 0) | ((u32)a->split_depth << 8) | ((u32)(least < 0 ? 0 : (least > 255 ? 255 : least)) << 16) |
         ((u32)popc(a->ttmask) << 24);
}
__device__ __forceinline__ u64 tt_mask(u32 cfg) { return (1ULL << (cfg >> 24)) - 1; }

// TABLE: none, shared (a transposition table, and with it a quiescence table and
// windows of one) or that of a search with a node budget.  The search without
// tables keeps no piece hash through quiescence and no reach: with one kernel
// for all it took 4 % longer.
template <int TABLE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 8))) void k_search(SearchArgs) {
  __shared__ Lds L;
  u32 *const mmove = L.mmove, *const mkey = L.mkey, *const killers = L.killers;
  const int lane = threadIdx.x;
  const LaneSq me = lane_sq(lane);
  L.lines[lane][0] = me.q.rank;
  L.lines[lane][1] = me.q.file;
  L.lines[lane][2] = me.q.diag;
  L.lines[lane][3] = me.q.anti;
  for (int k = lane; k < 7 * 64; k += 64) L.tab[k] = (int16_t)EVAL_SQ.v[k];
  for (;;) {
    const Args a = args();
    const bool serving = a->slots != nullptr;
    if (serving && blockIdx.x == gridDim.x - 1) {
      serve_scheduler(a, lane);
      return;
    }
    int r;
    u64 ticket = 0;
    if (serving) {
      r = serve_pick(a, lane, ticket);
    } else {
      const int hstart = (int)((blockIdx.x * 7919u) % (unsigned)(a->nroots > 0 ? a->nroots : 1));
      u32 ab = 0;
      if (lane == 0) ab = sys_load32(a->habort);
      r = uf(ab) ? -1 : pick_root(a, hstart, lane);
    }
    if (r < 0) return;
    int depth_r = a->depth;
    u32 cfg = search_config(a);

    if (serving) {
      depth_r = uf(ag_load(&a->dreq[r].depth));
      if (!(uf(ag_load(&a->dreq[r].flags)) & 1)) cfg &= ~CF_MLP;
      if (depth_r < 1) depth_r = 1;
      if (depth_r > MAXPLY - 1) depth_r = MAXPLY - 1;
    }

    // ---------------------------------------------------------------- root set-up
    // killers and counter moves start empty for every root (they persist
    // across its iterations), so a root's search does not depend on which
    // worker searched what before
    u16 *ctab = glob(a->ctab) + (size_t)blockIdx.x * NCOUNTER;
    for (int k = lane; k < MAXPLY + 2; k += 64) killers[k] = 0;
    for (int k = lane; k < NCOUNTER / 8; k += 64) ((uint4 *)ctab)[k] = make_uint4(0u, 0u, 0u, 0u);
    if (lane == 0) {
      L.root = r;
      L.depth = depth_r;
      L.ticket = ticket;
      L.final_score = 0;
      L.final_move = 0;
      const s32 hl = a->hist ? a->hlen[r] : 0;
      L.hlen = hl > ZETA_HISTORY ? ZETA_HISTORY : (hl < 0 ? 0 : hl);
    }
    if (TABLE == T_SHARED) {
      // (each with its place: a position that occurred twice would cancel itself)
      u64 h = 0;
      wsync();
      for (int k = lane; k < L.hlen; k += 64)
        h ^= hash_mix(a->hist[(size_t)r * ZETA_HISTORY + k] + (u64)(k + 1) * 0xD1B54A32D192ED03ULL);
      h = wave_xor(h);
      if (lane == 0) L.hsalt = h;
    }
    wsync();

    // per-root statistics in one vector register (counter k in lane k) rather
    // than in scalar registers, which the node state needs
    u32 cvec = 0;
    Poll poll = {};
    poll_load(a, r, lane, poll);
    bool aborted = false, failed = false;

    // a worker joining a root that others are already searching starts at the
    // iteration in progress: the earlier ones would only repeat work whose
    // moves are in the shared TT (the final iteration alone sets the score)
    int id0 = 1;
    if (lane == 0) id0 = (__atomic_load_n(&a->depth_done[r], __ATOMIC_RELAXED) & (serving ? 0xFFFF : ~0)) + 1;
    id0 = uf(id0);
    id0 = id0 < 1 ? 1 : (id0 > depth_r ? depth_r : id0);
    for (int id = id0; !aborted && !failed && id <= uf(L.depth); id++) {
      const Args a = args();
      // the best score any worker has found for a root move in this
      // iteration (refreshed at the poll); -INF until one has
      s32 ra = -INF;
      {
        // a worker joining the iteration starts from the bound the root's
        // other workers have published
        u64 rb = 0;
        if (lane == 0) {
          L.iteration = id;
          L.best_score = 0;  // DRAWSCORE until a root move raises alpha (src/zeta.cl:986)
          L.best_move = 0;
          rb = ag_load(&a->rbound[r]);
        }
        rb = uf(rb);
        if ((rb >> 32) == (uf(L.ticket) & 0xFFFFFFFFULL) && (int)((rb >> 16) & 0xFFFF) == id)
          ra = (s32)(rb & 0xFFFF) - 32768;
      }
      const int r = uf(L.root);
      Node n;
      {
        // (the root position is re-read at every iteration rather than held in
        // scalar registers through the search)
        u64 q[8];
        if (serving) {
          const u64 *const rootq = (const u64 *)a->dreq[r].pos;
          for (int k = 0; k < 8; k++) q[k] = uf(ag_load(&rootq[k]));
        } else {
          const u64 *const rootq = glob(a->roots) + (size_t)r * 8;
          for (int k = 0; k < 8; k++) q[k] = uf(rootq[k]);
        }
        n.p.b0 = q[0];
        n.p.b1 = q[1];
        n.p.b2 = q[2];
        n.p.b3 = q[3];
        n.p.cr = q[4];
        n.p.stm = (u32)(q[7] & 1u);
        n.hash = q[5];
        n.hmc = (u32)(q[6] & 0xFF);
      }
      n.phash = hash_pieces(n.p);
      n.alpha = -INF;
      n.beta = INF;
      n.depth = id;
      n.mbeg = 0;
      n.busy = false;
      n.move = 0;
      {
        const u64 occ = n.p.b1 | n.p.b2 | n.p.b3;
        const u64 kbb = n.p.b1 & n.p.b2 & ~n.p.b3 & (n.p.stm ? n.p.b0 : n.p.b0 ^ occ);
        n.kic = king_attacked(n.p, lds_lines(L, kbb ? lsb(kbb) : 0), kbb, n.p.stm ^ 1u);
      }
      int sd = 1;
      u32 lastmove = 0;    // the move that led to the node being entered
      s32 v = 0;
      List li = {};
      s32 qev = 0;  // S_QS: the node's evaluation, if its parent knows it
      bool qknown = false;
      int state = S_ENTER;
      bool again = false;  // S_NEXT: the move that a window of one was too small for

      for (;;) {
        const Args a = args();  // loads of arguments stay in this pass
        if (state == S_ENTER) {
          // ---------------- ENTER: extend, generate, terminal tests
          if (++poll.count >= POLL_EVERY && poll_root(a, L, lane, poll, ra)) {
            aborted = true;
            break;
          }
          const int plyn = sd - 1;
          if (n.kic || is_promo(lastmove)) n.depth++;
          const bool qs = n.depth <= 0;
          // Another worker's root move reached ra: at the root's side (odd
          // plies from 3 on) a value at or below ra - 1 cannot make this root
          // move the best, so the window starts there.  A root move then
          // reports max(its value, a bound below ra) -- below the best root
          // score, which stays exact, as does its move.
          if (floor_lifts(sd, ra, n.alpha, n.beta)) n.alpha = ra - 1;
          n.best = 0;
          n.pass2 = false;
          n.ndefer = 0;
          n.searched = 0;
          n.mcnt = 0;
          n.ttm = 0;
          n.reach = 0;
          if (qs) {
            // a quiescence node whose evaluation its parent did not know
            qknown = false;
            state = S_QS;
            continue;
          }
          const u64 ttmask = TABLE ? tt_mask(cfg) : 0;
          const u64 key = tt_key(n.hash, n.p.cr);
          u32x4 tte = {0u, 0u, 0u, 0u};
          if (TABLE && sd > 1) tte = tt_load<TABLE>(a->tt + 2 * (key & ttmask));
          const bool by_path = TABLE == T_SHARED && sd > 1 && n.depth >= PATH_DEPTH && n.hmc != 0;
          u64 key2 = 0;
          u32x4 tte2 = {0u, 0u, 0u, 0u};
          if (by_path) {
            key2 = key ^ path_key(L, n, sd, lane);
            tte2 = tt_load<TABLE>(a->tt + 2 * (key2 & ttmask));
          }
          // draws that hold with and without moves
          if (sd > 1 && (n.hmc >= 100 || popc(n.p.b1 | n.p.b2 | n.p.b3) <= 2)) {
            v = 0;
            state = S_RETURN;
            continue;
          }
          bool repeated = false;
          if (sd > 1 && n.hmc >= 2) {
            // repetition against plies plyn-2, plyn-4, .. >= plyn-hmc: the
            // searched path, then the game history before the root
            bool hit = false;
            const int nn = plyn - 2 - 2 * lane;
            if (nn >= plyn - (int)n.hmc) {
              if (nn >= 0) {
                const u32 *const w = L.ply[nn + 1].w;
                hit = (((u64)w[W_HASH + 1] << 32) | w[W_HASH]) == n.hash;
              } else if (-nn - 1 < L.hlen) {
                hit = a->hist[(size_t)L.root * ZETA_HISTORY + (-nn - 1)] == n.hash;
              }
            }
            repeated = __ballot(hit) != 0;
          }
          // TT probe, before any move is generated (a stored node had moves):
          // move for ordering; score where no path to the node changes it
          u32 ttmove = 0;
          if (TABLE && sd > 1) {
            lcount(cvec, C_TT_PROBE, 1);
            bool cut = false;
            auto use = [&](const u32x4 &t, u64 k, bool path) {
              const u64 w0 = uf(((u64)t.y << 32) | t.x), w1 = uf(((u64)t.w << 32) | t.z);
              if ((w0 ^ w1) != k || !((w1 >> 57) & 1)) return;
              if (!path) lcount(cvec, C_TT_HIT, 1);
              if (!ttmove) ttmove = (u32)w1;
              s32 ts = (s32)(int16_t)(u16)(w1 >> 32);
              const int d = (int)((w1 >> 48) & 0xFF);
              const u32 reach = (u32)(w1 >> 59) & 3u;
              if (is_mate(ts) && ts > 0) ts -= plyn;
              if (is_mate(ts) && ts < 0) ts += plyn;
              if (((w1 >> 56) & 1) && d == n.depth && ts > -INF && ts < INF && !repeated && sd < MAXPLY &&
                  (path || path_free(L, n, reach, sd))) {
                // an upper bound at or below alpha: the node fails low; a
                // lower bound raises alpha
                const bool upper = (w1 >> 58) & 1;
                if (upper ? ts <= n.alpha : ts > n.alpha) {
                  lcount(cvec, C_TT_CUT, 1);
                  n.reach = n.reach > reach ? n.reach : reach;
                  if (!upper) n.alpha = ts;
                  cut = upper || n.alpha >= n.beta;
                }
              }
            };
            use(tte, key, false);
            if (by_path && !cut) use(tte2, key2, true);
            if (cut) {
              v = n.alpha;
              state = S_RETURN;
              continue;
            }
          }
          u16 *const ctab = glob(a->ctab) + (size_t)blockIdx.x * NCOUNTER;
          const u32 kil = killers[sd], cm = (u32)ctab[counter_index(lastmove)];
          const int total = gen_moves<false>(L, me, lane, n.p, ~n.p.cr & RANKS45, n.kic, n.hmc, n.mbeg,
                                             n.depth == 1 && sd + 1 < MAXPLY, kil, cm, li);
          if (total < 0) {
            if (lane == 0) atomicOr(a->err, 1u);
            failed = true;
            break;
          }
          n.mcnt = total;
          n.left = all_moves(total);
          if ((cfg & CF_MLP) && n.depth >= (s32)((cfg >> 16) & 0xFFu) && total > 1) {
            // every move's score is its plain score plus the network's, in
            // plain-score units (zm::PLAIN_PER_LOGIT per unit of the network's
            // output, the scale the ranking loss is trained at); the TT move
            // still goes first
            mlp_score_moves(a, n.p, n.mbeg, total, lane, L.hpos, mmove, [&](int k, s32 out) {
              const u32 old = mkey[k];
              s32 sc = (s32)(old >> 16) - 32768 + out * zm::PLAIN_PER_LOGIT / 256;
              sc = sc > 31999 ? 31999 : (sc < -31999 ? -31999 : sc);
              mkey[k] = move_key(sc, old & 0xFFFFu);
            });
            wsync();
            lcount(cvec, C_MLP_NODES, 1);
            li = load_list(L, lane, n.mbeg);
          }
          // terminal / draw tests in the reference's order (src/zeta.cl:1554-1609)
          state = S_NEXT;
          if (repeated && total > 0) {
            v = 0;
            state = S_RETURN;
          } else if (total == 0) {
            v = n.kic ? -INF + plyn : 0;
            state = S_RETURN;
          } else if (sd >= MAXPLY) {
            lcount(cvec, C_MAXPLY, 1);
            v = static_eval(n.p, lane);
            state = S_RETURN;
          } else {
            if (TABLE && ttmove) {
              n.ttm = ttmove;
              first_move(L, lane, n, li, ttmove, TTMOVE_SCORE);
            }
            if (TABLE && (cfg & CF_HINT)) {
              // the hint table (a completed search's table): its move first
              const u32x4 he = *glob((const u32x4 *)(a->hint + 2 * (key & ttmask)));
              const u64 h0 = uf(((u64)he.y << 32) | he.x), h1 = uf(((u64)he.w << 32) | he.z);
              if ((h0 ^ h1) == key && ((h1 >> 57) & 1)) {
                first_move(L, lane, n, li, (u32)h1, HINT_SCORE);
              }
            }
          }
          wsync();
          continue;
        }

        if (state == S_NEXT) {
          // ---------------- NEXT: pick the best remaining move
          u32 m, mk;
          int k = 0;
          if (TABLE == T_SHARED && again) {
            m = n.move;
            mk = n.child;
          } else {
            k = pick_move(L, lane, n.mbeg, n.mcnt, li, n.left, n.depth == 1 && sd + 1 < MAXPLY ? -n.alpha : 2 * INF,
                          n.ndefer > 0, n.pass2, poll, n.searched, m, mk);
          }
          if (k < 0) {
            if (!n.pass2 && n.ndefer > 0) {
              n.pass2 = true;
              continue;
            }
            v = n.alpha;
            if (TABLE) lcount(cvec, C_TT_STORE, tt_store<TABLE>(a, tt_mask(cfg), L, n, sd, ra, lane));
            state = S_RETURN;
            continue;
          }
          const Pos c = apply(n.p, m, false);
          const bool quiet = (mk & 0xFFFFu) > KEY_OPEN;
          // Once a move has been searched, the others are expected to stay at
          // or below the floor: a window of one shows it with fewer nodes, and
          // a move that exceeds it is searched again with the node's window.
          // Six batches of 1024 positions, depth 4: 1101 -> 698 ms.
          const s32 lo = floor_of(n, sd, ra);
          const bool repeat = TABLE == T_SHARED && again;
          again = false;
          n.scout = TABLE == T_SHARED && !repeat && n.searched > 0 && n.beta - lo > 1;
          n.child = mk & 0xFFFFu;
          n.floor = lo;
          const s32 hi = n.scout ? lo + 1 : n.beta;
          u64 ch = 0, cph = 0;
          if (TABLE == T_SHARED || !quiet) child_hash(n, m, c, ch, cph);
          if (quiet) {
            // a quiescence node, not in check, its evaluation known
            if (!n.pass2 && !repeat) n.searched++;
            poll.nodes++;
            n.move = m;
            save(L.ply[sd], n, lane);
            n.alpha = -hi;
            n.beta = -lo;
            n.hmc = child_hmc(n.hmc, m);
            n.mbeg += n.mcnt;
            n.p = c;
            n.busy = false;
            n.kic = false;
            qev = (s32)(mk & 0xFFFFu) - 32768;
            qknown = true;
            n.phash = cph;
            sd++;
            wsync();
            state = S_QS;
            continue;
          }
          // ABDADA: defer a sibling that another worker is already searching
          bool cbusy = false;
          if ((cfg & CF_ABDADA) && n.depth - 1 >= (s32)((cfg >> 8) & 0xFFu)) {
            u32 *const bp = glob(a->busy) + ((u32)(tt_key(ch, c.cr) >> 40) & a->busymask);
            // test and mark in one: workers that start on a root together walk
            // in step, and with a load ahead of the mark they all find the child
            // free (16 workers on a position, depth 5: 184 -> 159 ms)
            u32 b = 0;
            if (lane == 0) b = atomicAdd(bp, 1u);
            b = uf(b);
            // batch searches defer a busy first child too, from ply 3 down:
            // a worker that finds it busy moves on to the siblings and comes
            // back to it in the second pass, which keeps helpers off the
            // path every worker starts on.  At the root and ply 2 the first
            // child is searched by every worker that reaches it: a sibling
            // searched before the first child has set the root's bound has
            // no bound to fail against (six positions, depth 5, 128 workers:
            // 107 ms this way, 130 with the deferral from ply 2, 103 from
            // ply 4; six batches of 250 with the network 270, 304, 267).
            // Served requests defer only later siblings
            if (!n.pass2 && !repeat && b && (n.searched > 0 || (!(cfg & CF_SERVING) && sd >= 3))) {
              n.left |= 1ULL << (k & 63);
              if (lane == 0) {
                atomicSub(bp, 1u);
                mkey[n.mbeg + k] = mk;
                mmove[n.mbeg + k] = m | DEFERRED;
              }
              n.ndefer++;
              lcount(cvec, C_DEFER, 1);
              wsync();
              continue;
            }
            cbusy = true;
          }
          if (!n.pass2 && !repeat) n.searched++;
          poll.nodes++;
          n.move = m;
          save(L.ply[sd], n, lane);
          // descend (ENTER sets the rest)
          n.hmc = child_hmc(n.hmc, m);
          n.p = c;
          n.hash = ch;
          n.phash = cph;
          n.alpha = -hi;
          n.beta = -lo;
          n.depth--;
          n.mbeg += n.mcnt;
          n.busy = cbusy;
          n.kic = (mk & 0xFFFFu) == KEY_CHECK;
          lastmove = m;
          sd++;
          wsync();
          state = S_ENTER;
          continue;
        }

        if (state == S_QS) {
          // ---------------- a quiescence node and all below it
          const int st = qsearch<TABLE == T_SHARED>(L, me, lane, n.p, n.alpha, n.beta, n.hmc, sd, n.mbeg, qev, qknown, n.kic, !qknown, n.phash,
                                 poll, ra,
                                 cvec, v);
          if (st != QS_DONE) {
            aborted = st == QS_ABORTED;
            failed = !aborted;
            break;
          }
        }

        // ---------------- RETURN v from node sd
        if (n.busy) busy_release(a, n.hash, n.p.cr, lane);
        if (sd == 1) break;
        // (quiescence nodes are not tested for repetition)
        const u32 below = state == S_QS || n.hmc == 0 ? 0u : (n.reach < 3 ? n.reach + 1 : 3u);
        sd--;
        wsync();
        restore(L.ply[sd], n, lane);
        if (TABLE) n.reach = n.reach > below ? n.reach : below;
        const s32 sc = -v;
        if (floor_lifts(sd, ra, n.alpha, n.beta)) {
          // the root bound rose while this node's children were searched:
          // its best move so far is below it, so no lower bound stands
          n.alpha = ra - 1;
          n.best = 0;
        }
        // (the floor it was searched with: the root's bound may have risen since)
        if (TABLE == T_SHARED && n.scout && sc > n.floor && sc < n.beta) {
          again = true;
          state = S_NEXT;
          wsync();
          continue;
        }
        if (sc > n.alpha) {
          n.alpha = sc;
          n.best = n.move;
          if (sd == 1 && lane == 0) {
            L.best_score = sc;
            L.best_move = n.move;
            atomicMax((unsigned long long *)&a->rbound[L.root],
                      (unsigned long long)(((L.ticket & 0xFFFFFFFFULL) << 32) | ((u64)(u32)L.iteration << 16) |
                                           (u64)(u16)(sc + 32768)));
          }
        }
        const bool cut = n.alpha >= n.beta;
        if (cut || reply_suffices(sd, ra, n.alpha)) {
          const u32 last = last_move(L, sd);
          u16 *const ctab = glob(a->ctab) + (size_t)blockIdx.x * NCOUNTER;
          // the move refuted the one before it (not where only the root's bound
          // ended the node, here or below)
          const bool refutes = cut && bound_holds(sd, ra, true, n.alpha);
          if (refutes && (cfg & CF_RECORDS) && n.depth >= 1 && n.searched >= 1 && n.mcnt >= 2 &&
              ((u32)(n.hash >> 40) & a->rec_mask) == 0) {
            u32 nrec = 0;
            log_pairs(a, n, lane, mmove, L.tab, n.ttm, killers[sd], (u32)ctab[counter_index(last)], nrec);
            lcount(cvec, C_RECORDS, nrec);
          }
          // a quiet move that fails high becomes the ply's killer and the
          // counter move of the move before it (src/zeta.cl:1916-1933)
          if (refutes && ((mv_pcpt(n.move) >> 1) & 7) == PNONE && lane == 0) {
            killers[sd] = n.move;
            ctab[counter_index(last)] = counter_code(n.move);
          }
          v = n.alpha;
          if (TABLE) lcount(cvec, C_TT_STORE, tt_store<TABLE>(a, tt_mask(cfg), L, n, sd, ra, lane));
          state = S_RETURN;
        } else {
          li = load_list(L, lane, n.mbeg);
          state = S_NEXT;
        }
        wsync();
      }

      if (aborted || failed) {
        // release the ABDADA marks still held along the path
        const Args a = args();
        if (n.busy) busy_release(a, n.hash, n.p.cr, lane);
        wsync();
        for (int k = 2; k < sd; k++) {
          Node y;
          restore(L.ply[k], y, lane);
          if (y.busy) busy_release(a, y.hash, y.p.cr, lane);
        }
        break;
      }
      const Args b = args();
      wsync();
      s32 fs = uf(L.best_score);
      if (fs == INF || fs == -INF) fs = 0;  // src/search.c:137
      if (lane == 0) {
        L.final_score = fs;
        L.final_move = L.best_move;
        if (cfg & CF_SERVING) slot_max_depth(&b->depth_done[L.root], L.ticket, id);
        else atomicMax(&b->depth_done[L.root], id);
      }
      // a mate within this iteration's depth is the score of every deeper
      // iteration too: iterative deepening stops there (src/search.c:177-186)
      if (is_mate(fs) && id >= (fs > 0 ? INF - fs : INF + fs)) break;
    }

    // ---------------------------------------------------------------- publish
    wsync();
    const s32 final_score = L.final_score;
    const u32 final_move = L.final_move;
    const u64 nodes = poll.nodes;
    ticket = L.ticket;
    r = L.root;
    if (lane < C_NODES && cvec) atomicAdd((unsigned long long *)&a->ctr[lane], (unsigned long long)cvec);
    if (lane == 0) {
      // before leaving: the last worker to leave publishes the request's
      // count, which then holds every worker's nodes
      if (serving) slot_add_nodes(&a->nodes[r], ticket, nodes);
      else atomicAdd((unsigned long long *)&a->nodes[r], (unsigned long long)nodes);
      atomicAdd((unsigned long long *)&a->ctr[C_NODES], (unsigned long long)nodes);
      if (serving) {
        serve_leave(a, r, ticket, aborted, failed, final_score, final_move);
      } else {
        if (!aborted && !failed && atomicCAS(&a->done[r], 0u, 1u) == 0u) {
          a->score[r] = final_score;
          a->bestmove[r] = final_move;
        }
        if (failed) atomicCAS(&a->done[r], 0u, 2u);
        atomicSub(&a->nworkers[r], 1);
      }
    }
    wsync();
  }
}

// the search's learned-ordering routine applied to given moves (for tests and
// external callers): one wave per position, up to MSTACK moves each
__global__ __launch_bounds__(64) void k_mlp_score(SearchArgs, const u64 *pos, const u32 *moves, const int *off,
                                                 float *out) {
  __shared__ u32 mmove[MSTACK];
  __shared__ float hpos[zm::NH1];
  const Args a = args();
  const int lane = threadIdx.x, i = blockIdx.x;
  const u64 *q = pos + (size_t)i * 8;
  Pos p;
  p.b0 = q[0];
  p.b1 = q[1];
  p.b2 = q[2];
  p.b3 = q[3];
  p.cr = q[4];
  p.stm = (u32)(q[7] & 1u);
  const int b = off[i], n = off[i + 1] - off[i];
  for (int k = lane; k < n; k += 64) mmove[k] = moves[b + k];
  wsync();
  mlp_score_moves(a, p, 0, n, lane, hpos, mmove, [&](int k, s32 sc) { out[b + k] = (float)sc / 256.f; });
}

// Principal variation after a search: the best root move, then the moves the
// transposition table holds for the positions that follow, each checked to
// be legal (the reference walks its TT the same way, src/zeta.cl:2450-2512).
// One thread per root; stops at a missing or mismatching entry.
__global__ void k_pv(const u64 *roots, const u32 *bestmove, int n, int len, const u64 *tt, u64 ttmask,
                     u32 *pv) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  u32 *out = pv + (size_t)i * len;
  for (int k = 0; k < len; k++) out[k] = 0;
  const u64 *q = roots + (size_t)i * 8;
  Pos p;
  p.b0 = q[0];
  p.b1 = q[1];
  p.b2 = q[2];
  p.b3 = q[3];
  p.cr = q[4];
  p.stm = (u32)(q[7] & 1u);
  Node nd;
  nd.hash = q[5];
  nd.phash = hash_pieces(p);
  u32 m = bestmove[i];
  for (int k = 0; k < len && m; k++) {
    const int f = (int)mv_from(m), t = (int)mv_to(m);
    Legal L;
    analyse(p, L);
    if (!((L.own >> f) & 1) || !((piece_targets(p, L, f, false) >> t) & 1) || make_code(p, f, t) != m) break;
    out[k] = m;
    const Pos c = apply(p, m, false);
    u64 h, ph;
    child_hash(nd, m, c, h, ph);
    nd.hash = h;
    nd.phash = ph;
    p = c;
    m = 0;
    if (ttmask) {
      const u64 key = tt_key(h, c.cr);
      const u64 w0 = tt[2 * (key & ttmask)], w1 = tt[2 * (key & ttmask) + 1];
      if ((w0 ^ w1) == key && ((w1 >> 57) & 1) && !((w1 >> 58) & 1)) m = (u32)w1;  // a move that raised alpha
    }
  }
}

__global__ void k_clear_u64(u64 *p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0;
}

struct SearchState {
  zr::DevBuf tt, busy, roots, queue, done, nworkers, score, bestmove, nodes, depth_done, err, ctr, hist, hlen, pv, hint,
      rbound, ctab, qtt;
  u64 tt_entries = 0;
  u64 last_ctr[C_NCTR] = {0};
};
SearchState g_ss;

// the quiescence table of a call with `grid` workers, empty: 32 KB a worker,
// between 2 MB (QT_BITS bits of index) and 32 MB
int qt_clear(unsigned grid, hipStream_t st, SearchArgs &sa) {
  u64 entries = QT_MIN;
  while (entries < QT_MAX && entries < (u64)grid * QT_WORKER) entries *= 2;
  const int r = zr::ensure(g_ss.qtt, entries * 8);
  if (r) return r;
  hipLaunchKernelGGL(k_clear_u64, dim3((unsigned)(entries / 1024)), dim3(256), 0, st, (u64 *)g_ss.qtt.p, (size_t)entries);
  ZCHECK(hipGetLastError());
  sa.qtt = (u64 *)g_ss.qtt.p;
  sa.qmask = entries - 1;
  return 0;
}

}  // namespace

const zm::Weights *mlp_weights();
void *records_buffer(u64 *cap, u64 **count);

void search_release() {
  zr::release(g_ss.tt); zr::release(g_ss.busy); zr::release(g_ss.roots); zr::release(g_ss.queue);
  zr::release(g_ss.done); zr::release(g_ss.nworkers); zr::release(g_ss.score); zr::release(g_ss.bestmove);
  zr::release(g_ss.nodes); zr::release(g_ss.depth_done); zr::release(g_ss.err);
  zr::release(g_ss.ctr); zr::release(g_ss.hist); zr::release(g_ss.hlen); zr::release(g_ss.pv);
  zr::release(g_ss.hint); zr::release(g_ss.rbound); zr::release(g_ss.ctab); zr::release(g_ss.qtt);
  g_ss.tt_entries = 0;
}

extern "C" int zeta_search_batch(const zeta_pos *pos, int n, const zeta_search_opts *opts, zeta_result *res) {
  int r = zr::require_up();
  if (r) return r;
  if (n < 0 || (n > 0 && (!pos || !res)) || !opts) return zr::fail(ZETA_EINVAL, "search: bad arguments");
  if (opts->depth < 1 || opts->depth > 40) return zr::fail(ZETA_EINVAL, "search: depth %d out of range", opts->depth);
  if (opts->split_depth < 0 || opts->split_depth > 40 || opts->waves_per_simd < 0 || opts->waves_per_simd > 16)
    return zr::fail(ZETA_EINVAL, "search: split_depth %d / waves_per_simd %d out of range", opts->split_depth,
                    opts->waves_per_simd);
  if (n == 0) return ZETA_OK;
  const int workers = opts->workers < 1 ? 1 : (opts->workers > 1024 ? 1024 : opts->workers);
  hipStream_t st = zr::ctx().stream;
  const int tt_log2 = opts->tt_log2 < 0 ? zr::ctx().cfg.tt_log2 : opts->tt_log2;
  const u64 tt_entries = tt_log2 > 0 ? (1ULL << tt_log2) : 0;
  if (tt_log2 > 34) return zr::fail(ZETA_EINVAL, "search: tt_log2 %d too large", tt_log2);
  const u32 busy_entries = 1u << 20;
  if ((r = zr::ensure(g_ss.roots, (size_t)n * sizeof(zeta_pos))) || (r = zr::ensure(g_ss.queue, 64)) ||
      (r = zr::ensure(g_ss.done, (size_t)n * 4)) || (r = zr::ensure(g_ss.nworkers, (size_t)n * 4)) ||
      (r = zr::ensure(g_ss.score, (size_t)n * 4)) || (r = zr::ensure(g_ss.bestmove, (size_t)n * 4)) ||
      (r = zr::ensure(g_ss.nodes, (size_t)n * 8)) || (r = zr::ensure(g_ss.depth_done, (size_t)n * 4)) ||
      (r = zr::ensure(g_ss.rbound, (size_t)n * 8)) ||
      (r = zr::ensure(g_ss.err, 64)) || (r = zr::ensure(g_ss.ctr, C_NCTR * 8)) ||
      (r = zr::ensure(g_ss.busy, (size_t)busy_entries * 4)))
    return r;
  if (opts->order_hint && (!tt_entries || g_ss.tt_entries != tt_entries))
    return zr::fail(ZETA_EINVAL, "search: order_hint needs the previous batch's table of the same size");
  if (tt_entries) {
    if ((r = zr::ensure(g_ss.tt, tt_entries * 16))) return r;
    if (opts->order_hint) {
      // the previous batch's table becomes the hint table before it is cleared
      if ((r = zr::ensure(g_ss.hint, tt_entries * 16))) return r;
      ZCHECK(hipMemcpyAsync(g_ss.hint.p, g_ss.tt.p, tt_entries * 16, hipMemcpyDeviceToDevice, st));
    }
    if (g_ss.tt_entries != tt_entries || opts->clear_tt) {
      ZLAUNCH(zr::K_SEARCH, 0, k_clear_u64, 4096, 256, 0, (u64 *)g_ss.tt.p, (size_t)(tt_entries * 2));
      g_ss.tt_entries = tt_entries;
    }
  }
  ZCHECK(hipMemcpyAsync(g_ss.roots.p, pos, (size_t)n * sizeof(zeta_pos), hipMemcpyHostToDevice, st));
  ZCHECK(hipMemsetAsync(g_ss.queue.p, 0, 64, st));
  ZCHECK(hipMemsetAsync(g_ss.done.p, 0, (size_t)n * 4, st));
  ZCHECK(hipMemsetAsync(g_ss.nworkers.p, 0, (size_t)n * 4, st));
  ZCHECK(hipMemsetAsync(g_ss.score.p, 0, (size_t)n * 4, st));
  ZCHECK(hipMemsetAsync(g_ss.bestmove.p, 0, (size_t)n * 4, st));
  ZCHECK(hipMemsetAsync(g_ss.nodes.p, 0, (size_t)n * 8, st));
  ZCHECK(hipMemsetAsync(g_ss.depth_done.p, 0, (size_t)n * 4, st));
  ZCHECK(hipMemsetAsync(g_ss.rbound.p, 0, (size_t)n * 8, st));
  ZCHECK(hipMemsetAsync(g_ss.err.p, 0, 64, st));
  ZCHECK(hipMemsetAsync(g_ss.ctr.p, 0, C_NCTR * 8, st));
  ZCHECK(hipMemsetAsync(g_ss.busy.p, 0, (size_t)busy_entries * 4, st));

  const int table = !tt_entries ? T_NONE : (opts->max_nodes ? T_BUDGET : T_SHARED);
  const auto kernel = table == T_NONE ? k_search<T_NONE> : (table == T_BUDGET ? k_search<T_BUDGET> : k_search<T_SHARED>);
  int per_cu = 0;
  ZCHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 64, 0));
  if (opts->waves_per_simd > 0 && 4 * opts->waves_per_simd < per_cu) per_cu = 4 * opts->waves_per_simd;
  if (per_cu < 1) per_cu = 1;
  const u64 cap = (u64)per_cu * (u64)zr::ctx().cu_count;
  u64 want = (u64)n * (u64)workers;
  const unsigned grid = (unsigned)(want < cap ? want : cap);
  if ((r = zr::ensure(g_ss.ctab, (size_t)grid * NCOUNTER * 2))) return r;

  SearchArgs sa;
  sa.roots = (const u64 *)g_ss.roots.p;
  sa.nroots = n;
  sa.depth = opts->depth;
  sa.workers = workers;
  sa.split_depth = opts->split_depth > 0 ? opts->split_depth : default_split(workers);
  sa.tt = (u64 *)g_ss.tt.p;
  sa.ttmask = tt_entries ? tt_entries - 1 : 0;
  sa.qtt = nullptr;
  sa.qmask = 0;
  if (table == T_SHARED && (r = qt_clear(grid, st, sa))) return r;
  sa.hint = opts->order_hint ? (const u64 *)g_ss.hint.p : nullptr;
  sa.rbound = (u64 *)g_ss.rbound.p;
  sa.busy = (u32 *)g_ss.busy.p;
  sa.busymask = busy_entries - 1;
  sa.ctab = (u16 *)g_ss.ctab.p;
  sa.queue = (int *)g_ss.queue.p;
  sa.done = (u32 *)g_ss.done.p;
  sa.nworkers = (int *)g_ss.nworkers.p;
  sa.score = (s32 *)g_ss.score.p;
  sa.bestmove = (u32 *)g_ss.bestmove.p;
  sa.nodes = (u64 *)g_ss.nodes.p;
  sa.depth_done = (s32 *)g_ss.depth_done.p;
  sa.err = (u32 *)g_ss.err.p;
  sa.habort = zr::ctx().abort_dev;
  sa.max_nodes = opts->max_nodes;
  sa.ctr = (u64 *)g_ss.ctr.p;
  sa.use_mlp = 0;
  sa.mlp_min_depth = opts->mlp_min_depth;
  memset(&sa.w, 0, sizeof(sa.w));
  if (opts->use_mlp) {
    const zm::Weights *w = mlp_weights();
    if (!w) return zr::fail(ZETA_ESTATE, "search: use_mlp set but no network loaded (zeta_mlp_init/zeta_mlp_set)");
    sa.w = *w;
    sa.use_mlp = 1;
  }
  sa.recs = nullptr;
  sa.rec_count = nullptr;
  sa.rec_cap = 0;
  sa.rec_mask = (opts->log_shift > 0 && opts->log_shift < 24) ? ((1u << opts->log_shift) - 1u) : 0u;
  sa.hist = nullptr;
  sa.hlen = nullptr;
  if (opts->history) {
    if (!opts->history_len) return zr::fail(ZETA_EINVAL, "search: history without history_len");
    if ((r = zr::ensure(g_ss.hist, (size_t)n * ZETA_HISTORY * 8)) || (r = zr::ensure(g_ss.hlen, (size_t)n * 4)))
      return r;
    ZCHECK(hipMemcpyAsync(g_ss.hist.p, opts->history, (size_t)n * ZETA_HISTORY * 8, hipMemcpyHostToDevice, st));
    ZCHECK(hipMemcpyAsync(g_ss.hlen.p, opts->history_len, (size_t)n * 4, hipMemcpyHostToDevice, st));
    sa.hist = (const u64 *)g_ss.hist.p;
    sa.hlen = (const s32 *)g_ss.hlen.p;
  }
  sa.sh = nullptr;
  sa.squeue = nullptr;
  sa.sack = nullptr;
  sa.scancel = nullptr;
  sa.slots = nullptr;
  sa.nslots = 0;
  sa.qcap = 0;
  sa.sv = nullptr;
  sa.sw = nullptr;
  sa.dreq = nullptr;
  sa.dcancel = nullptr;
  sa.watchdog_ticks = 0;
  if (opts->log_records) {
    u64 cap = 0, *cnt = nullptr;
    void *recs = records_buffer(&cap, &cnt);
    if (!recs || !cap) return zr::fail(ZETA_ESTATE, "search: log_records set but no record buffer (zeta_records_reserve)");
    sa.recs = (u64 *)recs;
    sa.rec_count = cnt;
    sa.rec_cap = cap;
  }
  ZLAUNCH(zr::K_SEARCH, (u64)n, kernel, grid, 64, 0, sa);

  std::vector<s32> score(n), dd(n);
  std::vector<u32> bm(n), done(n);
  std::vector<u64> nodes(n);
  u32 err = 0;
  ZCHECK(hipMemcpyAsync(score.data(), g_ss.score.p, (size_t)n * 4, hipMemcpyDeviceToHost, st));
  ZCHECK(hipMemcpyAsync(bm.data(), g_ss.bestmove.p, (size_t)n * 4, hipMemcpyDeviceToHost, st));
  ZCHECK(hipMemcpyAsync(done.data(), g_ss.done.p, (size_t)n * 4, hipMemcpyDeviceToHost, st));
  ZCHECK(hipMemcpyAsync(nodes.data(), g_ss.nodes.p, (size_t)n * 8, hipMemcpyDeviceToHost, st));
  ZCHECK(hipMemcpyAsync(dd.data(), g_ss.depth_done.p, (size_t)n * 4, hipMemcpyDeviceToHost, st));
  ZCHECK(hipMemcpyAsync(&err, g_ss.err.p, 4, hipMemcpyDeviceToHost, st));
  ZCHECK(hipMemcpyAsync(g_ss.last_ctr, g_ss.ctr.p, sizeof(g_ss.last_ctr), hipMemcpyDeviceToHost, st));
  ZCHECK(hipStreamSynchronize(st));
  zr::time_collect();
  // a root the workers left without a result was stopped by zeta_search_abort
  const bool host_abort = __atomic_load_n(zr::ctx().abort_host, __ATOMIC_ACQUIRE) != 0u;
  int incomplete = -1;
  for (int i = 0; i < n; i++) {
    res[i].score = score[i];
    res[i].bestmove = bm[i];
    res[i].nodes = nodes[i];
    res[i].depth = dd[i];
    res[i].status = done[i] == 1 ? ZETA_OK
                  : done[i] == 2 ? ZETA_ENOMEM
                  : done[i] == 3 ? ZETA_EBUDGET
                  : host_abort ? ZETA_ECANCELED : ZETA_ESTATE;
    if (res[i].status == ZETA_ESTATE && incomplete < 0) incomplete = i;
  }
  if (opts->pv && opts->pv_len > 0) {
    const int len = opts->pv_len > MAXPLY ? MAXPLY : opts->pv_len;
    if ((r = zr::ensure(g_ss.pv, (size_t)n * len * 4))) return r;
    hipLaunchKernelGGL(k_pv, dim3((n + 63) / 64), dim3(64), 0, st, (const u64 *)g_ss.roots.p,
                       (const u32 *)g_ss.bestmove.p, n, len, (const u64 *)g_ss.tt.p, sa.ttmask, (u32 *)g_ss.pv.p);
    ZCHECK(hipGetLastError());
    std::vector<u32> pvh((size_t)n * len);
    ZCHECK(hipMemcpyAsync(pvh.data(), g_ss.pv.p, pvh.size() * 4, hipMemcpyDeviceToHost, st));
    ZCHECK(hipStreamSynchronize(st));
    for (int i = 0; i < n; i++)
      for (int k = 0; k < opts->pv_len; k++) opts->pv[(size_t)i * opts->pv_len + k] = k < len ? pvh[(size_t)i * len + k] : 0u;
  }
  if (err & 1u) return zr::fail(ZETA_ENOMEM, "search: move stack overflow (more than %d moves on one path)", MSTACK);
  if (incomplete >= 0) return zr::fail(ZETA_ESTATE, "search: root %d did not complete", incomplete);
  return ZETA_OK;
}

extern "C" int zeta_search_abort(int on) {
  // may run on another host thread while zeta_search_batch waits: it touches
  // the abort word only
  int r = zr::require_init();
  if (r) return r;
  __atomic_store_n(zr::ctx().abort_host, on ? 1u : 0u, __ATOMIC_RELEASE);
  return ZETA_OK;
}

extern "C" int zeta_search_counters(uint64_t *out, int n) {
  int r = zr::require_up();
  if (r) return r;
  if (!out || n < 0) return zr::fail(ZETA_EINVAL, "zeta_search_counters: bad arguments");
  for (int i = 0; i < n && i < C_NCTR; i++) out[i] = g_ss.last_ctr[i];
  return ZETA_OK;
}

extern "C" int zeta_mlp_score(const zeta_pos *pos, int npos, const uint32_t *moves, const int32_t *offsets,
                              float *scores) {
  int r = zr::require_up();
  if (r) return r;
  const zm::Weights *w = mlp_weights();
  if (!w) return zr::fail(ZETA_ESTATE, "zeta_mlp_score: no network loaded");
  if (npos <= 0 || !pos || !moves || !offsets || !scores) return zr::fail(ZETA_EINVAL, "zeta_mlp_score: bad arguments");
  for (int i = 0; i < npos; i++)
    if (offsets[i + 1] < offsets[i] || offsets[i + 1] - offsets[i] > MSTACK)
      return zr::fail(ZETA_EINVAL, "zeta_mlp_score: bad offsets at %d", i);
  const int nm = offsets[npos];
  zr::DevBuf dp, dm, doff, dout;
  if ((r = zr::ensure(dp, (size_t)npos * sizeof(zeta_pos))) || (r = zr::ensure(dm, (size_t)nm * 4 + 4)) ||
      (r = zr::ensure(doff, (size_t)(npos + 1) * 4)) || (r = zr::ensure(dout, (size_t)nm * 4 + 4))) {
    zr::release(dp); zr::release(dm); zr::release(doff); zr::release(dout);
    return r;
  }
  hipStream_t st = zr::ctx().stream;
  SearchArgs sa;
  memset(&sa, 0, sizeof(sa));
  sa.w = *w;
  sa.use_mlp = 1;
  hipError_t e = hipMemcpyAsync(dp.p, pos, (size_t)npos * sizeof(zeta_pos), hipMemcpyHostToDevice, st);
  if (e == hipSuccess) e = hipMemcpyAsync(dm.p, moves, (size_t)nm * 4, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) e = hipMemcpyAsync(doff.p, offsets, (size_t)(npos + 1) * 4, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_mlp_score, dim3(npos), dim3(64), 0, st, sa, (const u64 *)dp.p, (const u32 *)dm.p,
                       (const int *)doff.p, (float *)dout.p);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpyAsync(scores, dout.p, (size_t)nm * 4, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  zr::release(dp); zr::release(dm); zr::release(doff); zr::release(dout);
  if (e != hipSuccess) return zr::hip_fail(e, "zeta_mlp_score", __FILE__, __LINE__);
  return ZETA_OK;
}

// ============================================================== serving
namespace {

struct ServeState {
  bool on = false;
  int nslots = 0, qcap = 0, workers = 1;
  void *pinned = nullptr;  // ServeHost + queue + ack + cancel + slots (hipHostMalloc, coherent)
  ServeHost *sh = nullptr;
  u64 *queue = nullptr, *ack = nullptr, *cancel = nullptr;
  ServeSlot *slots = nullptr;
  zr::DevBuf sv, sw, dreq, dcancel, nodes, depth_done, busy, ctr, err, rbound, dres, ctab;
  std::vector<u64> slot_ticket;  // ticket + 1 held by the slot, 0 = free
  std::vector<u64> slot_cost;
  std::vector<int> free_slots;
  u64 next_ticket = 0;
  u64 budget = 0, in_use = 0, tt_bytes = 0, worker_bytes = 0;
  bool use_mlp = false;
};
ServeState g_sv;

inline void sv_heartbeat() {
  __atomic_fetch_add(&g_sv.sh->heartbeat, 1ULL, __ATOMIC_RELEASE);
}

u64 sv_cost(int workers) {
  return (u64)workers * g_sv.worker_bytes + (g_sv.nslots ? g_sv.tt_bytes / (u64)g_sv.nslots : 0);
}

int sv_require() {
  int r = zr::require_init();
  if (r) return r;
  if (!g_sv.on) return zr::fail(ZETA_ESTATE, "serving not started (zeta_serve_start)");
  return ZETA_OK;
}

// the grid has exited on its own (watchdog or protocol error): report it
int sv_check_alive() {
  hipError_t q = hipStreamQuery(zr::ctx().stream);
  if (q == hipErrorNotReady) return ZETA_OK;
  if (q != hipSuccess) return zr::hip_fail(q, "serving grid", __FILE__, __LINE__);
  ServeDev d;
  memset(&d, 0, sizeof(d));
  (void)hipMemcpy(&d, g_sv.sv.p, sizeof(d), hipMemcpyDeviceToHost);
  return zr::fail(ZETA_ESTATE,
                  "serving grid has exited (reason %u: 2 watchdog, 3 host protocol error; now/ticket %llu, "
                  "arg %llu, xcc %#x, claimed %llu, mirror %llu); call zeta_serve_stop",
                  d.shut, (unsigned long long)d.exit_now, (unsigned long long)d.exit_arg, d.exit_xcc,
                  (unsigned long long)d.claimed, (unsigned long long)d.sub);
}

void sv_take(int s, zeta_result *res) {
  ServeSlot &sl = g_sv.slots[s];
  res->score = sl.score;
  res->bestmove = sl.bestmove;
  res->nodes = sl.nodes;
  res->depth = sl.depth_done;
  res->status = sl.status == SV_DONE ? ZETA_OK : (sl.status == SV_FAILED ? ZETA_ENOMEM : ZETA_ECANCELED);
  __atomic_store_n(&sl.state, 0u, __ATOMIC_RELEASE);
  g_sv.in_use -= g_sv.slot_cost[s];
  g_sv.slot_cost[s] = 0;
  g_sv.slot_ticket[s] = 0;
  g_sv.free_slots.push_back(s);
}

void sv_free_all() {
  zr::release(g_sv.sv); zr::release(g_sv.sw); zr::release(g_sv.dreq); zr::release(g_sv.dcancel);
  zr::release(g_sv.nodes); zr::release(g_sv.depth_done); zr::release(g_sv.busy); zr::release(g_sv.ctr);
  zr::release(g_sv.err); zr::release(g_sv.rbound); zr::release(g_sv.dres);
  zr::release(g_sv.ctab);
  if (g_sv.pinned) (void)hipHostFree(g_sv.pinned);
  g_sv.pinned = nullptr;
  g_sv.sh = nullptr;
  g_sv.slots = nullptr;
  g_sv.on = false;
  zr::ctx().serving = false;
}

}  // namespace

extern "C" int zeta_serve_start(const zeta_serve_opts *o) {
  int r = zr::require_up();
  if (r) return r;
  if (!o) return zr::fail(ZETA_EINVAL, "zeta_serve_start: null options");
  if (o->slots < 1 || o->slots > 4096) return zr::fail(ZETA_EINVAL, "zeta_serve_start: slots %d not in 1..4096", o->slots);
  if (o->workers < 1 || o->workers > 255)  // 8 bits of the slot word
    return zr::fail(ZETA_EINVAL, "zeta_serve_start: workers %d not in 1..255", o->workers);
  const int tt_log2 = o->tt_log2 < 0 ? zr::ctx().cfg.tt_log2 : o->tt_log2;
  if (tt_log2 > 34) return zr::fail(ZETA_EINVAL, "zeta_serve_start: tt_log2 %d too large", tt_log2);
  const zm::Weights *w = nullptr;
  if (o->use_mlp) w = mlp_weights();  // no network loaded: plain ordering for every request
  hipStream_t st = zr::ctx().stream;
  ZCHECK(hipStreamSynchronize(st));

  ServeState &S = g_sv;
  S = ServeState();
  S.nslots = o->slots;
  S.qcap = 2 * o->slots;
  S.workers = o->workers;
  S.budget = o->mem_budget;
  S.use_mlp = w != nullptr;
  hipFuncAttributes fa;
  ZCHECK(hipFuncGetAttributes(&fa, reinterpret_cast<const void *>(k_search<T_SHARED>)));
  S.worker_bytes = (u64)fa.sharedSizeBytes;
  const u64 tt_entries = tt_log2 > 0 ? (1ULL << tt_log2) : 0;
  S.tt_bytes = tt_entries * 16;

  const size_t hbytes = sizeof(ServeHost) + (size_t)(2 * S.qcap + S.nslots) * 8 + (size_t)S.nslots * sizeof(ServeSlot);
  hipError_t e = hipHostMalloc(&S.pinned, hbytes, hipHostMallocCoherent | hipHostMallocMapped);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    S.pinned = nullptr;
    return zr::fail(ZETA_ENOMEM, "zeta_serve_start: hipHostMalloc of %zu bytes failed (%s)", hbytes, hipGetErrorString(e));
  }
  memset(S.pinned, 0, hbytes);
  char *hp = (char *)S.pinned;
  S.sh = (ServeHost *)hp;
  S.queue = (u64 *)(hp + sizeof(ServeHost));
  S.ack = S.queue + S.qcap;
  S.cancel = S.ack + S.qcap;
  S.slots = (ServeSlot *)(S.cancel + S.nslots);
  void *dev_pinned = nullptr;
  e = hipHostGetDevicePointer(&dev_pinned, S.pinned, 0);
  if (e != hipSuccess) {
    sv_free_all();
    return zr::hip_fail(e, "hipHostGetDevicePointer", __FILE__, __LINE__);
  }
  const ptrdiff_t dd = (char *)dev_pinned - (char *)S.pinned;
  auto dp = [dd](void *p) { return (void *)((char *)p + dd); };

  const u32 busy_entries = 1u << 20;
  if ((r = zr::ensure(S.sv, sizeof(ServeDev))) || (r = zr::ensure(S.sw, (size_t)S.nslots * 8)) ||
      (r = zr::ensure(S.dreq, (size_t)S.nslots * sizeof(ServeReq))) || (r = zr::ensure(S.dcancel, (size_t)S.nslots * 8)) ||
      (r = zr::ensure(S.nodes, (size_t)S.nslots * 8)) || (r = zr::ensure(S.depth_done, (size_t)S.nslots * 4)) ||
      (r = zr::ensure(S.busy, (size_t)busy_entries * 4)) || (r = zr::ensure(S.ctr, C_NCTR * 8)) || (r = zr::ensure(S.err, 64)) ||
      (r = zr::ensure(S.rbound, (size_t)S.nslots * 8)) || (r = zr::ensure(S.dres, (size_t)S.nslots * 8))) {
    sv_free_all();
    return r;
  }
  if (tt_entries && ((r = zr::ensure(g_ss.tt, tt_entries * 16)))) {
    sv_free_all();
    return r;
  }
#define SV_CHECK(call)                                                          \
  do {                                                                          \
    hipError_t e_ = (call);                                                     \
    if (e_ != hipSuccess) {                                                     \
      int rc_ = zr::hip_fail(e_, #call, __FILE__, __LINE__);                    \
      sv_free_all();                                                            \
      return rc_;                                                               \
    }                                                                           \
  } while (0)
  if (tt_entries && g_ss.tt_entries != tt_entries) {
    hipLaunchKernelGGL(k_clear_u64, dim3(4096), dim3(256), 0, st, (u64 *)g_ss.tt.p, (size_t)(tt_entries * 2));
    SV_CHECK(hipGetLastError());
    g_ss.tt_entries = tt_entries;
  }
  SV_CHECK(hipMemsetAsync(S.sv.p, 0, sizeof(ServeDev), st));
  SV_CHECK(hipMemsetAsync(S.sw.p, 0, (size_t)S.nslots * 8, st));
  SV_CHECK(hipMemsetAsync(S.dcancel.p, 0, (size_t)S.nslots * 8, st));
  SV_CHECK(hipMemsetAsync(S.nodes.p, 0, (size_t)S.nslots * 8, st));
  SV_CHECK(hipMemsetAsync(S.depth_done.p, 0, (size_t)S.nslots * 4, st));
  SV_CHECK(hipMemsetAsync(S.busy.p, 0, (size_t)busy_entries * 4, st));
  SV_CHECK(hipMemsetAsync(S.ctr.p, 0, C_NCTR * 8, st));
  SV_CHECK(hipMemsetAsync(S.err.p, 0, 64, st));
  SV_CHECK(hipMemsetAsync(S.rbound.p, 0, (size_t)S.nslots * 8, st));
  SV_CHECK(hipStreamSynchronize(st));

  int rate_khz = 0;
  SV_CHECK(hipDeviceGetAttribute(&rate_khz, hipDeviceAttributeWallClockRate, zr::ctx().device));
  if (rate_khz <= 0) rate_khz = 100000;
  const int wd_ms = o->watchdog_ms > 0 ? o->watchdog_ms : 10000;

  int per_cu = 0;
  const auto kernel = tt_entries ? k_search<T_SHARED> : k_search<T_NONE>;
  SV_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 64, 0));
  if (per_cu < 1) per_cu = 1;
  const int cap = per_cu * zr::ctx().cu_count;
  int grid = o->grid > 0 && o->grid < cap ? o->grid : cap;
  if (grid < 2) grid = 2;  // one scheduler wavefront + at least one worker
  if ((r = zr::ensure(S.ctab, (size_t)grid * NCOUNTER * 2))) {
    sv_free_all();
    return r;
  }

  SearchArgs sa;
  memset(&sa, 0, sizeof(sa));
  sa.workers = S.workers;
  sa.split_depth = default_split(S.workers);
  sa.tt = (u64 *)g_ss.tt.p;
  sa.ttmask = tt_entries ? tt_entries - 1 : 0;
  sa.busy = (u32 *)S.busy.p;
  sa.busymask = busy_entries - 1;
  sa.ctab = (u16 *)S.ctab.p;
  if (tt_entries && (r = qt_clear((unsigned)grid, st, sa))) {
    sv_free_all();
    return r;
  }
  sa.nodes = (u64 *)S.nodes.p;
  sa.depth_done = (s32 *)S.depth_done.p;
  sa.err = (u32 *)S.err.p;
  sa.ctr = (u64 *)S.ctr.p;
  sa.habort = zr::ctx().abort_dev;
  sa.rbound = (u64 *)S.rbound.p;
  sa.dres = (u64 *)S.dres.p;
  sa.use_mlp = S.use_mlp ? 1 : 0;
  sa.mlp_min_depth = o->mlp_min_depth;
  if (w) sa.w = *w;
  sa.sh = (ServeHost *)dp(S.sh);
  sa.squeue = (const u64 *)dp(S.queue);
  sa.sack = (u64 *)dp(S.ack);
  sa.scancel = (const u64 *)dp(S.cancel);
  sa.slots = (ServeSlot *)dp(S.slots);
  sa.nslots = S.nslots;
  sa.qcap = S.qcap;
  sa.sv = (ServeDev *)S.sv.p;
  sa.sw = (u64 *)S.sw.p;
  sa.dreq = (ServeReq *)S.dreq.p;
  sa.dcancel = (u64 *)S.dcancel.p;
  sa.watchdog_ticks = (u64)wd_ms * (u64)rate_khz;
  S.free_slots.clear();
  for (int s = S.nslots - 1; s >= 0; s--) S.free_slots.push_back(s);
  S.slot_ticket.assign(S.nslots, 0);
  S.slot_cost.assign(S.nslots, 0);
  S.on = true;
  zr::ctx().serving = true;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(64), 0, st, sa);
  SV_CHECK(hipGetLastError());
#undef SV_CHECK
  return ZETA_OK;
}

extern "C" int zeta_serve_cost(int workers, uint64_t *bytes) {
  int r = sv_require();
  if (r) return r;
  if (!bytes) return zr::fail(ZETA_EINVAL, "zeta_serve_cost: null out pointer");
  if (workers <= 0) workers = g_sv.workers;
  if (workers > g_sv.workers) workers = g_sv.workers;
  *bytes = sv_cost(workers);
  return ZETA_OK;
}

extern "C" int zeta_serve_submit(const zeta_serve_request *req, uint64_t *ticket) {
  int r = sv_require();
  if (r) return r;
  ServeState &S = g_sv;
  sv_heartbeat();
  if (!req || !ticket) return zr::fail(ZETA_EINVAL, "zeta_serve_submit: null argument");
  if (req->depth < 1 || req->depth > MAXPLY - 1)
    return zr::fail(ZETA_EINVAL, "zeta_serve_submit: depth %d not in 1..%d", req->depth, MAXPLY - 1);
  if ((r = sv_check_alive())) return r;
  int workers = req->workers <= 0 ? S.workers : req->workers;
  if (workers > S.workers) workers = S.workers;
  const u64 cost = sv_cost(workers);
  if (S.budget && cost > S.budget)
    return zr::fail(ZETA_ENOMEM, "zeta_serve_submit: request needs %llu bytes, budget is %llu",
                    (unsigned long long)cost, (unsigned long long)S.budget);
  if (S.free_slots.empty()) return zr::fail(ZETA_EBUSY, "zeta_serve_submit: all %d slots in use", S.nslots);
  if (S.budget && S.in_use + cost > S.budget)
    return zr::fail(ZETA_EBUSY, "zeta_serve_submit: memory budget in use (%llu of %llu bytes)",
                    (unsigned long long)S.in_use, (unsigned long long)S.budget);
  const u64 t = S.next_ticket;
  const int qi = (int)(t % (u64)S.qcap);
  // the queue entry's previous ticket must have been claimed
  if (t >= (u64)S.qcap && __atomic_load_n(&S.ack[qi], __ATOMIC_ACQUIRE) != t - (u64)S.qcap + 1)
    return zr::fail(ZETA_EBUSY, "zeta_serve_submit: claim queue full");
  const int s = S.free_slots.back();
  S.free_slots.pop_back();
  ServeSlot &sl = S.slots[s];
  memcpy(sl.req.pos, &req->pos, sizeof(zeta_pos));
  sl.req.depth = req->depth;
  sl.req.flags = req->flags;
  sl.req.workers = workers;
  sl.req.pad = 0;
  __atomic_store_n(&sl.state, 0u, __ATOMIC_RELAXED);
  __atomic_store_n(&S.cancel[s], 0ULL, __ATOMIC_RELAXED);
  __atomic_store_n(&S.queue[qi], (u64)s, __ATOMIC_RELAXED);
  S.next_ticket = t + 1;
  __atomic_store_n(&S.sh->submitted, t + 1, __ATOMIC_RELEASE);
  S.slot_ticket[s] = t + 1;
  S.slot_cost[s] = cost;
  S.in_use += cost;
  *ticket = t;
  return ZETA_OK;
}

extern "C" int zeta_serve_poll(uint64_t ticket, zeta_result *res) {
  int r = sv_require();
  if (r) return r;
  sv_heartbeat();
  if (!res) return zr::fail(ZETA_EINVAL, "zeta_serve_poll: null result");
  for (int s = 0; s < g_sv.nslots; s++) {
    if (g_sv.slot_ticket[s] != ticket + 1) continue;
    if (!__atomic_load_n(&g_sv.slots[s].state, __ATOMIC_ACQUIRE)) {
      if ((r = sv_check_alive())) return r;
      return ZETA_PENDING;
    }
    sv_take(s, res);
    return ZETA_OK;
  }
  return zr::fail(ZETA_EINVAL, "zeta_serve_poll: ticket %llu is not in flight", (unsigned long long)ticket);
}

extern "C" int zeta_serve_reap(zeta_serve_done *out, int max, int *n) {
  int r = sv_require();
  if (r) return r;
  sv_heartbeat();
  if (!out || !n || max < 0) return zr::fail(ZETA_EINVAL, "zeta_serve_reap: bad arguments");
  int k = 0;
  for (int s = 0; s < g_sv.nslots && k < max; s++) {
    if (!g_sv.slot_ticket[s] || !__atomic_load_n(&g_sv.slots[s].state, __ATOMIC_ACQUIRE)) continue;
    out[k].ticket = g_sv.slot_ticket[s] - 1;
    sv_take(s, &out[k].res);
    k++;
  }
  *n = k;
  if (k == 0 && (r = sv_check_alive())) return r;
  return ZETA_OK;
}

extern "C" int zeta_serve_cancel(uint64_t ticket) {
  int r = sv_require();
  if (r) return r;
  sv_heartbeat();
  for (int s = 0; s < g_sv.nslots; s++) {
    if (g_sv.slot_ticket[s] != ticket + 1) continue;
    __atomic_store_n(&g_sv.cancel[s], ticket + 1, __ATOMIC_RELAXED);
    __atomic_fetch_add(&g_sv.sh->cancel_gen, 1u, __ATOMIC_RELEASE);
    return ZETA_OK;
  }
  return zr::fail(ZETA_EINVAL, "zeta_serve_cancel: ticket %llu is not in flight", (unsigned long long)ticket);
}

extern "C" int zeta_serve_stop(uint64_t *total_nodes) {
  int r = sv_require();
  if (r) return r;
  ServeState &S = g_sv;
  __atomic_store_n(&S.sh->shutdown, 1u, __ATOMIC_RELEASE);
  sv_heartbeat();
  hipError_t e = hipStreamSynchronize(zr::ctx().stream);
  u64 ctr[C_NCTR] = {0};
  u32 err = 0;
  if (e == hipSuccess) e = hipMemcpy(ctr, S.ctr.p, sizeof(ctr), hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(&err, S.err.p, 4, hipMemcpyDeviceToHost);
  if (e == hipSuccess) memcpy(g_ss.last_ctr, ctr, sizeof(ctr));
  if (total_nodes) *total_nodes = ctr[C_NODES];
  sv_free_all();
  if (e != hipSuccess) return zr::hip_fail(e, "zeta_serve_stop", __FILE__, __LINE__);
  return ZETA_OK;
}
