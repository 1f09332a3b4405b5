// chess.h -- device chess core for gfx950 (also compiles for the host so the
// same source can be unit-tested without a GPU; the library itself only runs
// it on the device).
//
// Positions use the reference's quad-bitboard (src/types.h:60-66):
//   b0 = black pieces, b1..b3 = piece-type bit planes (type = b1 + 2*b2 + 4*b3:
//   1 pawn, 2 knight, 3 king, 4 bishop, 5 rook, 6 queen), cr = "moved" flags
//   (castle rights live on a1/e1/h1/a8/e8/h8, the e.p. pawn is the one cleared
//   bit of ranks 4/5).
//
// The generator here is set-wise, not the reference's 64-lane square-wise one:
// one lane analyses a whole position with Kogge-Stone occluded fills (the
// opponent's slider rays give the attack map, and against the king's own rays
// the checkers, check rays, pins and the squares attacked through the king),
// then counts legal moves direction by direction (every target of a
// direction/offset has exactly one origin, so popcounts count moves).  It
// generates exactly the reference's legal move set, including its quirks:
// queen-only promotion (Q1, src/zetaperft.cl:1380-1384), the SMCRALL castle
// precondition (Q2, src/zetaperft.cl:1254), e.p. only from the moved flags
// with a full make/test legality check (src/zetaperft.cl:1222-1248), and
// 6-bit-masked shift counts (Q4).
#pragma once
#include <stdint.h>
#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define ZD __host__ __device__ __forceinline__
#define ZC_CONST __constant__
#else
// host-only build of this header (CPU unit tests of the device logic)
#define ZD static inline
#define ZC_CONST
#endif

namespace zc {

typedef uint64_t u64;
typedef uint32_t u32;
typedef int32_t s32;
typedef uint16_t u16;
typedef uint8_t u8;

constexpr u64 NOTA = 0xFEFEFEFEFEFEFEFEULL;
constexpr u64 NOTH = 0x7F7F7F7F7F7F7F7FULL;
constexpr u64 FULL = ~0ULL;
constexpr u64 RANKS45 = 0x000000FFFF000000ULL;
constexpr u64 RANK4 = 0x00000000FF000000ULL;
constexpr u64 RANK5 = 0x000000FF00000000ULL;
constexpr u64 RANK3 = 0x0000000000FF0000ULL;
constexpr u64 RANK6 = 0x0000FF0000000000ULL;
constexpr u64 SMCRALL = 0x8900000000000091ULL;     // src/types.h:114 (d8, not e8)
constexpr u64 SMCRWHITEQ = 0x0000000000000011ULL;  // src/types.h:119-124
constexpr u64 SMCRWHITEK = 0x0000000000000090ULL;
constexpr u64 SMCRBLACKQ = 0x1100000000000000ULL;
constexpr u64 SMCRBLACKK = 0x9000000000000000ULL;

enum { PNONE = 0, PAWN = 1, KNIGHT = 2, KING = 3, BISHOP = 4, ROOK = 5, QUEEN = 6 };

ZD int popc(u64 x) { return __builtin_popcountll(x); }
ZD int lsb(u64 x) { return __builtin_ctzll(x); }
ZD int msb(u64 x) { return 63 - __builtin_clzll(x); }
// Q4: shift counts are taken modulo 64, as OpenCL C does.
ZD u64 bit(int sq) { return u64(1) << (sq & 63); }
ZD u64 shlm(u64 x, int n) { return x << (n & 63); }
ZD u64 shrm(u64 x, int n) { return x >> (n & 63); }
ZD u64 sel(bool c, u64 x) { return x & (0ULL - (u64)c); }

// A 64-bit value the device compiler must keep whole in a register pair (an
// empty asm statement): it then shifts it with one v_lshlrev_b64 instead of
// splitting the shift into 32-bit halves for consumers that use halves.
ZD u64 whole(u64 x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm("" : "+v"(x));
#endif
  return x;
}
// (a & b) | c.  The compiler splits 64-bit AND and OR into 32-bit halves
// before it looks for the fused v_and_or_b32, so plain C costs four VALU
// instructions here; written out per half it is two.  Per-lane values only
// (the operands are forced into vector registers).
ZD u64 and_or(u64 a, u64 b, u64 c) {
#if defined(__HIP_DEVICE_COMPILE__)
  u32 lo, hi;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(lo) : "v"((u32)a), "v"((u32)b), "v"((u32)c));
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(hi) : "v"((u32)(a >> 32)), "v"((u32)(b >> 32)), "v"((u32)(c >> 32)));
  return whole(((u64)hi << 32) | lo);
#else
  return (a & b) | c;
#endif
}

// Any function of three boards in one v_bitop3_b32 a half: F is its truth
// table, written as the same expression of TA, TB and TC.
constexpr u32 TA = 0xF0, TB = 0xCC, TC = 0xAA;
template <u32 F>
ZD u64 bop3(u64 a, u64 b, u64 c) {
#if defined(__HIP_DEVICE_COMPILE__)
  const u32 lo = __builtin_amdgcn_bitop3_b32((u32)a, (u32)b, (u32)c, F & 0xFF);
  const u32 hi = __builtin_amdgcn_bitop3_b32((u32)(a >> 32), (u32)(b >> 32), (u32)(c >> 32), F & 0xFF);
  return whole(((u64)hi << 32) | lo);
#else
  u64 r = 0;
  for (u32 k = 0; k < 8; k++)
    if (F >> k & 1) r |= (k & 4 ? a : ~a) & (k & 2 ? b : ~b) & (k & 1 ? c : ~c);
  return r;
#endif
}

// ---- move code: the reference's 32-bit packing (src/types.h:67-74,126-141)
ZD u32 mv_from(u32 m) { return m & 63; }
ZD u32 mv_to(u32 m) { return (m >> 6) & 63; }
ZD u32 mv_cpt(u32 m) { return (m >> 12) & 63; }
ZD u32 mv_pfrom(u32 m) { return (m >> 18) & 15; }
ZD u32 mv_pto(u32 m) { return (m >> 22) & 15; }
ZD u32 mv_pcpt(u32 m) { return (m >> 26) & 15; }
ZD u32 mv_make(u32 f, u32 t, u32 c, u32 pf, u32 pt, u32 pc) {
  return f | (t << 6) | (c << 12) | (pf << 18) | (pt << 22) | (pc << 26);
}
constexpr u32 NULLMOVE = 0x41u;

struct Pos {
  u64 b0, b1, b2, b3, cr;
  u32 stm;
};

ZD u32 piece_at(const Pos &p, int sq) {
  return (u32)((shrm(p.b0, sq) & 1) | ((shrm(p.b1, sq) & 1) << 1) | ((shrm(p.b2, sq) & 1) << 2) |
               ((shrm(p.b3, sq) & 1) << 3));
}

// ---- one-step shifts and Kogge-Stone occluded fills for the 8 directions
// dir: 0 N, 1 S, 2 E, 3 W, 4 NE, 5 NW, 6 SE, 7 SW
ZD u64 step(u64 x, int d) {
  switch (d) {
    case 0: return x << 8;
    case 1: return x >> 8;
    case 2: return (x << 1) & NOTA;
    case 3: return (x >> 1) & NOTH;
    case 4: return (x << 9) & NOTA;
    case 5: return (x << 7) & NOTH;
    case 6: return (x >> 7) & NOTA;
    default: return (x >> 9) & NOTH;
  }
}
// one doubling step of an occluded fill: g | (e & (g shifted by SH)).  A
// shift by 32 or more moves one half into the other, which plain C already
// does without instructions; shorter shifts use the fused AND-OR.
template <int SH, bool UP>
ZD u64 fill_step(u64 g, u64 e) {
  const u64 t = UP ? g << SH : g >> SH;
  if (SH >= 32) return g | (e & t);
  return and_or(e, whole(t), g);
}
// occluded fill: generators plus every square reachable through `empty`
template <int D>
ZD u64 ks_fill(u64 g, u64 e) {
  constexpr int s = (D == 0 || D == 1) ? 8 : (D == 2 || D == 3) ? 1 : (D == 4 || D == 7) ? 9 : 7;
  constexpr bool up = (D == 0 || D == 2 || D == 4 || D == 5);
  constexpr u64 m = (D == 2 || D == 4 || D == 6) ? NOTA : (D == 3 || D == 5 || D == 7) ? NOTH : FULL;
  e &= m;
  if (up) {
    g = fill_step<s, true>(g, e);
    e &= e << s;
    g = fill_step<2 * s, true>(g, e);
    e &= e << (2 * s);
    g = fill_step<4 * s, true>(g, e);
  } else {
    g = fill_step<s, false>(g, e);
    e &= e >> s;
    g = fill_step<2 * s, false>(g, e);
    e &= e >> (2 * s);
    g = fill_step<4 * s, false>(g, e);
  }
  return g;
}
// the one-step shift of direction D without its edge-file mask (NOTA for
// E, NE, SE; NOTH for W, NW, SW; none for N, S): directions that share a
// mask can be masked once, after their union or on the target set
template <int D>
ZD u64 shift_raw(u64 x) {
  return D == 0 ? x << 8 : D == 1 ? x >> 8 : D == 2 ? x << 1 : D == 3 ? x >> 1
       : D == 4 ? x << 9 : D == 5 ? x << 7 : D == 6 ? x >> 7 : x >> 9;
}
// squares a slider set attacks in direction D (through empties, incl. first blocker)
template <int D>
ZD u64 slide(u64 g, u64 empty) {
  return step(ks_fill<D>(g, empty), D);
}
// the same without the edge-file mask
template <int D>
ZD u64 slide_raw(u64 g, u64 empty) {
  return shift_raw<D>(ks_fill<D>(g, empty));
}
template <int D>
struct Dir {
  static constexpr int value = D;
};
ZD u64 rook_att(u64 g, u64 empty) {
  return slide<0>(g, empty) | slide<1>(g, empty) | slide<2>(g, empty) | slide<3>(g, empty);
}
ZD u64 bishop_att(u64 g, u64 empty) {
  return slide<4>(g, empty) | slide<5>(g, empty) | slide<6>(g, empty) | slide<7>(g, empty);
}
ZD u64 knight_att(u64 n) {
  u64 l1 = (n >> 1) & NOTH, l2 = (n >> 2) & 0x3F3F3F3F3F3F3F3FULL;
  u64 r1 = (n << 1) & NOTA, r2 = (n << 2) & 0xFCFCFCFCFCFCFCFCULL;
  u64 h1 = l1 | r1, h2 = l2 | r2;
  return (h1 << 16) | (h1 >> 16) | (h2 << 8) | (h2 >> 8);
}
ZD u64 king_att(u64 k) {
  u64 a = k | ((k << 1) & NOTA) | ((k >> 1) & NOTH);
  a |= (a << 8) | (a >> 8);
  return a ^ k;
}
// the same for boards that differ by lane (a uniform one keeps to the scalar
// unit above): fused logic and whole shifts
ZD u64 knight_att_v(u64 n) {
  const u64 h1 = and_or(whole(n >> 1), NOTH, whole(n << 1) & NOTA);
  const u64 h2 = and_or(whole(n >> 2), 0x3F3F3F3F3F3F3F3FULL, whole(n << 2) & 0xFCFCFCFCFCFCFCFCULL);
  return bop3<(TA | TB | TC)>(whole(h1 << 16), whole(h1 >> 16), whole(h2 << 8)) | whole(h2 >> 8);
}
ZD u64 king_att_v(u64 k) {
  const u64 a = and_or(whole(k << 1), NOTA, and_or(whole(k >> 1), NOTH, k));
  return bop3<(TA | TB | TC)>(a, whole(a << 8), whole(a >> 8)) ^ k;
}
ZD u64 pawn_att(u64 p, u32 color) {
  return color ? (((p >> 7) & NOTA) | ((p >> 9) & NOTH)) : (((p << 9) & NOTA) | ((p << 7) & NOTH));
}
// full board lines through square k
ZD u64 rank_line(int k) { return 0xFFULL << (k & 56); }
ZD u64 file_line(int k) { return 0x0101010101010101ULL << (k & 7); }
ZD u64 diag_line(int k) {  // a1-h8 direction
  int d = (k & 7) - (k >> 3);
  return d >= 0 ? (0x8040201008040201ULL >> (8 * d)) : (0x8040201008040201ULL << (-8 * d));
}
ZD u64 anti_line(int k) {  // h1-a8 direction
  int s = (k & 7) + (k >> 3);
  return s <= 7 ? (0x0102040810204080ULL >> (8 * (7 - s))) : (0x0102040810204080ULL << (8 * (s - 7)));
}

// ---- single-square slider attacks (hyperbola quintessence with a full
// 64-bit bit reversal, which orders every line -- ranks included -- so the
// borrow of a subtraction runs along it in both directions).  One slider
// per lane: the search analyses one position with 64 lanes, lane = square.
ZD u64 rev64(u64 x) {
#if defined(__clang__)
  return __builtin_bitreverse64(x);
#else
  u64 r = x;
  r = ((r >> 1) & 0x5555555555555555ULL) | ((r & 0x5555555555555555ULL) << 1);
  r = ((r >> 2) & 0x3333333333333333ULL) | ((r & 0x3333333333333333ULL) << 2);
  r = ((r >> 4) & 0x0F0F0F0F0F0F0F0FULL) | ((r & 0x0F0F0F0F0F0F0F0FULL) << 4);
  return __builtin_bswap64(r);
#endif
}
// attacks of a slider on sq along the line `mask` (mask excludes sq)
ZD u64 line_att(int sq, u64 occ, u64 mask) {
  const u64 b = bit(sq);
  const u64 o = occ & mask;
  const u64 f = o - b;
  const u64 r = rev64(rev64(o) - rev64(b));
  return (f ^ r) & mask;
}
ZD u64 rook_sq(int sq, u64 occ) {
  const u64 b = bit(sq);
  return line_att(sq, occ, rank_line(sq) ^ b) | line_att(sq, occ, file_line(sq) ^ b);
}
ZD u64 bishop_sq(int sq, u64 occ) {
  const u64 b = bit(sq);
  return line_att(sq, occ, diag_line(sq) ^ b) | line_att(sq, occ, anti_line(sq) ^ b);
}

// ---- per-position legality context
struct Legal {
  u64 own, opp, occ, kbb;
  u64 pawns, knights, kings, rq, bq;
  u64 A;         // opponent attacks as if the own king were not on the board
  u64 checkers;  // opponent pieces giving check
  u64 cmask;     // allowed targets of non-king moves: ~0, block/capture set, or 0 (double check)
  u64 pinR, pinF, pinD, pinA;  // own pieces pinned on the king's rank, file, diagonal, anti-diagonal
  int ksq;
  u32 stm;
};

// ---- rank rays by a carry: added to the empty squares, a piece shifted one
// square on runs through them and sets the first that is not empty (a blocker
// or the edge file, which `e` leaves out).  Pieces are not empty, so a ray ends
// at the next one and all rays of a set come from one addition.  West runs on
// the reversed board.  s: occupied squares; e: empty & NOTH.
ZD u64 ray_east(u64 s, u64 e) { return whole(((s & NOTH) << 1) + e) ^ e; }

// Legality context of a board with several own kings (no game reaches it):
// the check rays are all the kings' rays in a checked direction, and so are
// the squares behind them.
ZD void many_kings(Legal &L, u64 e, u64 &A, u64 &chkray) {
  const u64 orq = L.opp & L.rq, obq = L.opp & L.bq;
  auto line = [&](u64 S, u64 Ku, u64 Kv) {
    const bool hu = (Ku & S) != 0, hv = (Kv & S) != 0;
    chkray |= sel(hu, Ku) | sel(hv, Kv);
    A |= sel(hu, Kv) | sel(hv, Ku);
  };
  chkray = 0;
  line(orq, slide<0>(L.kbb, e), slide<1>(L.kbb, e));
  line(orq, slide<2>(L.kbb, e), slide<3>(L.kbb, e));
  line(obq, slide<4>(L.kbb, e), slide<7>(L.kbb, e));
  line(obq, slide<5>(L.kbb, e), slide<6>(L.kbb, e));
}

// Per line through the king, from occluded fills in its two directions U and
// V: R = the rays of the opponent's sliders that move along the line, K = the
// king's own rays (each up to and including the first blocker).  Where a ray
// of the king meets the opposite ray of a slider, an own piece is pinned and
// an empty square lies between the king and a checker.  Both lie strictly
// inside the line, never on an edge file of a rank or diagonal: the diagonals'
// rays go unmasked (their last step may wrap onto an edge file) and the wraps
// fall to the mask of what meets them, or to one mask a union.
// A holds, of the squares behind the king on a checked line, the next one: the
// king steps no further, and a king in check does not castle.
// Bound: VALU issue where a lane takes a position (perft).  The three fills of
// a direction share the doubled empty sets; three-operand logic and the rank
// carries, here, in apply_v and in count_legal, took a perft leaf from 990 to
// 865 lane-instructions (128.9 M leaves: 3.41 to 2.9 ms).
ZD void analyse(const Pos &p, Legal &L) {
  const u64 occ = bop3<(TA | TB | TC)>(p.b1, p.b2, p.b3);
  const u64 black = 0 - (u64)(p.stm & 1u);
  L.stm = p.stm;
  L.occ = occ;
  L.own = bop3<(TA ^ (TB & ~TC))>(p.b0, occ, black);
  L.opp = bop3<(TA ^ (TB & TC))>(p.b0, occ, black);
  L.pawns = bop3<(TA & ~TB & ~TC)>(p.b1, p.b2, p.b3);
  L.knights = bop3<(~TA & TB & ~TC)>(p.b1, p.b2, p.b3);
  L.kings = bop3<(TA & TB & ~TC)>(p.b1, p.b2, p.b3);
  L.rq = bop3<((TA ^ TB) & TC)>(p.b1, p.b2, p.b3);  // rook 101, queen 110
  L.bq = p.b3 & ~p.b1;                              // bishop 100, queen 110
  const u64 kbb = L.own & L.kings;
  L.kbb = kbb;
  L.ksq = kbb ? lsb(kbb) : 0;
  const u64 orq = L.opp & L.rq, obq = L.opp & L.bq;
  const u64 opawns = L.opp & L.pawns, oknights = L.opp & L.knights;
  const u64 e = ~occ;
  constexpr u64 INNER = NOTA & NOTH;
  // a slider's ray that reaches the (one) king goes one square on
  const bool many = (kbb & (kbb - 1)) != 0;
  const u64 kx = sel(!many, kbb), kxA = kx & NOTA, kxH = kx & NOTH;
  auto ray = [&](auto D, u64 k, u64 g) {
    constexpr int d = decltype(D)::value;
    return shift_raw<d>(and_or(shift_raw<d>(g), k, g));
  };
  // files
  const u64 rn = ray(Dir<0>(), kx, ks_fill<0>(orq, e)), rs = ray(Dir<1>(), kx, ks_fill<1>(orq, e));
  const u64 kn = slide_raw<0>(kbb, e), ks = slide_raw<1>(kbb, e);
  const u64 xf = and_or(kn, rs, ks & rn);
  // ranks
  const u64 ee = e & NOTH, er = rev64(e) & NOTH;
  u64 re = ray_east(orq, ee), rw = ray_east(rev64(orq), er);
  const u64 ke = ray_east(kbb, ee), kw = rev64(ray_east(rev64(kbb), er));
  rw = rev64(rw);
  re |= whole((re & kxH) << 1);
  rw |= whole((rw & kxA) >> 1);
  const u64 xr = and_or(ke, rw, kw & re);
  // diagonals
  const u64 rne = ray(Dir<4>(), kxA, ks_fill<4>(obq, e)), rsw = ray(Dir<7>(), kxH, ks_fill<7>(obq, e));
  const u64 kne = slide_raw<4>(kbb, e), ksw = slide_raw<7>(kbb, e);
  const u64 xd = and_or(kne, rsw, ksw & rne);
  const u64 rnw = ray(Dir<5>(), kxH, ks_fill<5>(obq, e)), rse = ray(Dir<6>(), kxA, ks_fill<6>(obq, e));
  const u64 knw = slide_raw<5>(kbb, e), kse = slide_raw<6>(kbb, e);
  const u64 xa = and_or(knw, rse, kse & rnw);
  L.pinF = xf & L.own;
  L.pinR = xr & L.own;
  const u64 owni = L.own & INNER;
  L.pinD = xd & owni;
  L.pinA = xa & owni;
  u64 chkray = bop3<((TA | TB) & TC)>(xf, xr, e) | bop3<((TA | TB) & TC)>(xd, xa, e & INNER);
  // the opponent's pawns one rank on, and the king's
  const int up = p.stm & 1u ? 0 : 8, down = 8 - up;
  const u64 pf = (opawns << down) >> up, kf = (kbb << up) >> down;
  const u64 kpawn = and_or(whole(kf << 1), NOTA, whole(kf >> 1) & NOTH);
  u64 A = bop3<(TA | TB | TC)>(rn, rs, re) | rw;
  A = bop3<(TA | TB | TC)>(A, knight_att_v(oknights), king_att_v(L.opp & L.kings));
  A = and_or(bop3<(TA | TB | TC)>(rne, rse, whole(pf << 1)), NOTA, A);
  A = and_or(bop3<(TA | TB | TC)>(rnw, rsw, whole(pf >> 1)), NOTH, A);
  u64 ch = bop3<((TA | TB) & TC)>(bop3<(TA | TB | TC)>(kn, ks, ke), kw, orq);
  ch |= bop3<((TA | TB) & TC)>(kne, kse, obq & NOTA);
  ch |= bop3<((TA | TB) & TC)>(knw, ksw, obq & NOTH);
  ch = and_or(kpawn, opawns, ch);
  ch = and_or(knight_att_v(kbb), oknights, ch);
  if (many) many_kings(L, e, A, chkray);
  L.A = A;
  L.checkers = ch;
  const int n = popc(ch);
  L.cmask = n == 0 ? FULL : (n == 1 ? (ch | chkray) : 0ULL);
}

// is the side to move's king attacked after the e.p. capture from->to taking
// sqep?  A knight or pawn checks it after the capture exactly when it checks
// it before (unless it is the captured pawn); sliders by the line attacks of
// the king's square on the new occupancy (two single-square slider lookups,
// not eight occluded fills); a king never checks
ZD bool ep_legal(const Legal &L, int from, int to, int sqep) {
  if (!L.kbb) return true;
  // nearly always nothing can open: no check, the capturing pawn not pinned,
  // and the captured one neither on the king's rank nor on its diagonals (its
  // file stays closed by the capturing pawn).  Boards that no game reaches may
  // break the last: their e.p. flag can name an empty square or any piece, so
  // an opponent's pawn has to stand there, and the capture's target be empty.
  const int dr = (sqep >> 3) - (L.ksq >> 3), df = (sqep & 7) - (L.ksq & 7);
  const u64 pinned = L.pinR | L.pinF | L.pinD | L.pinA;
  const bool plain = ((L.opp & L.pawns) >> sqep & 1) && !((L.occ >> to) & 1) && L.cmask == FULL;
  if (plain && !((pinned >> from) & 1) && dr != 0 && dr != df && dr != -df) return true;
  const u64 occ2 = (L.occ ^ bit(from) ^ bit(sqep)) | bit(to);
  const u64 opp2 = L.opp & ~bit(sqep);
  const u64 att = (rook_sq(L.ksq, occ2) & opp2 & L.rq) | (bishop_sq(L.ksq, occ2) & opp2 & L.bq) |
                  (L.checkers & ~(L.rq | L.bq) & ~bit(sqep));
  return att == 0;
}

// e.p.: the pawn that just double-pushed is the lowest cleared bit of ranks 4/5
// (src/zetaperft.cl:1224-1230); returns the own pawns that may capture it.
ZD u64 ep_candidates(const Pos &p, const Legal &L, int &sqep) {
  const u64 w = ~p.cr & RANKS45;
  sqep = w ? lsb(w) : 0;
  u64 c = L.own & L.pawns & (p.stm ? RANK4 : RANK5);
  return c & (bit(sqep + 1) | bit(sqep - 1));
}

// castling targets of the king (src/zetaperft.cl:1249-1297).  The rule
// looks at the eight squares k-4 .. k+3 around the king (the reference's
// bit() takes them modulo 64), so the rook, occupancy and attack sets are
// rotated right by k-4: bit i is square k-4+i for every king square, with no
// branch on where the king stands.  A set bit of `bad` is a failed condition:
// queen side bits 0-4 (rook on k-4, k-3..k-1 empty, k-2..k not attacked),
// king side bits 4-7 (k+1, k+2 empty, k..k+2 not attacked, rook on k+3).
ZD u64 rotr64(u64 x, int n) { return shrm(x, n) | shlm(x, 64 - n); }
ZD u64 castle_targets(const Pos &p, const Legal &L) {
  const u64 cr = p.cr;
  if (!(cr & SMCRALL)) return 0;
  const bool okq = p.stm ? ((~cr & SMCRBLACKQ) == SMCRBLACKQ) : ((~cr & SMCRWHITEQ) == SMCRWHITEQ);
  const bool okk = p.stm ? ((~cr & SMCRBLACKK) == SMCRBLACKK) : ((~cr & SMCRWHITEK) == SMCRWHITEK);
  if (!okq && !okk) return 0;
  const u64 ownrooks = L.own & L.rq & ~p.b2;  // rook = 101 (queen has b2 set)
  const int q = (L.ksq - 4) & 63;
  const u32 rk = (u32)rotr64(ownrooks, q), oc = (u32)rotr64(L.occ, q), at = (u32)rotr64(L.A, q);
  const u32 bad = (~rk & 0x81u) | (oc & 0x6Eu) | (at & 0x7Cu);
  const u32 t = ((okq && !(bad & 0x1Fu)) ? 0x04u : 0u) | ((okk && !(bad & 0xF0u)) ? 0x40u : 0u);
  return rotr64((u64)t, (64 - q) & 63);  // back: bit 2 -> k-2, bit 6 -> k+2
}

// Number of legal moves (qs: captures and e.p. only, as the kernels' quiescence).
ZD int count_legal(const Pos &p, const Legal &L, bool qs) {
  const u64 own = L.own, occ = L.occ;
  const u64 T = (qs ? L.opp : ~own) & L.cmask;
  // the target set with each edge-file mask applied once (a shifted set
  // masked and then intersected with T is the shifted set intersected with
  // the masked T)
  const u64 TnA = T & NOTA, TnH = T & NOTH;
  const u64 pinned = bop3<(TA | TB | TC)>(L.pinR, L.pinF, L.pinD) | L.pinA;
  int cnt = popc(bop3<(TA & TB & ~TC)>(king_att_v(L.kbb), qs ? L.opp : ~own, L.A));
  const u64 kn = bop3<(TA & TB & ~TC)>(own, L.knights, pinned);
  const u64 TAB = T & 0xFCFCFCFCFCFCFCFCULL, TGH = T & 0x3F3F3F3F3F3F3F3FULL;
  cnt += popc(whole(kn << 17) & TnA) + popc(whole(kn << 15) & TnH) + popc(whole(kn << 10) & TAB) + popc(whole(kn << 6) & TGH);
  cnt += popc(whole(kn >> 6) & TAB) + popc(whole(kn >> 10) & TGH) + popc(whole(kn >> 15) & TnA) + popc(whole(kn >> 17) & TnH);
  const u64 e = ~occ;
  const u64 orq = own & L.rq, obq = own & L.bq;
  const u64 sf = bop3<(TA & (~TB | TC))>(orq, pinned, L.pinF), sr = bop3<(TA & (~TB | TC))>(orq, pinned, L.pinR);
  const u64 sd = bop3<(TA & (~TB | TC))>(obq, pinned, L.pinD), sa = bop3<(TA & (~TB | TC))>(obq, pinned, L.pinA);
  cnt += popc(slide_raw<0>(sf, e) & T);
  cnt += popc(slide_raw<1>(sf, e) & T);
  const u64 ee = e & NOTH, er = rev64(e) & NOTH;
  cnt += popc(ray_east(sr, ee) & T);
  cnt += popc(ray_east(rev64(sr), er) & rev64(T));
  cnt += popc(slide_raw<4>(sd, e) & TnA);
  cnt += popc(slide_raw<7>(sd, e) & TnH);
  cnt += popc(slide_raw<5>(sa, e) & TnH);
  cnt += popc(slide_raw<6>(sa, e) & TnA);
  // pawns: one rank on, then one file east or west.  East captures run along
  // the a1-h8 diagonals for white and the others for black.
  const u64 P = own & L.pawns;
  const int up = p.stm & 1u ? 0 : 8, down = 8 - up;
  const u64 pinE = p.stm & 1u ? L.pinA : L.pinD, pinW = p.stm & 1u ? L.pinD : L.pinA;
  const u64 capE = (bop3<(TA & (~TB | TC))>(P, pinned, pinE) << up) >> down;
  const u64 capW = (bop3<(TA & (~TB | TC))>(P, pinned, pinW) << up) >> down;
  const u64 tgt = L.opp & L.cmask;
  cnt += popc(bop3<(TA & TB & TC)>(whole(capE << 1), tgt, NOTA)) + popc(bop3<(TA & TB & TC)>(whole(capW >> 1), tgt, NOTH));
  if (!qs) {
    const u64 pp = bop3<(TA & (~TB | TC))>(P, pinned, L.pinF);
    const u64 s1 = whole((pp << up) >> down) & e;
    const u64 s2 = whole(((s1 & (p.stm & 1u ? RANK6 : RANK3)) << up) >> down);
    cnt += popc(s1 & L.cmask) + popc(bop3<(TA & TB & TC)>(s2, e, L.cmask));
    cnt += popc(castle_targets(p, L));
  }
  int sqep;
  u64 cand = ep_candidates(p, L, sqep);
  while (cand) {
    const int f = lsb(cand);
    cand &= cand - 1;
    const int to = (p.stm ? sqep - 8 : sqep + 8) & 63;
    cnt += ep_legal(L, f, to, sqep) ? 1 : 0;
  }
  return cnt;
}

// Legal targets of the own piece on `sq` (used to enumerate moves in
// canonical order: origin ascending, then target ascending).
ZD u64 piece_targets(const Pos &p, const Legal &L, int sq, bool qs) {
  const u64 b = bit(sq);
  const u64 own = L.own, occ = L.occ;
  const u32 type = (u32)((shrm(p.b1, sq) & 1) | ((shrm(p.b2, sq) & 1) << 1) | ((shrm(p.b3, sq) & 1) << 2));
  if (type == KING) {
    u64 t = king_att(b) & (qs ? L.opp : ~own) & ~L.A;
    if (!qs) t |= castle_targets(p, L);
    return t;
  }
  u64 pinmask = FULL;
  if (L.pinR & b) pinmask = rank_line(L.ksq);
  if (L.pinF & b) pinmask = file_line(L.ksq);
  if (L.pinD & b) pinmask = diag_line(L.ksq);
  if (L.pinA & b) pinmask = anti_line(L.ksq);
  const u64 T = (qs ? L.opp : ~own) & L.cmask & pinmask;
  const u64 e = ~occ;
  u64 t = 0;
  switch (type) {
    case PAWN: {
      t = pawn_att(b, p.stm) & L.opp & L.cmask & pinmask;
      if (!qs) {
        u64 s1 = (p.stm ? (b >> 8) : (b << 8)) & e;
        u64 s2 = (p.stm ? ((s1 & RANK6) >> 8) : ((s1 & RANK3) << 8)) & e;
        t |= (s1 | s2) & L.cmask & pinmask;
      }
      int sqep;
      const u64 cand = ep_candidates(p, L, sqep);
      if (cand & b) {
        const int to = (p.stm ? sqep - 8 : sqep + 8) & 63;
        if (ep_legal(L, sq, to, sqep)) t |= bit(to);
      }
      return t;
    }
    case KNIGHT: return knight_att(b) & T;
    case BISHOP: return bishop_att(b, e) & T;
    case ROOK: return rook_att(b, e) & T;
    case QUEEN: return (rook_att(b, e) | bishop_att(b, e)) & T;
    default: return 0;
  }
}

// Index of the k-th set bit (k from 0) of x, which has more than k set bits:
// a binary search on popcounts, with no loop over the bits.
ZD int nth_bit(u64 x, int k) {
  u32 w = (u32)x;
  int base = 0;
  const int c32 = popc((u64)w);
  if (k >= c32) {
    k -= c32;
    w = (u32)(x >> 32);
    base = 32;
  }
#pragma unroll
  for (int s = 16; s >= 1; s >>= 1) {
    const int c = popc((u64)(w & ((1u << s) - 1u)));
    if (k >= c) {
      k -= c;
      w >>= s;
      base += s;
    }
  }
  return base;
}

// ---- node analysis with one lane per square (the search's wave-per-node
// layout).  The uniform part is cheap (king-square attackers); everything
// set-wise is replaced by per-square questions answered by all 64 lanes at
// once and combined with a ballot:
//   attacked(sq): is sq attacked by the opponent with the own king removed?
//   the legal targets of the own piece on sq (pin line, check mask, king
//   safety from the attacked-square mask).
struct Node0 {
  u64 own, opp, occ, kbb;
  u64 pawns, knights, kings, rq, bq;
  u64 checkers, cmask;
  int ksq;
  u32 stm;
};

ZD void node_basics(const Pos &p, Node0 &B) {
  const u64 occ = p.b1 | p.b2 | p.b3;
  const u64 white = p.b0 ^ occ;
  B.stm = p.stm;
  B.occ = occ;
  B.own = p.stm ? p.b0 : white;
  B.opp = p.stm ? white : p.b0;
  B.pawns = p.b1 & ~p.b2 & ~p.b3;
  B.knights = ~p.b1 & p.b2 & ~p.b3;
  B.kings = p.b1 & p.b2 & ~p.b3;
  B.rq = p.b3 & (p.b1 ^ p.b2);
  B.bq = p.b3 & ~p.b1;
  B.kbb = B.own & B.kings;
  B.ksq = B.kbb ? lsb(B.kbb) : 0;
  const u64 orq = B.opp & B.rq, obq = B.opp & B.bq;
  u64 ch = (rook_sq(B.ksq, occ) & orq) | (bishop_sq(B.ksq, occ) & obq);
  ch |= knight_att(B.kbb) & B.opp & B.knights;
  ch |= pawn_att(B.kbb, p.stm) & B.opp & B.pawns;
  ch = sel(B.kbb != 0, ch);
  B.checkers = ch;
  const int n = popc(ch);
  u64 cm = 0;
  if (n == 0) cm = FULL;
  if (n == 1) {
    // the checker, plus the squares between it and the king for a slider
    const int c = lsb(ch);
    const u64 r = rook_sq(B.ksq, occ) & rook_sq(c, occ);
    const u64 d = bishop_sq(B.ksq, occ) & bishop_sq(c, occ);
    const bool rl = (rank_line(B.ksq) & ch) || (file_line(B.ksq) & ch);
    const bool slider = ((B.rq | B.bq) & ch) != 0;
    cm = ch | sel(slider, rl ? r : d);
  }
  B.cmask = cm;
}

// The lines through a square (the square itself taken out), its bit and the
// reversed bit: what the slider attacks of one square need besides the
// occupancy.  The search holds the set of its lane's square in registers.
struct SqLines {
  u64 b, rb, rank, file, diag, anti;
};
ZD SqLines sq_lines(int sq) {
  const u64 b = bit(sq);
  return SqLines{b, rev64(b), rank_line(sq) ^ b, file_line(sq) ^ b, diag_line(sq) ^ b, anti_line(sq) ^ b};
}
ZD u64 line_att(const SqLines &q, u64 occ, u64 mask) {  // mask: one of q's lines
  const u64 o = occ & mask;
  return ((o - q.b) ^ rev64(rev64(o) - q.rb)) & mask;
}
ZD u64 rook_sq(const SqLines &q, u64 occ) { return line_att(q, occ, q.rank) | line_att(q, occ, q.file); }
ZD u64 bishop_sq(const SqLines &q, u64 occ) { return line_att(q, occ, q.diag) | line_att(q, occ, q.anti); }

// what move generation needs of the lane's square, in registers for good
struct LaneSq {
  SqLines q;
  u64 knight, king, wpawn, bpawn;
};
ZD LaneSq lane_sq(int sq) {
  const u64 b = bit(sq);
  return LaneSq{sq_lines(sq), knight_att(b), king_att(b), pawn_att(b, 0), pawn_att(b, 1)};
}

// Does the side `by` attack the king of the other side?  q = the lines of its
// square, knight and pawn = the squares from which those attack it (king false:
// there is none).
// One position per lane, the same king square in every lane: the checkers of
// node_basics without the check mask.
ZD bool king_attacked(const Pos &p, const SqLines &q, bool king, u64 knight, u64 pawn, u32 by) {
  const u64 occ = p.b1 | p.b2 | p.b3;
  const u64 them = by ? p.b0 : (p.b0 ^ occ);
  const u64 rq = p.b3 & (p.b1 ^ p.b2), bq = p.b3 & ~p.b1;
  u64 a = (rook_sq(q, occ) & rq) | (bishop_sq(q, occ) & bq);
  a |= knight & ~p.b1 & p.b2 & ~p.b3;
  a |= pawn & p.b1 & ~p.b2 & ~p.b3;
  return king && (a & them);
}
ZD bool king_attacked(const Pos &p, const SqLines &q, u64 kb, u32 by) {
  return king_attacked(p, q, kb != 0, knight_att(kb), pawn_att(kb, by ^ 1u), by);
}

// is sq attacked by the opponent, the own king taken off the board?
ZD bool attacked_nk(const Node0 &B, int sq) {
  const u64 b = bit(sq);
  const u64 occ = B.occ ^ B.kbb;
  u64 a = (rook_sq(sq, occ) & B.rq) | (bishop_sq(sq, occ) & B.bq);
  a |= knight_att(b) & B.knights;
  a |= king_att(b) & B.kings;
  a |= pawn_att(b, B.stm) & B.pawns;
  return (a & B.opp) != 0;
}

// the line through the king and sq when the own piece on sq is pinned, else ~0
ZD u64 pin_line(const Node0 &B, int sq) {
  const int k = B.ksq;
  const u64 b = bit(sq);
  u64 m = 0, sl = 0;
  if ((sq >> 3) == (k >> 3)) { m = rank_line(k); sl = B.rq; }
  else if ((sq & 7) == (k & 7)) { m = file_line(k); sl = B.rq; }
  else if (diag_line(k) & b) { m = diag_line(k); sl = B.bq; }
  else if (anti_line(k) & b) { m = anti_line(k); sl = B.bq; }
  if (!m || !B.kbb) return FULL;
  const u64 me = m ^ bit(k);
  const u64 seen = line_att(k, B.occ, me);
  if (!(seen & b)) return FULL;  // not the first piece seen from the king
  const u64 behind = line_att(k, B.occ ^ b, me) & ~seen;
  return (behind & B.opp & sl) ? m : FULL;
}

ZD bool ep_legal0(const Node0 &B, int from, int to, int sqep) {
  const u64 occ2 = (B.occ ^ bit(from) ^ bit(sqep)) | bit(to);
  const u64 opp2 = B.opp & ~bit(sqep);
  u64 att = (rook_sq(B.ksq, occ2) & opp2 & B.rq) | (bishop_sq(B.ksq, occ2) & opp2 & B.bq);
  att |= knight_att(B.kbb) & opp2 & B.knights;
  att |= pawn_att(B.kbb, B.stm) & opp2 & B.pawns;
  att |= king_att(B.kbb) & opp2 & B.kings;
  return att == 0;
}

// castling targets of the king on k, its own rooks and the attack map A given
// (castle_targets with each square's condition written out: one king a wave)
ZD u64 castle_squares(const Pos &p, u64 ownrooks, u64 occ, u64 A, int k) {
  const bool okq = p.stm ? ((~p.cr & SMCRBLACKQ) == SMCRBLACKQ) : ((~p.cr & SMCRWHITEQ) == SMCRWHITEQ);
  const bool okk = p.stm ? ((~p.cr & SMCRBLACKK) == SMCRBLACKK) : ((~p.cr & SMCRWHITEK) == SMCRWHITEK);
  const u64 q = sel(okq && (ownrooks & bit(k - 4)) && !(occ & (bit(k - 1) | bit(k - 2) | bit(k - 3))) &&
                        !(A & (bit(k) | bit(k - 1) | bit(k - 2))),
                    bit(k - 2));
  return q | sel(okk && (ownrooks & bit(k + 3)) && !(occ & (bit(k + 1) | bit(k + 2))) &&
                     !(A & (bit(k) | bit(k + 1) | bit(k + 2))),
                 bit(k + 2));
}

// legal targets of the own piece on sq; A = squares attacked with the own
// king transparent (only read for the king)
ZD u64 lane_targets(const Pos &p, const Node0 &B, u64 A, int sq, bool qs) {
  const u64 b = bit(sq);
  const u32 type = (u32)((shrm(p.b1, sq) & 1) | ((shrm(p.b2, sq) & 1) << 1) | ((shrm(p.b3, sq) & 1) << 2));
  const u64 own = B.own, occ = B.occ;
  if (type == KING) {
    u64 t = king_att(b) & (qs ? B.opp : ~own) & ~A;
    if (!qs && (p.cr & SMCRALL)) t |= castle_squares(p, own & B.rq & ~p.b2, occ, A, sq);
    return t;
  }
  const u64 pm = pin_line(B, sq);
  const u64 T = (qs ? B.opp : ~own) & B.cmask & pm;
  u64 t;
  if (type == PAWN) {
    t = pawn_att(b, p.stm) & B.opp & B.cmask & pm;
    if (!qs) {
      const u64 e = ~occ;
      const u64 s1 = (p.stm ? (b >> 8) : (b << 8)) & e;
      const u64 s2 = (p.stm ? ((s1 & RANK6) >> 8) : ((s1 & RANK3) << 8)) & e;
      t |= (s1 | s2) & B.cmask & pm;
    }
    const u64 w = ~p.cr & RANKS45;
    const int sqep = w ? lsb(w) : 0;
    const bool cand = (p.stm ? (RANK4 & b) : (RANK5 & b)) && ((bit(sqep + 1) | bit(sqep - 1)) & b) && w;
    if (cand) {
      const int to = (p.stm ? sqep - 8 : sqep + 8) & 63;
      if (ep_legal0(B, sq, to, sqep)) t |= bit(to);
    }
    return t;
  }
  // pieces: branch-free over the type (no divergence across lanes)
  const bool rk = type == ROOK || type == QUEEN, bs = type == BISHOP || type == QUEEN;
  t = sel(rk, rook_sq(sq, occ)) | sel(bs, bishop_sq(sq, occ)) | sel(type == KNIGHT, knight_att(b));
  return t & T;
}

// Do lane_targets, square by square, find the moves that for_each_legal does?
// The set-wise form takes boards no game reaches in its own way: several kings,
// and an e.p. flag that is not alone on a pawn that can have stepped two past an
// empty square, or next to which the kings stand side by side.
ZD bool lanes_serve(const Pos &p, const Node0 &B) {
  const u64 okb = B.opp & B.kings, w = ~p.cr & RANKS45;
  bool serve = (popc(B.kbb) == 1) & ((okb & (okb - 1)) == 0);
  if (w) {
    const u64 stepped = B.opp & B.pawns & (p.stm ? RANK4 : RANK5);
    serve &= !(w & (w - 1)) & ((w & stepped) != 0) & !((p.stm ? w >> 8 : w << 8) & B.occ) & !(king_att(B.kbb) & okb);
  }
  return serve;
}

// ---- lane = square of one position whose king is not in check: what a slider
// on the lane's square would see
struct LaneRays {
  u64 rank, file, diag, anti;
};
ZD LaneRays lane_rays(const LaneSq &me, u64 occ) {
  return LaneRays{line_att(me.q, occ, me.q.rank), line_att(me.q, occ, me.q.file), line_att(me.q, occ, me.q.diag),
                  line_att(me.q, occ, me.q.anti)};
}
// is the lane's square attacked by the side that is not to move (the own king
// a blocker)?
ZD bool lane_attacked(const Pos &p, const LaneSq &me, const LaneRays &y) {
  const u64 opp = p.stm ? p.b0 ^ (p.b1 | p.b2 | p.b3) : p.b0;
  const u64 rq = p.b3 & (p.b1 ^ p.b2), bq = p.b3 & ~p.b1;
  u64 a = ((y.rank | y.file) & rq) | ((y.diag | y.anti) & bq);
  a |= (me.knight & ~p.b1 & p.b2 & ~p.b3) | (me.king & p.b1 & p.b2 & ~p.b3);
  a |= (p.stm ? me.bpawn : me.wpawn) & p.b1 & ~p.b2 & ~p.b3;
  return (a & opp) != 0;
}
// legal targets of the own piece on the lane's square; A: the squares that
// lane_attacked is true for.  A piece that sees its king and, the other way on
// the line, a slider of the line is pinned to it.
ZD u64 lane_free_targets(const Pos &p, const LaneSq &me, const LaneRays &y, u64 A, int sq) {
  const u64 b = me.q.b, occ = p.b1 | p.b2 | p.b3;
  const u64 opp = p.stm ? p.b0 ^ occ : p.b0, own = occ ^ opp;
  if (!(own & b)) return 0;
  const u64 rq = p.b3 & (p.b1 ^ p.b2), bq = p.b3 & ~p.b1;
  const u64 king = own & p.b1 & p.b2 & ~p.b3;
  const u32 type = (u32)((p.b1 & b ? 1 : 0) | (p.b2 & b ? 2 : 0) | (p.b3 & b ? 4 : 0));
  u64 pm = FULL;
  if ((y.rank & king) && (y.rank & opp & rq)) pm = me.q.rank;
  if ((y.file & king) && (y.file & opp & rq)) pm = me.q.file;
  if ((y.diag & king) && (y.diag & opp & bq)) pm = me.q.diag;
  if ((y.anti & king) && (y.anti & opp & bq)) pm = me.q.anti;
  u64 t = sel(type == ROOK || type == QUEEN, y.rank | y.file) | sel(type == BISHOP || type == QUEEN, y.diag | y.anti) |
          sel(type == KNIGHT, me.knight);
  t &= ~own;
  if (type == KING) {
    t = me.king & ~own & ~A;
    if (p.cr & SMCRALL) t |= castle_squares(p, own & rq & ~p.b2, occ, A, sq);
  }
  if (type == PAWN) {
    const u64 s1 = (p.stm ? b >> 8 : b << 8) & ~occ;
    const u64 s2 = (p.stm ? (s1 & RANK6) >> 8 : (s1 & RANK3) << 8) & ~occ;
    t = ((p.stm ? me.bpawn : me.wpawn) & opp) | s1 | s2;
  }
  t &= pm;
  const u64 w = ~p.cr & RANKS45;
  if (type == PAWN && w) {
    const int sqep = lsb(w);
    if ((p.stm ? RANK4 : RANK5) & (bit(sqep + 1) | bit(sqep - 1)) & b) {
      Node0 B;
      node_basics(p, B);
      const int to = (p.stm ? sqep - 8 : sqep + 8) & 63;
      if (ep_legal0(B, sq, to, sqep)) t |= bit(to);
    }
  }
  return t;
}

// z modulo n, n from 1 to 256, sixteen bits at a time: a remainder and the next
// bits are below 2^24, where a float quotient is off by one at most
ZD u32 mod_small(u64 z, u32 n) {
  const float inv = 1.0f / (float)n;
  u32 r = 0;
  for (int s = 48; s >= 0; s -= 16) {
    const u32 t = (r << 16) | (u32)((z >> s) & 0xFFFF);
    const int d = (int)(t - (u32)((float)t * inv) * n);
    r = (u32)(d < 0 ? d + (int)n : d >= (int)n ? d - (int)n : d);
  }
  return r;
}

// Pack from->to with the reference movepicker rules (src/zetaperft.cl:1363-1386):
// e.p. capture square, captured piece, queen-only promotion (Q1).
ZD u32 make_code(const Pos &p, int from, int to) {
  const u32 pfrom = piece_at(p, from);
  int sqcpt = to;
  u32 pcpt = piece_at(p, to);
  const bool pawn = ((pfrom >> 1) & 7) == PAWN;
  if (pawn && p.stm && from - to != 8 && from - to != 16 && pcpt == PNONE) sqcpt = to + 8;
  if (pawn && !p.stm && to - from != 8 && to - from != 16 && pcpt == PNONE) sqcpt = to - 8;
  pcpt = piece_at(p, sqcpt);
  const int rrank = p.stm ? ((to >> 3) ^ 7) : (to >> 3);
  const u32 pto = (pawn && rrank == 7) ? ((QUEEN << 1) | (pfrom & 1)) : pfrom;
  return mv_make((u32)from, (u32)to, (u32)sqcpt, pfrom, pto, pcpt);
}

ZD void put_piece(Pos &c, int sq, u32 pc) {
  c.b0 |= shlm((u64)(pc & 1), sq);
  c.b1 |= shlm((u64)((pc >> 1) & 1), sq);
  c.b2 |= shlm((u64)((pc >> 2) & 1), sq);
  c.b3 |= shlm((u64)((pc >> 3) & 1), sq);
}

// Apply a move: pieces as the kernels' domove (src/zetaperft.cl:413-484), then
// the moved flags.  rook_flag selects the perft/host variant that also flags
// the castle rook's origin (src/zetaperft.cl:1452-1455) or the alpha-beta
// variant that does not (src/zeta.cl:2333-2345, quirk Q6).
ZD Pos apply(const Pos &p, u32 m, bool rook_flag) {
  Pos c = p;
  const int f = (int)mv_from(m), t = (int)mv_to(m), x = (int)mv_cpt(m);
  const u32 pf = mv_pfrom(m);
  const bool king = ((pf >> 1) & 7) == KING;
  const bool qside = king && f - t == 2, kside = king && t - f == 2;
  u64 keep = ~bit(f) & ~bit(x) & ~bit(t);
  if (qside) keep &= ~bit(f - 4);
  if (kside) keep &= ~bit(f + 3);
  c.b0 &= keep;
  c.b1 &= keep;
  c.b2 &= keep;
  c.b3 &= keep;
  put_piece(c, t, mv_pto(m));
  const u32 rook = (ROOK << 1) | (pf & 1);
  if (qside) put_piece(c, t + 1, rook);
  if (kside) put_piece(c, t - 1, rook);
  u64 cr = p.cr | bit(f) | bit(t) | bit(x);
  if (rook_flag && qside) cr |= bit(f - 4);
  if (rook_flag && kside) cr |= bit(f + 3);
  const u32 col = pf & 1;
  const int rf = col ? ((f >> 3) ^ 7) : (f >> 3), rt = col ? ((t >> 3) ^ 7) : (t >> 3);
  const bool dbl = ((pf >> 1) & 7) == PAWN && rt - rf == 2;
  cr |= RANKS45;
  if (dbl) cr &= ~bit(t);
  c.cr = cr;
  c.stm = p.stm ^ 1u;
  return c;
}

// apply() where every lane has a position of its own (perft): fused logic, the
// castling rook behind a branch that few wavefronts take
ZD Pos apply_v(const Pos &p, u32 m) {
  Pos c;
  const int f = (int)mv_from(m), t = (int)mv_to(m);
  const u64 tb = bit(t);
  const u64 gone = bop3<(TA | TB | TC)>(bit(f), bit((int)mv_cpt(m)), tb);
  const u32 pf = mv_pfrom(m), pt = mv_pto(m);
  c.b0 = and_or(0 - (u64)(pt & 1), tb, p.b0 & ~gone);
  c.b1 = and_or(0 - (u64)((pt >> 1) & 1), tb, p.b1 & ~gone);
  c.b2 = and_or(0 - (u64)((pt >> 2) & 1), tb, p.b2 & ~gone);
  c.b3 = and_or(0 - (u64)((pt >> 3) & 1), tb, p.b3 & ~gone);
  u64 cr = bop3<(TA | TB | TC)>(p.cr, gone, RANKS45);
  const u32 type = (pf >> 1) & 7;
  if (type == KING && (f - t == 2 || t - f == 2)) {
    // the rook goes to the king's other side
    const int r = f - t == 2 ? f - 4 : f + 3, s = f - t == 2 ? t + 1 : t - 1;
    const u64 keep = ~bit(r);
    c.b0 &= keep;
    c.b1 &= keep;
    c.b2 &= keep;
    c.b3 &= keep;
    put_piece(c, s, (ROOK << 1) | (pf & 1));
    cr |= bit(r);
  }
  const u32 col = pf & 1;
  const int rf = col ? ((f >> 3) ^ 7) : (f >> 3), rt = col ? ((t >> 3) ^ 7) : (t >> 3);
  if (type == PAWN && rt - rf == 2) cr &= ~tb;
  c.cr = cr;
  c.stm = p.stm ^ 1u;
  return c;
}

// apply_v() of a position that is only counted: the e.p. flag is dropped when
// no pawn stands to use it (positions that differ only there have the same
// legal moves and descendants).
ZD Pos apply_count(const Pos &p, u32 m) {
  Pos c = apply_v(p, m);
  const u64 w = ~c.cr & RANKS45;
  if (w) {
    const u64 occ = c.b1 | c.b2 | c.b3;
    const u64 mine = c.stm ? c.b0 : c.b0 ^ occ;
    const int sq = lsb(w);
    const u64 cand = mine & c.b1 & ~c.b2 & ~c.b3 & (c.stm ? RANK4 : RANK5) & (bit(sq + 1) | bit(sq - 1));
    if (!cand) c.cr |= RANKS45;
  }
  return c;
}

// apply() of a capture (e.p. and promotions included, no castling): the
// planes and the side to move; the moved flags are the parent's.
ZD Pos apply_capture(const Pos &p, u32 m) {
  Pos c = p;
  const u64 t = bit((int)mv_to(m));
  const u64 keep = ~(bit((int)mv_from(m)) | bit((int)mv_cpt(m)) | t);
  const u32 pt = mv_pto(m);
  c.b0 = (p.b0 & keep) | sel(pt & 1, t);
  c.b1 = (p.b1 & keep) | sel((pt >> 1) & 1, t);
  c.b2 = (p.b2 & keep) | sel((pt >> 2) & 1, t);
  c.b3 = (p.b3 & keep) | sel((pt >> 3) & 1, t);
  c.stm = p.stm ^ 1u;
  return c;
}

// ---- Zobrist hashing, rotate-left scheme: key(piece) rotated left by the
// square (src/bitboard.c:461-508, src/zeta.cl:2297-2359).  12 piece keys
// (colour*6 + type-1), 4 castle keys, 1 e.p. key rotated by the file; the
// values are the reference's (src/zobrist.h:28-35) so hashes crossing the
// boundary stay comparable.
static ZC_CONST const u64 ZOBRIST[18] = {
    0x9D39247E33776D41ULL, 0x2AF7398005AAA5C7ULL, 0x44DB015024623547ULL, 0x9C15F73E62A76AE2ULL,
    0x75834465489C0C89ULL, 0x3290AC3A203001BFULL, 0x0FBBAD1F61042279ULL, 0xE83A908FF2FB60CAULL,
    0x0D7E765D58755C10ULL, 0x1A083822CEAFE02DULL, 0x9605D5F0E25EC3B0ULL, 0xD021FF5CD13A2ED5ULL,
    0x40BDF15D4A672E32ULL, 0x011355146FD56395ULL, 0x5DB4832046F3D9E5ULL, 0x239F8B2D7FF719CCULL,
    0x05D1A1AE85B49AA1ULL, 0x679F848F6E8FC971ULL};

ZD u64 rotl(u64 z, int s) { return shlm(z, s) | shrm(z, 64 - s); }
ZD u64 piece_key(u32 pc, int sq) { return rotl(ZOBRIST[(pc & 1) * 6 + ((pc >> 1) & 7) - 1], sq); }
ZD u64 hash_pieces(const Pos &p) {
  u64 h = 0;
  u64 occ = p.b1 | p.b2 | p.b3;
  while (occ) {
    int sq = lsb(occ);
    occ &= occ - 1;
    h ^= piece_key(piece_at(p, sq), sq);
  }
  return h;
}
ZD u64 hash_castle(u64 cr) {
  u64 h = 0;
  h ^= sel((~cr & SMCRWHITEQ) != 0, ZOBRIST[12]);
  h ^= sel((~cr & SMCRWHITEK) != 0, ZOBRIST[13]);
  h ^= sel((~cr & SMCRBLACKQ) != 0, ZOBRIST[14]);
  h ^= sel((~cr & SMCRBLACKK) != 0, ZOBRIST[15]);
  return h;
}
// host computehash (src/bitboard.c:461-508)
ZD u64 hash_full(const Pos &p) {
  u64 h = hash_pieces(p) ^ hash_castle(p.cr);
  u64 w = ~p.cr & RANKS45;
  int sqep = w ? lsb(w) : 0;
  if (sqep) h ^= rotl(ZOBRIST[16], sqep & 7);
  if (p.stm) h ^= 1ULL;
  return h;
}

// k-th legal move in canonical order (origin ascending, then target ascending)
ZD u32 nth_legal(const Pos &p, const Legal &L, int k) {
  u64 pcs = L.own;
  while (pcs) {
    const int sq = lsb(pcs);
    pcs &= pcs - 1;
    u64 t = piece_targets(p, L, sq, false);
    const int c = popc(t);
    if (k < c) {
      while (k-- > 0) t &= t - 1;
      return make_code(p, sq, lsb(t));
    }
    k -= c;
  }
  return 0;
}

// Origin of a slider move to `to` in direction d: the path from the origin is
// empty, so it is the nearest occupied square back along the direction.
ZD int slider_from(int d, int to, u64 occ) {
  const u64 b = bit(to), below = b - 1, above = ~(below | b);
  switch (d) {
    case 0: return msb(occ & file_line(to) & below);  // moved north
    case 1: return lsb(occ & file_line(to) & above);  // south
    case 2: return msb(occ & rank_line(to) & below);  // east
    case 3: return lsb(occ & rank_line(to) & above);  // west
    case 4: return msb(occ & diag_line(to) & below);  // north-east
    case 5: return msb(occ & anti_line(to) & below);  // north-west
    case 6: return lsb(occ & anti_line(to) & above);  // south-east
    default: return lsb(occ & diag_line(to) & above);  // south-west
  }
}

// Every legal move (the set count_legal(qs = false) counts, so exactly that
// many calls of emit(code)), grouped by kind instead of by origin: each
// kind's target set is built for all its pieces at once, as in count_legal,
// and each target gives back its origin -- a fixed offset for king, knight and
// pawn moves, slider_from() for sliders.  Codes equal make_code(p, from, to);
// the order is not the canonical one (nth_legal).
template <class Emit>
ZD void for_each_legal(const Pos &p, const Legal &L, Emit &&emit) {
  const u32 stm = p.stm;
  const u64 own = L.own, occ = L.occ, e = ~occ;
  const u64 T = ~own & L.cmask;
  const u64 TA = T & NOTA, TH = T & NOTH;
  const u64 pinned = L.pinR | L.pinF | L.pinD | L.pinA;
  // one kind with a fixed origin offset (from = to - delta) and moving piece pf
  auto fixed = [&](u64 t, int delta, u32 pf) {
    while (t) {
      const int to = lsb(t);
      t &= t - 1;
      emit(mv_make((u32)(to - delta), (u32)to, (u32)to, pf, pf, piece_at(p, to)));
    }
  };
  // king (castling included: the rook's move is implied by the code)
  {
    const u32 pk = (KING << 1) | stm;
    u64 t = (king_att(L.kbb) & ~own & ~L.A) | castle_targets(p, L);
    while (t) {
      const int to = lsb(t);
      t &= t - 1;
      emit(mv_make((u32)L.ksq, (u32)to, (u32)to, pk, pk, piece_at(p, to)));
    }
  }
  // knights, one offset at a time
  {
    const u64 kn = own & L.knights & ~pinned;
    const u64 TAB = T & 0xFCFCFCFCFCFCFCFCULL, TGH = T & 0x3F3F3F3F3F3F3F3FULL;
    const u32 pn = (KNIGHT << 1) | stm;
    fixed((kn << 17) & TA, 17, pn);
    fixed((kn << 15) & TH, 15, pn);
    fixed((kn << 10) & TAB, 10, pn);
    fixed((kn << 6) & TGH, 6, pn);
    fixed((kn >> 6) & TAB, -6, pn);
    fixed((kn >> 10) & TGH, -10, pn);
    fixed((kn >> 15) & TA, -15, pn);
    fixed((kn >> 17) & TH, -17, pn);
  }
  // sliders, one direction at a time
  {
    const u64 orq = own & L.rq, obq = own & L.bq;
    auto dir = [&](int d, u64 t) {
      while (t) {
        const int to = lsb(t);
        t &= t - 1;
        const int from = slider_from(d, to, occ);
        const u32 pf = piece_at(p, from);
        emit(mv_make((u32)from, (u32)to, (u32)to, pf, pf, piece_at(p, to)));
      }
    };
    dir(0, slide_raw<0>(orq & (~pinned | L.pinF), e) & T);
    dir(1, slide_raw<1>(orq & (~pinned | L.pinF), e) & T);
    dir(2, slide_raw<2>(orq & (~pinned | L.pinR), e) & TA);
    dir(3, slide_raw<3>(orq & (~pinned | L.pinR), e) & TH);
    dir(4, slide_raw<4>(obq & (~pinned | L.pinD), e) & TA);
    dir(7, slide_raw<7>(obq & (~pinned | L.pinD), e) & TH);
    dir(5, slide_raw<5>(obq & (~pinned | L.pinA), e) & TH);
    dir(6, slide_raw<6>(obq & (~pinned | L.pinA), e) & TA);
  }
  // pawns: pushes, double pushes, captures (queen-only promotion, Q1), e.p.
  {
    const u64 P = own & L.pawns;
    const u32 pp_ = (PAWN << 1) | stm, pq = (QUEEN << 1) | stm;
    const int last = stm ? 0 : 7;
    auto pawn = [&](u64 t, int delta) {
      while (t) {
        const int to = lsb(t);
        t &= t - 1;
        const u32 pt = (to >> 3) == last ? pq : pp_;
        emit(mv_make((u32)(to - delta), (u32)to, (u32)to, pp_, pt, piece_at(p, to)));
      }
    };
    const u64 pp = P & (~pinned | L.pinF);
    const u64 capD = P & (~pinned | L.pinD), capA = P & (~pinned | L.pinA);
    const u64 tgt = L.opp & L.cmask;
    if (stm) {
      const u64 s1 = (pp >> 8) & e, s2 = ((s1 & RANK6) >> 8) & e;
      pawn(s1 & L.cmask, -8);
      pawn(s2 & L.cmask, -16);
      pawn(((capD >> 9) & NOTH) & tgt, -9);
      pawn(((capA >> 7) & NOTA) & tgt, -7);
    } else {
      const u64 s1 = (pp << 8) & e, s2 = ((s1 & RANK3) << 8) & e;
      pawn(s1 & L.cmask, 8);
      pawn(s2 & L.cmask, 16);
      pawn(((capD << 9) & NOTA) & tgt, 9);
      pawn(((capA << 7) & NOTH) & tgt, 7);
    }
    int sqep;
    u64 cand = ep_candidates(p, L, sqep);
    while (cand) {
      const int f = lsb(cand);
      cand &= cand - 1;
      const int to = (stm ? sqep - 8 : sqep + 8) & 63;
      if (ep_legal(L, f, to, sqep)) emit(make_code(p, f, to));
    }
  }
}

// How many moves for_each_legal emits: a board with several kings of one side
// can have a king step and a castling with one target, which is one move there.
ZD int count_emitted(const Pos &p, const Legal &L) {
  return count_legal(p, L, false) - popc(king_att(L.kbb) & ~L.own & ~L.A & castle_targets(p, L));
}

// host domove half-move clock rule (src/bitboard.c:604-689): +1, reset by
// pawn moves, captures and castling
ZD u32 next_hmc(u32 hmc, u32 m) {
  const u32 pf = mv_pfrom(m);
  const int f = (int)mv_from(m), t = (int)mv_to(m);
  const u32 ty = (pf >> 1) & 7;
  if (ty == PAWN || ((mv_pcpt(m) >> 1) & 7) != PNONE) return 0;
  if (ty == KING && (f - t == 2 || t - f == 2)) return 0;
  return hmc + 1;
}

}  // namespace zc
