// evaltab.h -- the reference evaluation's constants (src/zeta.cl:272-359):
// material {P 100, N 400, K 0, B 400, R 600, Q 1200}, square-control bonus and
// the piece-square tables (Michniewski's "simplified evaluation"), all in
// black view (white indexes sq^56).  They are data the root scores depend on,
// so they must be the reference's values exactly.
#pragma once
#include <stdint.h>

namespace zc {

static constexpr int32_t EVAL_VALUE[7] = {0, 100, 400, 0, 400, 600, 1200};

static constexpr int32_t EVAL_CONTROL[64] = {
    0, 0, 5, 5, 5, 5, 0, 0,   5, 0, 5, 5, 5, 5, 0, 5,   0, 0, 10, 5, 5, 10, 0, 0, 0, 5, 5, 10, 10, 5, 5, 0,
    0, 5, 5, 10, 10, 5, 5, 0, 0, 0, 10, 5, 5, 10, 0, 0, 0, 0, 5, 5, 5, 5, 0, 0,   0, 0, 5, 5, 5, 5, 0, 0};

static constexpr int32_t EVAL_PST[7 * 64] = {
    // none
    0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0,
    0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0,
    // pawn
    0, 0, 0, 0, 0, 0, 0, 0, 50, 50, 50, 50, 50, 50, 50, 50, 30, 30, 30, 30, 30, 30, 30, 30,
    5, 5, 5, 10, 10, 5, 5, 5, 3, 3, 3, 8, 8, 3, 3, 3, 2, 2, 2, 2, 2, 2, 2, 2,
    0, 0, 0, -5, -5, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0,
    // knight
    -50, -40, -30, -30, -30, -30, -40, -50, -40, -20, 0, 0, 0, 0, -20, -40,
    -30, 0, 10, 15, 15, 10, 0, -30, -30, 5, 15, 20, 20, 15, 5, -30,
    -30, 0, 15, 20, 20, 15, 0, -30, -30, 5, 10, 15, 15, 10, 5, -30,
    -40, -20, 0, 5, 5, 0, -20, -40, -50, -40, -30, -30, -30, -30, -40, -50,
    // king
    -1, -1, -1, -1, -1, -1, -1, -1, -1, 0, 0, 0, 0, 0, 0, -1, -1, 0, 0, 0, 0, 0, 0, -1,
    -1, 0, 0, 0, 0, 0, 0, -1, -1, 0, 0, 0, 0, 0, 0, -1, -1, 0, 0, 0, 0, 0, 0, -1,
    -1, 0, 0, 0, 0, 0, 0, -1, -1, -1, -1, -1, -1, -1, -1, -1,
    // bishop
    -20, -10, -10, -10, -10, -10, -10, -20, -10, 0, 0, 0, 0, 0, 0, -10,
    -10, 0, 5, 10, 10, 5, 0, -10, -10, 5, 5, 10, 10, 5, 5, -10,
    -10, 0, 10, 10, 10, 10, 0, -10, -10, 10, 10, 10, 10, 10, 10, -10,
    -10, 5, 0, 0, 0, 0, 5, -10, -20, -10, -10, -10, -10, -10, -10, -20,
    // rook
    0, 0, 0, 0, 0, 0, 0, 0, 5, 10, 10, 10, 10, 10, 10, 5, -5, 0, 0, 0, 0, 0, 0, -5,
    -5, 0, 0, 0, 0, 0, 0, -5, -5, 0, 0, 0, 0, 0, 0, -5, -5, 0, 0, 0, 0, 0, 0, -5,
    -5, 0, 0, 0, 0, 0, 0, -5, 0, 0, 0, 5, 5, 0, 0, 0,
    // queen
    -20, -10, -10, -5, -5, -10, -10, -20, -10, 0, 0, 0, 0, 0, 0, -10,
    -10, 0, 5, 5, 5, 5, 0, -10, -5, 0, 5, 5, 5, 5, 0, -5,
    -5, 0, 5, 5, 5, 5, 0, -5, -10, 0, 5, 5, 5, 5, 0, -10,
    -10, 0, 0, 0, 0, 0, 0, -10, -20, -10, -10, -5, -5, -10, -10, -20};

// One square's share of the x64 evaluation (src/zeta.cl:1482-1521), white
// positive: +10 per piece, material, piece-square, square control, and the
// pawn terms (blocked -15, chain +10 per diagonal-behind own pawn, -30 per
// own pawn behind on the file).  The bishop pair (src/zeta.cl:1522-1531) is
// added once per position by the caller.
// 10 + material + piece-square + square control of a piece type on a square
// (black view), folded into one table so a square costs one lookup
struct EvalSq {
  int32_t v[7 * 64];
};
constexpr EvalSq make_eval_sq() {
  EvalSq t{};
  for (int ty = 1; ty < 7; ty++)
    for (int sq = 0; sq < 64; sq++) t.v[ty * 64 + sq] = 10 + EVAL_VALUE[ty] + EVAL_PST[ty * 64 + sq] + EVAL_CONTROL[sq];
  return t;
}
static ZC_CONST const EvalSq EVAL_SQ = make_eval_sq();

ZD int32_t eval_square(const Pos &p, int sq) {
  const u32 pc = piece_at(p, sq);
  const int type = (int)((pc >> 1) & 7);
  if (type == PNONE) return 0;
  const int color = (int)(pc & 1);
  const int sqf = color ? sq : (sq ^ 56);
  int32_t s = EVAL_SQ.v[type * 64 + sqf];
  if (type == PAWN) {
    const u64 occ = p.b1 | p.b2 | p.b3;
    const u64 pawns = p.b1 & ~p.b2 & ~p.b3;
    const u64 me = color ? p.b0 : (p.b0 ^ occ);
    const u64 opp = color ? (p.b0 ^ occ) : p.b0;
    const u64 mp = pawns & me;
    const u64 file = 0x0101010101010101ULL << (sq & 7);
    if (color == 0) {
      if ((sq >> 3) < 7 && (opp & bit(sq + 8))) s -= 15;
      if ((sq & 7) < 7 && (mp & bit(sq - 7))) s += 10;
      if ((sq & 7) > 0 && (mp & bit(sq - 9))) s += 10;
      // own pawns behind on the file, ranks 2 .. rank-1 (the reference's loop
      // runs t = sq-8, sq-16, .. while t > 7)
      if (sq >= 8) s -= 30 * popc(mp & file & (bit(sq) - 1) & ~0xFFULL);
      else
        for (uint8_t t = (uint8_t)(sq - 8); t > 7; t = (uint8_t)(t - 8))
          if (mp & bit(t)) s -= 30;
    } else {
      if ((sq >> 3) > 0 && (opp & bit(sq - 8))) s -= 15;
      if ((sq & 7) > 0 && (mp & bit(sq + 7))) s += 10;
      if ((sq & 7) < 7 && (mp & bit(sq + 9))) s += 10;
      // ranks rank+1 .. 7 (t = sq+8, sq+16, .. while t < 56)
      s -= 30 * popc(mp & file & ~((bit(sq) << 1) - 1) & ~(0xFFULL << 56));
    }
  }
  return color ? -s : s;
}

ZD int32_t eval_bishop_pair(const Pos &p) {
  const u64 occ = p.b1 | p.b2 | p.b3;
  const u64 bishops = ~p.b1 & ~p.b2 & p.b3;
  return (popc((p.b0 ^ occ) & bishops) == 2 ? 25 : 0) - (popc(p.b0 & bishops) == 2 ? 25 : 0);
}

// The pawn terms of eval_square summed over the board, white minus black, set
// by set: blocked by an opponent's piece in front (-15), defended by an own
// pawn (+10 for each side), own pawns behind on the file (-30 each, so -30 for
// every pair on a file).  Equal to the per-square terms when no pawn stands on
// the first or the last rank (the reference's ranges there wrap).
ZD int32_t pawn_terms(u64 pawns, u64 white, u64 black) {
  const u64 w = pawns & white, b = pawns & black;
  const int block = popc((w << 8) & black) - popc((b >> 8) & white);
  const int chain = popc(w & (w << 7) & NOTH) + popc(w & (w << 9) & NOTA) - popc(b & (b >> 7) & NOTA) -
                    popc(b & (b >> 9) & NOTH);
  int pairs = 0;
#pragma unroll
  for (int k = 8; k <= 40; k += 8) pairs += popc(w & (w << k)) - popc(b & (b << k));
  return 10 * chain - 15 * block - 30 * pairs;
}

// material + piece-square + square control of a coloured piece, white
// positive, from a table in EVAL_SQ's layout (the search keeps one in LDS)
template <class T>
ZD int32_t eval_piece(const T *tab, u32 pc, int sq) {
  const int v = (int)tab[((pc >> 1) & 7) * 64 + ((pc & 1) ? sq : (sq ^ 56))];
  return (pc & 1) ? -v : v;
}

// How a move of `stm` changes the sum of eval_piece over the board (white
// positive); CASTLING: the move may be one, the rook's step is included.
template <bool CASTLING, class T>
ZD int32_t eval_move_delta(const T *tab, u32 stm, u32 m) {
  const u32 flip = stm ? 0 : 56;
  const u32 f = mv_from(m), t = mv_to(m), pf = (mv_pfrom(m) >> 1) & 7;
  // (no captured piece: the table's first 64 entries are 0)
  int32_t d = (int32_t)tab[((mv_pto(m) >> 1) & 7) * 64 + (t ^ flip)] - (int32_t)tab[pf * 64 + (f ^ flip)] +
              (int32_t)tab[((mv_pcpt(m) >> 1) & 7) * 64 + (mv_cpt(m) ^ flip ^ 56)];
  if (CASTLING && pf == KING && (f - t == 2 || t - f == 2)) {
    const u32 to = f - t == 2 ? t + 1 : t - 1, from = f - t == 2 ? f - 4 : f + 3;
    d += (int32_t)tab[ROOK * 64 + ((to & 63) ^ flip)] - (int32_t)tab[ROOK * 64 + ((from & 63) ^ flip)];
  }
  return stm ? -d : d;
}

// EVAL_VALUE / 100 of the seven piece types as nibbles of a constant: no load
ZD int32_t piece_value(u32 type) { return (int32_t)((0xC640410u >> (4 * type)) & 15u) * 100; }

// Move-ordering score of the reference picker (src/zeta.cl:2059-2071):
// captures MVV-LVA (16*V[captured] - V[mover]), quiet moves by the change of
// material + piece-square + control value.
// tab: a table in EVAL_SQ's layout, whose constant part cancels.
template <class T>
ZD int32_t order_score(const T *tab, u32 stm, u32 m) {
  const u32 tf = (mv_pto(m) >> 1) & 7, ff = (mv_pfrom(m) >> 1) & 7, cf = (mv_pcpt(m) >> 1) & 7;
  if (cf != PNONE) return piece_value(cf) * 16 - piece_value(tf);
  const u32 flip = stm ? 0 : 56;
  return (int32_t)tab[tf * 64 + (mv_to(m) ^ flip)] - (int32_t)tab[ff * 64 + (mv_from(m) ^ flip)];
}

}  // namespace zc
