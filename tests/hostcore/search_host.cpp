// Host build of the per-lane pieces of the search's refuted-move test
// (zeta_amd/csrc/chess.h, evaltab.h) for CPU unit tests.  Test-only.
#include "../../zeta_amd/csrc/chess.h"
#include "../../zeta_amd/csrc/evaltab.h"

using namespace zc;

// For a position and one of its moves, on the child: out[0] the evaluation
// (white positive) from the parent's piece sum, the move's change of it and
// the set-wise pawn terms; out[1] the sum of the per-square terms; out[2] the
// child's side to move in check; out[3] the same from node_basics.
extern "C" void hs_child(const uint64_t *b, int stm, uint32_t m, int32_t *out) {
  Pos p;
  p.b0 = b[0]; p.b1 = b[1]; p.b2 = b[2]; p.b3 = b[3]; p.cr = b[4]; p.stm = (u32)stm;
  int32_t base = 0;
  for (int sq = 0; sq < 64; sq++) {
    const u32 pc = piece_at(p, sq);
    if (((pc >> 1) & 7) != PNONE) base += eval_piece(EVAL_SQ.v, pc, sq);
  }
  const Pos c = apply(p, m, false);
  const u64 occ = c.b1 | c.b2 | c.b3;
  out[0] = base + eval_move_delta<true>(EVAL_SQ.v, p.stm, m) + pawn_terms(c.b1 & ~c.b2 & ~c.b3, c.b0 ^ occ, c.b0) + eval_bishop_pair(c);
  if (((m >> 27) & 7) != PNONE) {  // captures: the two short forms
    const Pos q = apply_capture(p, m);
    if (q.b0 != c.b0 || q.b1 != c.b1 || q.b2 != c.b2 || q.b3 != c.b3 || q.stm != c.stm) out[0] = 1 << 30;
    if (eval_move_delta<false>(EVAL_SQ.v, p.stm, m) != eval_move_delta<true>(EVAL_SQ.v, p.stm, m)) out[0] = 1 << 30;
  }
  out[1] = eval_bishop_pair(c);
  for (int sq = 0; sq < 64; sq++) out[1] += eval_square(c, sq);
  const u64 kb = c.b1 & c.b2 & ~c.b3 & (c.stm ? c.b0 : (c.b0 ^ occ));
  out[2] = king_attacked(c, sq_lines(kb ? lsb(kb) : 0), kb, c.stm ^ 1u) ? 1 : 0;
  Node0 B;
  node_basics(c, B);
  out[3] = B.checkers ? 1 : 0;
}
extern "C" int32_t hs_piece_value(int type) { return piece_value((u32)type); }
extern "C" int32_t hs_piece_value_table(int type) { return EVAL_VALUE[type]; }
