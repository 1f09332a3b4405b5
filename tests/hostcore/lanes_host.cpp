// Host build of the square-by-square move generation (zeta_amd/csrc/chess.h)
// against the set-wise one for CPU unit tests.  Test-only.
#include "../../zeta_amd/csrc/chess.h"

using namespace zc;

// 1 where the lanes take a board's moves: -1 if they differ from those emitted;
// 0 where one lane does
extern "C" int lh_serve(const uint64_t *b, int stm) {
  Pos p;
  p.b0 = b[0]; p.b1 = b[1]; p.b2 = b[2]; p.b3 = b[3]; p.cr = b[4]; p.stm = (u32)stm;
  Node0 B;
  node_basics(p, B);
  if (!lanes_serve(p, B)) return 0;
  u64 A = 0;
  for (int sq = 0; sq < 64; sq++)
    if (attacked_nk(B, sq)) A |= bit(sq);
  u64 t[64] = {0};
  Legal L;
  analyse(p, L);
  int n = 0;
  for_each_legal(p, L, [&](u32 m) {
    t[mv_from(m)] |= bit((int)mv_to(m));
    n++;
  });
  for (int sq = 0; sq < 64; sq++) {
    const u64 l = (B.own >> sq) & 1 ? lane_targets(p, B, A, sq, false) : 0;
    if (l != t[sq]) return -1;
    n -= popc(l);
  }
  return n ? -1 : 1;
}
