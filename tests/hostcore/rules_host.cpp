// Host build of the move counts (zeta_amd/csrc/chess.h) for CPU unit tests.
// Test-only.
#include "../../zeta_amd/csrc/chess.h"

using namespace zc;

// out[0] the count of legal moves, out[1] how many for_each_legal emits (-1: a
// move whose two forms of apply differ, -2: one whose count changes with the
// e.p. flag that apply_count drops), out[2] how many it should
extern "C" void rh_count(const uint64_t *b, int stm, int32_t *out) {
  Pos p;
  p.b0 = b[0]; p.b1 = b[1]; p.b2 = b[2]; p.b3 = b[3]; p.cr = b[4]; p.stm = (u32)stm;
  Legal L;
  analyse(p, L);
  out[0] = count_legal(p, L, false);
  out[1] = 0;
  out[2] = count_emitted(p, L);
  bool same = true, counts = true;
  for_each_legal(p, L, [&](u32 m) {
    const Pos a = apply(p, m, true), v = apply_v(p, m);
    same = same && a.b0 == v.b0 && a.b1 == v.b1 && a.b2 == v.b2 && a.b3 == v.b3 && a.cr == v.cr && a.stm == v.stm;
    const Pos k = apply_count(p, m);
    if (k.cr != a.cr) {
      Legal A, K;
      analyse(a, A);
      analyse(k, K);
      counts = counts && count_legal(a, A, false) == count_legal(k, K, false);
    }
    out[1]++;
  });
  if (!same) out[1] = -1;
  if (!counts) out[1] = -2;
}

// 0 when the east and west rays of `s` by carry are those of the fills
extern "C" int rh_rays(uint64_t s, uint64_t occ) {
  const u64 e = ~occ;
  const u64 east = ray_east(s, e & NOTH), west = rev64(ray_east(rev64(s), rev64(e) & NOTH));
  return (east != slide<2>(s, e)) | (west != slide<3>(s, e)) << 1;
}

// the moves of a position whose king is not in check, lane by lane: their count
// (-1 where a square's targets are not those of lane_targets, -2 in check)
extern "C" int rh_lanes(const uint64_t *b, int stm) {
  Pos p;
  p.b0 = b[0]; p.b1 = b[1]; p.b2 = b[2]; p.b3 = b[3]; p.cr = b[4]; p.stm = (u32)stm;
  Node0 B;
  node_basics(p, B);
  u64 A = 0, An = 0;
  for (int sq = 0; sq < 64; sq++) {
    const LaneSq me = lane_sq(sq);
    if (lane_attacked(p, me, lane_rays(me, B.occ))) A |= bit(sq);
    if (attacked_nk(B, sq)) An |= bit(sq);
  }
  if ((A & B.kbb) != (B.checkers ? B.kbb : 0)) return -1;
  if (B.checkers) return -2;
  int n = 0;
  for (int sq = 0; sq < 64; sq++) {
    const LaneSq me = lane_sq(sq);
    const u64 t = lane_free_targets(p, me, lane_rays(me, B.occ), A, sq);
    if (t != ((B.own >> sq) & 1 ? lane_targets(p, B, An, sq, false) : 0)) return -1;
    n += popc(t);
  }
  return n;
}
extern "C" uint32_t rh_mod(uint64_t z, uint32_t n) { return mod_small(z, n); }
