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
