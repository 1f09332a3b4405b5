// Host model of the search's windows (zeta_amd/csrc/bounds.h, the control flow
// of search.hip's k_search and qsearch) on random game graphs whose values are
// known by plain minimax, with the bound of the root's other workers rising at
// any visit.  Test-only.
#include <stdint.h>

#include <random>
#include <vector>

#include "../../zeta_amd/csrc/bounds.h"

using namespace zc;

namespace {
constexpr int INF = 32000;
constexpr int STATES = 48, MOVES = 4, CAPTURES = 3, MAXDEPTH = 5;

struct Entry {
  bool have = false, upper = false;
  int v = 0;
};

struct Model {
  std::mt19937 rng;
  bool shared;
  // side to move: the parity of the state; moves lead to the other parity,
  // captures to a higher state too, so that quiescence ends
  int move[STATES][MOVES], eval[STATES];
  std::vector<int> capture[STATES];
  int q[STATES], val[MAXDEPTH + 1][STATES];  // minimax, for the side to move
  Entry tt[MAXDEPTH + 1][STATES];
  uint32_t qkind[STATES];
  int qval[STATES];
  int ra = -INF, most = 0;  // most: the bound may rise to it
  long stores = 0, wrong = 0;

  int pick(int n) { return (int)(rng() % (unsigned)n); }
  Model(uint32_t seed, bool s) : rng(seed), shared(s) {
    for (int i = STATES - 1; i >= 0; i--) {
      for (int m = 0; m < MOVES; m++) move[i][m] = 2 * pick(STATES / 2) + !(i & 1);
      eval[i] = pick(41) - 20;
      for (int k = pick(CAPTURES + 1); k > 0; k--) {
        const int c = i + 1 + 2 * pick(6);
        if (c < STATES) capture[i].push_back(c);
      }
      q[i] = eval[i];
      for (int c : capture[i]) q[i] = q[i] > -q[c] ? q[i] : -q[c];
      qkind[i] = Q_NONE;
      val[0][i] = q[i];
    }
    for (int d = 1; d <= MAXDEPTH; d++)
      for (int i = 0; i < STATES; i++) {
        val[d][i] = -INF;
        for (int m : move[i]) val[d][i] = val[d][i] > -val[d - 1][m] ? val[d][i] : -val[d - 1][m];
      }
  }
  void visit() {
    if (pick(6) == 0) {
      const int b = most - pick(12);
      ra = b > ra ? b : ra;
    }
  }
  void store(int d, int i, bool lower, int v) {
    tt[d][i] = Entry{true, !lower, v};
    stores++;
    wrong += lower ? val[d][i] < v : val[d][i] > v;
  }
  void qstore(int i, uint32_t kind, int v) {
    if (kind == Q_NONE) return;
    qkind[i] = kind;
    qval[i] = v;
    stores++;
    wrong += ((kind & Q_LOWER) && q[i] < v) || ((kind & Q_UPPER) && q[i] > v);
  }

  int quiesce(int i, int sd, int alpha, int beta) {
    visit();
    if (floor_lifts(sd, ra, alpha, beta)) alpha = ra - 1;
    if (eval[i] >= beta) return eval[i];
    bool raised = false;
    if (shared && qkind[i] != Q_NONE) {
      if (qkind[i] == Q_EXACT || (qkind[i] == Q_LOWER && qval[i] >= beta) || (qkind[i] == Q_UPPER && qval[i] <= alpha))
        return qval[i];
      if (qkind[i] == Q_LOWER && qval[i] > alpha) {
        alpha = qval[i];
        raised = true;
      }
    }
    if (capture[i].empty()) {
      qstore(i, Q_EXACT, eval[i]);
      return eval[i];
    }
    if (eval[i] > alpha) {
      alpha = eval[i];
      raised = true;
    }
    for (int c : capture[i]) {
      const int v = -quiesce(c, sd + 1, -beta, -alpha);
      if (floor_lifts(sd, ra, alpha, beta)) {
        alpha = ra - 1;
        raised = false;
      }
      if (v > alpha) {
        alpha = v;
        raised = true;
      }
      if (alpha >= beta) {
        if (bound_holds(sd, ra, true, alpha)) qstore(i, Q_LOWER, alpha);
        return alpha;
      }
    }
    qstore(i, bound_kind(sd, ra, raised, alpha), alpha);
    return alpha;
  }

  int full(int i, int d, int sd, int alpha, int beta) {
    visit();
    if (floor_lifts(sd, ra, alpha, beta)) alpha = ra - 1;
    if (sd > 1 && tt[d][i].have) {
      const Entry &e = tt[d][i];
      if (e.upper ? e.v <= alpha : e.v > alpha) {
        if (!e.upper) alpha = e.v;
        if (e.upper || alpha >= beta) return alpha;
      }
    }
    bool best = false, again = false, scout = false;
    const int first = pick(MOVES);
    for (int k = 0; k < MOVES; k += !again) {
      const int c = move[i][(first + k) % MOVES];
      const int lo = sd == 1 && ra - 1 > alpha ? ra - 1 : alpha;
      scout = shared && !again && k > 0 && beta - lo > 1;
      again = false;
      const int hi = scout ? lo + 1 : beta;
      const int sc = -(d > 1 ? full(c, d - 1, sd + 1, -hi, -lo) : quiesce(c, sd + 1, -hi, -lo));
      if (floor_lifts(sd, ra, alpha, beta)) {
        alpha = ra - 1;
        best = false;
      }
      if (scout && sc > lo && sc < beta) {
        again = true;
        continue;
      }
      if (sc > alpha) {
        alpha = sc;
        best = true;
      }
      if (alpha >= beta || reply_suffices(sd, ra, alpha)) break;
    }
    if (bound_holds(sd, ra, best, alpha)) store(d, i, best, alpha);
    return alpha;
  }
};
}  // namespace

// Searches from every state on one table that is kept, iteration by iteration.
// out: bounds stored, bounds that minimax contradicts, searches, searches whose
// score is not the root's value.
extern "C" void hs_bounds(uint32_t seed, int shared, int64_t *out) {
  Model m(seed, shared != 0);
  int64_t searches = 0, off = 0;
  for (int round = 0; round < 4; round++)
    for (int i = 0; i < STATES; i++)
      for (int d = 1; d <= MAXDEPTH; d++) {
        m.ra = -INF;
        m.most = m.val[d][i];
        off += m.full(i, d, 1, -INF, INF) != m.val[d][i];
        searches++;
      }
  out[0] = m.stores;
  out[1] = m.wrong;
  out[2] = searches;
  out[3] = off;
}

// plies that captures from ply sd on a board of `pieces` can reach
extern "C" int hs_deepest(int sd, int pieces) {
  while (pieces > 2) {
    sd++;
    pieces--;
  }
  return sd;
}
extern "C" int hs_any_ply(int sd, int pieces, int maxply) { return any_ply(sd, pieces, maxply); }
