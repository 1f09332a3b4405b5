// bounds.h -- windows under the bound that a root's workers share.
//
// `ra` is the best score that any worker has found for a move of the root in
// this iteration (-INF: none yet).  It only rises.  A root move with a value at
// or below ra - 1 cannot become the best one, so values at the root's side (odd
// plies, the root is ply 1) below ra - 1 are not told apart: a search below the
// root finds max(value, ra - 1) of a node there, and of a node of the other
// side min(value, 1 - ra).  What it found before ra rose holds of that too.
#pragma once
#include "chess.h"

namespace zc {

// odd plies from 3 on: the window starts at ra - 1, unless it ends below
ZD bool floor_lifts(int sd, int32_t ra, int32_t alpha, int32_t beta) {
  return (sd & 1) && sd >= 3 && ra - 1 > alpha && ra - 1 < beta;
}

// even plies: no better reply is needed to keep the root move at or below
// ra - 1.  The node is left, whether a reply has reached alpha or the window
// began there.
ZD bool reply_suffices(int sd, int32_t ra, int32_t alpha) { return !(sd & 1) && alpha >= 1 - ra; }

// Does a bound v of a node's value, found under ra, hold of the value itself,
// for any root and iteration?  The value that the search found is the larger
// one at an odd ply, the smaller one at an even ply; where v is on the far side
// of the floor the two compare with v alike.
ZD bool bound_holds(int sd, int32_t ra, bool lower, int32_t v) {
  return sd & 1 ? !lower || v >= ra : lower || v <= -ra;
}

// What a node that has seen all its moves with the result v, below beta, may
// store: a move (or the stand pat) raised alpha to v, or none did.
enum { Q_NONE = 0, Q_LOWER = 1, Q_UPPER = 2, Q_EXACT = 3 };
ZD uint32_t bound_kind(int sd, int32_t ra, bool raised, int32_t v) {
  return (raised && bound_holds(sd, ra, true, v) ? Q_LOWER : Q_NONE) | (bound_holds(sd, ra, false, v) ? Q_UPPER : Q_NONE);
}

// Is a quiescence value at ply sd out of the ply limit's reach, whatever the
// captures below?  Each takes a piece off, and two that are left are a draw.
ZD bool any_ply(int sd, int pieces, int maxply) { return sd + pieces <= maxply; }

}  // namespace zc
