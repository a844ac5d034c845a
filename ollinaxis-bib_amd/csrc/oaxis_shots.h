// Which speculative shots of a horizon search finished ones exclude.  Included
// by oaxis_ah.hip after oaxis_device.h (OA_HD).
//
// A march shoots from positions 0, 1, .. n - 1 down the axis and ends at the
// first pair of neighbours whose end slopes differ in sign: the shots past a
// finished such pair are not needed.  A bisection's tree is a heap: node at has
// the children 2 at + 1 (left) and 2 at + 2 (right), and its end slope sends the
// walk into one of them; the other's subtree is not needed.
#pragma once

namespace oax {

// the march ends between two neighbours with these end slopes (a NaN ends it)
OA_HD bool march_ends(double d, double o) { return !(d * o >= 0.0); }
// shot at of n is past the pair; word: how many shots are from the nearest
// finished pair's second shot on (0: no pair)
OA_HD bool march_excluded(int at, int n, int word) { return word > 0 && at > n - word; }

// what a finished node excludes, from p = drada d: its right subtree (bit 2 of
// its word) or its left one (bit 1).  drada is the slope at the interval's start
// when the tree was launched; the walk replaces it only by slopes of its sign.
// A NaN excludes nothing.
OA_HD bool excludes_right(double p) { return p <= 0.0; }
OA_HD bool excludes_left(double p) { return p > 0.0; }
// 1 + the node `up` steps above node at, or 0
OA_HD int tree_number(int at, int up) { return (at + 1) >> up; }
// that ancestor's word excludes node at
OA_HD bool tree_excluded(int at, int up, int word) {
  const bool right = (((at + 1) >> (up - 1)) & 1) != 0;
  return (word & (right ? 2 : 1)) != 0;
}

}  // namespace oax
