"""CPU: which speculative shots of a horizon search finished ones exclude
(oaxis_shots.h), against the walk that asks for them (horizon_finder.f90:434-855):
for random end slopes and random orders of finishing, a shot that the walk needs
is never excluded, the first of a launch never is whatever the slopes, and some
shots are excluded.  A NaN sends the walk on with a start slope that the launch
does not know, so only the first shot is promised there."""
import ctypes

import numpy as np
import pytest

import host_probe

PROBE = r"""
#define OA_HD inline
#include "oaxis_shots.h"
using namespace oax;

// finish the shots of a march in the given order; dropped[q]: shot q would have
// ended early, had it looked last of all
extern "C" void march(int n, const double* slope, const int* order, int* dropped) {
  int word = 0;
  char fin[4096] = {};
  for (int t = 0; t < n; ++t) {
    const int at = order[t];
    dropped[at] = march_excluded(at, n, word);
    if (dropped[at]) continue;          // a dropped shot has no result
    fin[at] = 1;
    for (int q = at - 1; q <= at + 1; q += 2) {
      if (q < 0 || q >= n || !fin[q]) continue;
      const int end = at > q ? at : q;
      if (march_ends(slope[at], slope[q]) && n - end > word) word = n - end;
    }
  }
}

extern "C" void tree(int n, double drada, const double* slope, const int* order, int* dropped) {
  int word[4096] = {};
  for (int t = 0; t < n; ++t) {
    const int at = order[t];
    dropped[at] = 0;
    for (int up = 1; tree_number(at, up) > 0; ++up)
      if (tree_excluded(at, up, word[tree_number(at, up) - 1])) dropped[at] = 1;
    if (dropped[at]) continue;
    const double p = drada * slope[at];
    word[at] = excludes_right(p) ? 2 : excludes_left(p) ? 1 : 0;
  }
}
"""

DP, IP = ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_int)


@pytest.fixture(scope="module")
def probe(tmp_path_factory, oaxis_mod):
    return host_probe.build(tmp_path_factory.mktemp("shots"), PROBE)


def finish(fn, head, slope, order):
    dropped = np.zeros(slope.size, dtype=np.int32)
    fn(*head, slope.ctypes.data_as(DP), order.ctypes.data_as(IP), dropped.ctypes.data_as(IP))
    return dropped.astype(bool)


def march_needs(slope):
    """The march stops after the first neighbours of different sign."""
    for q in range(1, slope.size):
        if not slope[q] * slope[q - 1] >= 0.0:
            return q + 1
    return slope.size


def tree_needs(slope, drada):
    """The nodes the bisection walks through (:774-792)."""
    path, at = [], 0
    while at < slope.size:
        path.append(at)
        if drada * slope[at] <= 0.0:
            at = 2 * at + 1
        else:
            drada = slope[at]
            at = 2 * at + 2
    return path


@pytest.mark.parametrize("n", [1, 2, 3, 17, 324, 1024])
@pytest.mark.parametrize("change", [0.0, 0.01, 0.5])
def test_march(probe, n, change):
    rng = np.random.default_rng(n)
    excluded = 0
    for _ in range(50):
        sign = np.cumprod(np.where(rng.random(n) < change, -1.0, 1.0))
        slope = sign * rng.uniform(0.0, 2.0, n)
        slope[rng.random(n) < 0.02] = 0.0
        order = rng.permutation(n).astype(np.int32)
        dropped = finish(probe.march, (n,), slope, order)
        assert not dropped[:march_needs(slope)].any()
        slope[rng.random(n) < 0.1] = np.nan                  # ends the march, as a change of sign does
        with_nan = finish(probe.march, (n,), slope, order)
        assert not with_nan[:march_needs(slope)].any()
        excluded += dropped.sum()
    if n >= 17:
        assert (excluded > 0) == (change > 0.0)


@pytest.mark.parametrize("depth", [1, 2, 5, 10])
def test_tree(probe, depth):
    rng = np.random.default_rng(depth)
    n, excluded = (1 << depth) - 1, 0
    for _ in range(100):
        slope = rng.standard_normal(n)
        slope[rng.random(n) < 0.02] = 0.0
        drada = rng.choice((-1.0, 1.0)) * rng.uniform(0.1, 2.0)
        order = rng.permutation(n).astype(np.int32)
        dropped = finish(probe.tree, (n, ctypes.c_double(drada)), slope, order)
        assert not dropped[tree_needs(slope, drada)].any()
        excluded += dropped.sum()
        slope[rng.random(n) < 0.2] = np.nan
        assert not finish(probe.tree, (n, ctypes.c_double(drada)), slope, order)[0]
    if depth > 1:
        assert excluded > 0
