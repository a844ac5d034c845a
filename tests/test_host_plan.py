"""CPU: the launch records of a plan (oa_plan.h), formed on the host.  A
substep called on its own takes a fine level's outer rows beside the rows
inside them, in the two-phase kernel as a second item of the same level: the
launch still advances Nr x Nz points."""
import ctypes

import pytest

import host_probe

PROBE = r"""
#include "oa_plan.h"
using namespace oax;

// points of the record of one substep of a level, whole (frame = 1) or
// without the rows that finebound fills
extern "C" double substep_points(int Nr, int Nz, int eqsym, int shift, int scalar, int frame, int* items) {
  RhsItem it{};
  it.G.Nr = Nr;
  it.G.Nz = Nz;
  it.G.g = 3;
  it.G.eqsym = eqsym;
  it.G.jlo = eqsym ? 1 : -2;
  bool inner = true;
  if (rhs_tiles(&it, rhs_by_parts(shift != 0, scalar != 0), &inner) != OA_OK) return -1.0;
  std::vector<RhsItem> v(1, it);
  if (frame && inner) rhs_add_frame(&v, rhs_by_parts(shift != 0, scalar != 0));
  *items = static_cast<int>(v.size());
  Plan p;
  p.add(K_RHS, shift != 0, scalar != 0, false, v);
  return p.launches.front().points;
}
"""


@pytest.fixture(scope="module")
def probe(tmp_path_factory, oaxis_mod):
    lib = host_probe.build(tmp_path_factory.mktemp("plan"), PROBE)
    lib.substep_points.restype = ctypes.c_double
    return lib


@pytest.mark.parametrize("shift,scalar", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("frame", [0, 1])
@pytest.mark.parametrize("Nr,Nz,eqsym", [(16, 17, 1), (19, 24, 0), (64, 128, 1), (93, 210, 0)])
def test_a_substep_counts_each_point_once(probe, Nr, Nz, eqsym, shift, scalar, frame):
    items = ctypes.c_int()
    pts = probe.substep_points(Nr, Nz, eqsym, shift, scalar, frame, ctypes.byref(items))
    assert pts == float(Nr * Nz), (pts, items.value)
    # the two-phase kernel (Gamma-driver in vacuum) is where the frame is an item
    if frame and Nr > 19:
        assert items.value == (2 if shift and not scalar else 1)
