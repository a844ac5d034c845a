"""GPU: the right-hand side at the edges of its tiling, against the oracle.

A fine level's substep computes the rows inside those that finebound fills,
in 16 x 16 tiles, unless fewer than 16 points would be left in a direction;
the base level computes every row, with closures in its outer tiles.  Sizes
here leave 13, 16, 17 and 33 points inside (the whole-level fallback, one
tile, a tile of one overlap row, a remainder of one) with the odd z sizes the
grid forces, for every set of fields the split kernel has variants for: in
vacuum, with the scalar field alone, and with the Gamma-driver and the scalar
field (centred and upwinded advection).  Three coarse steps of both sides,
1e-10 of each array's maximum (the parity tests' bar)."""
import pytest

from parity_util import TOL, run_pair, worst

pytestmark = pytest.mark.gpu

PULSE = """
mattertype = scalar
idata = scalarpulse
scalarpulse_type = shell
scalar_a0 = 0.2
scalar_r0 = 0.0
scalar_z0 = 0.0
scalar_sr0 = 1.0
scalar_sz0 = 0.8
scalardiss = 0.1
"""

PHYSICS = {
    "vacuum": "idata = schwarzschild\nBH1mass = 1.0\nilapse = psiminus2\nintegrator = icn\n",
    "scalar": PULSE + "scalarmethod = first\nscalarpotential = phi2\nscalar_mass = 0.5\nintegrator = rk4\n",
    "scalar_shift": PULSE + "shift = Gammadriver2\ndrivercsi = 0.75\ndriveradv = .true.\nintegrator = rk4\n",
    "scalar_shift_centred": PULSE + "shift = Gammadriver2\nshiftadvect = .false.\ndrivereta = 0.5\nintegrator = icn\n",
}

SIZES = [(16, 16, True), (19, 22, False), (20, 19, True), (36, 39, False)]


@pytest.mark.parametrize("Nr,Nz,eqsym", SIZES)
@pytest.mark.parametrize("physics", sorted(PHYSICS))
def test_tile_edges_match_oracle(physics, Nr, Nz, eqsym, oaxis_mod, oracle_mod):
    text = """
order = four
dtfac = 0.25
boundtype = radiative
geodiss = 0.1
slicing = 1+log
gauge_f = 2.0
dr0 = 0.15
dz0 = 0.15
Nl0 = 1
Nrtotal = %d
Nztotal = %d
eqsym = %s
""" % (Nr, Nz, ".true." if eqsym else ".false.") + PHYSICS[physics]
    _, errs, times = run_pair(oaxis_mod, oracle_mod, text, 3)
    w, k = worst(errs)
    print("%s %dx%d eqsym %s: worst %.3e at %s" % (physics, Nr, Nz, eqsym, w, k))
    for tg, to in times:
        assert tg == to
    assert w <= TOL, "evolution differs: %.3e at %s" % (w, k)
