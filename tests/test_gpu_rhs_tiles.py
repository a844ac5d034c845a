"""GPU: the right-hand side at the edges of its tiling, against the oracle.

A fine level's substep computes the rows inside those that finebound fills,
in 16 x 16 tiles, unless fewer than 16 points would be left in a direction.
The base level computes every row: by parts the outer 3 rows are strips, of 64
points along z at the outer rho edge and of 62 points along rho at each z edge
(the last strip along z is anchored to the level's end and overlaps the one
before), and the rest tiles; the Gamma-driver in vacuum, in two phases, takes
tiles over the whole level.

The smaller sizes leave 13, 16, 17 and 33 points inside (the whole-level
fallback, one tile, a tile of one overlap row, a remainder of one); the larger
ones end a strip one before, on and after its end: 64, 65 and 127 points along
z, 62, 63 and 64 along rho.  Every set of fields the kernels have variants for:
in vacuum, with the scalar field alone, with the Gamma-driver alone, and with
both (centred and upwinded advection).  Three coarse steps of both sides, 1e-10
of each array's maximum (the parity tests' bar); the pieces called one by one,
whose fine substeps take the outer rows too, equal the planned step bit for
bit at sizes with one and with two strips a side."""
import numpy as np
import pytest

from parity_util import TOL, run_pair, worst
from test_gpu_piecewise import onestep

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
    "shift": "idata = BrillWave\nbrill_a0 = 2.0\nbrill_sr0 = 1.0\nbrill_sz0 = 1.0\nshift = Gammadriver2\n"
             "drivercsi = 0.75\nintegrator = icn\n",
    "scalar_shift": PULSE + "shift = Gammadriver2\ndrivercsi = 0.75\ndriveradv = .true.\nintegrator = rk4\n",
    "scalar_shift_centred": PULSE + "shift = Gammadriver2\nshiftadvect = .false.\ndrivereta = 0.5\nintegrator = icn\n",
}

SIZES = [(16, 16, True), (19, 22, False), (20, 19, True), (36, 39, False), (65, 64, True), (66, 65, True),
         (67, 127, True), (65, 62, False), (66, 124, False)]


def text_of(physics, Nr, Nz, eqsym):
    # 100 relaxation steps of psi are enough for data that both sides start from
    cap = "WE_maxiter = 100\n" if Nr > 60 or physics == "shift" else ""
    return """
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
""" % (Nr, Nz, ".true." if eqsym else ".false.") + PHYSICS[physics] + cap


@pytest.mark.parametrize("Nr,Nz,eqsym", SIZES)
@pytest.mark.parametrize("physics", sorted(PHYSICS))
def test_tile_edges_match_oracle(physics, Nr, Nz, eqsym, oaxis_mod, oracle_mod):
    _, errs, times = run_pair(oaxis_mod, oracle_mod, text_of(physics, Nr, Nz, eqsym), 3)
    w, k = worst(errs)
    print("%s %dx%d eqsym %s: worst %.3e at %s" % (physics, Nr, Nz, eqsym, w, k), flush=True)
    for tg, to in times:
        assert tg == to
    assert w <= TOL, "evolution differs: %.3e at %s" % (w, k)


@pytest.mark.parametrize("Nr,Nz,eqsym", [(36, 39, False), (66, 65, True)])
@pytest.mark.parametrize("physics", sorted(PHYSICS))
def test_pieces_equal_the_planned_step(physics, Nr, Nz, eqsym, oaxis_mod):
    oaxis = oaxis_mod
    p = oaxis.params_from_text(text_of(physics, Nr, Nz, eqsym))
    with oaxis.Spacetime(p) as whole, oaxis.Spacetime(p) as piece:
        for st in (whole, piece):
            st.initial_data()
            st.initial_aux()
        for _ in range(3):
            whole.coarse_step()
            onestep(oaxis, piece, p, 0)
        for lev in range(whole.nlevels):
            assert whole.time(lev) == piece.time(lev)
            for name in oaxis.state_fields(p):
                a, b = whole.download(name, lev), piece.download(name, lev)
                assert np.array_equal(a, b), (lev, name, np.abs(a - b).max())
