"""GPU: the relaxation's level steps at the edges of their tiles (elliptic.hip;
wave_elliptic.f90:542-1164), against the oracle's solve with the same number
of steps.  A level step of the default relaxation runs by tiles of 8 x 16
points along rho and z, and by tiles of 16 x 16 where those number 256 or more
(256 x 256 points and up): the grids end one point before, on and after a tile
of each form, with and without equatorial symmetry, a fine boundary and the
u^5 term, and 240 x 271 (255 tiles) is the last size of the smaller one.  RK4
goes iteration by iteration, here with a fine level's boundary.  Bound: the steps
are the same sums in another order, rounded at 2^-53 each; a step has under
2^7 of them and the damped relaxation does not amplify, so 120 coarse steps
(with subcycling under 2^9 level steps) stay within 2^-53 * 2^16 < 1e-10 of
the field's largest value."""
import pytest

from parity_util import compare_state
from test_gpu_elliptic import BRILL, PULSE

pytestmark = pytest.mark.gpu

STEPS = "WE_maxiter = 120\nWE_epsilon = 1.0D-30\n"
CASES = {
    "tile_16": (PULSE, 16, 16, 1, "eqsym = .true.\n"),
    "one_past_17x33": (PULSE, 17, 33, 1, "eqsym = .true.\n"),
    "one_before_31x47": (PULSE, 31, 47, 1, "eqsym = .true.\n"),
    "whole_plane_18x45": (PULSE, 18, 45, 1, "eqsym = .false.\n"),
    "potential_33x16": (PULSE, 33, 16, 2, "eqsym = .true.\nscalarpotential = phi2\nscalar_mass = 0.1\n"),
    "brill_49x31": (BRILL, 49, 31, 0, ""),
    "last_of_8_rows_240x271": (PULSE, 240, 271, 0, "eqsym = .true.\n"),
    "rows_16_tiles_256x271": (PULSE, 256, 271, 0, "eqsym = .true.\n"),
    "rows_16_one_past_257x273": (PULSE, 257, 273, 0, "eqsym = .true.\n"),
    "rows_16_one_before_271x271": (BRILL, 271, 271, 0, ""),
    "rows_16_fine_259x256": (PULSE, 259, 256, 1, "eqsym = .false.\n"),
    "rows_16_potential_257x272": (PULSE, 257, 272, 1, "eqsym = .true.\nscalarpotential = phi2\nscalar_mass = 0.1\n"),
    "rk4_18x34": (PULSE, 18, 34, 1, "eqsym = .false.\nWE_method = rk4\n"),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_level_steps_at_tile_edges(oaxis_mod, oracle_mod, case):
    oaxis = oaxis_mod
    text, nr, nz, nl, more = CASES[case]
    p = oaxis.params_from_text(text + "dr0 = 0.3\ndz0 = 0.3\nNrtotal = %d\nNztotal = %d\nNl0 = %d\n" % (nr, nz, nl)
                               + STEPS + more)
    print("case", case, flush=True)
    oracle_mod.ell_stationary(False)
    try:
        orc = oracle_mod.Oracle(p)
        orc.initial_data()
    finally:
        oracle_mod.ell_stationary(True)
    with oaxis.Spacetime(p) as st:
        st.initial_data(stationary_exit=False)
        s_dev, s_orc = st.elliptic_stats(), orc.ell_stats()
        assert (s_dev["steps0"], s_dev["steps1"]) == (s_orc["steps0"], s_orc["steps1"])
        orc.initial_aux()
        st.initial_aux()
        errs = compare_state(oaxis, st, orc, p)
    orc.close()
    worst = max(errs.items(), key=lambda kv: kv[1])
    print("  worst %s" % (worst,), flush=True)
    bad = {k: v for k, v in errs.items() if not v <= 1e-10}
    assert not bad, bad
