"""GPU: a search whose launches drop the shots that finished ones exclude
(horizon_finder.f90:434-855) is the search of the oracle, which integrates no
shot ahead: where the march ends at its first pair, late or never, and where the
bisection ends inside the first tree of steps, after it or needs several.  Which
shots a launch drops depends on when its waves finish, so no run here can say
that one was; which ones may be is checked on the CPU (test_host_shots.py).  The
sequence of shots is the oracle's exactly; where a horizon is found the surfaces
agree to the finder's 1e-10 (fields that differ by rounding; the last shot of a
search that finds none runs away and amplifies them)."""
import pytest

from test_gpu_horizon import compare, synthetic
from test_oracle_horizon import schwarzschild_fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extra", ["ahepsilon_shoot = 1.0D-2\n", "ahepsilon_shoot = 1.0D-5\nahzinit = 1.03\n",
                                   "ahepsilon_shoot = 1.0D-12\n"], ids=["one_tree", "first_pair", "many_trees"])
@pytest.mark.parametrize("mass", [2.0, 0.1], ids=["found", "too_small"])
def test_search_is_the_oracles(oaxis_mod, oracle_mod, extra, mass):
    dev, ref = synthetic(oaxis_mod, oracle_mod, 0.05, schwarzschild_fields(mass), extra=extra)
    for key in ("found", "shots", "errorflag", "zinit", "zcenter"):
        assert dev[key] == ref[key], (key, dev[key], ref[key])
    if ref["found"]:
        compare(dev, ref, extra)
