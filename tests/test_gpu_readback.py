"""GPU: arrays and norms read back through the handle's pinned plane
(save2Ddata.f90, save0Ddata.f90:200-260): every size around the transposing
kernel's 32 x 32 tiles (ghosts included), wider leading dimensions and a
growing plane.  An upload followed by a download moves bits unchanged, so the
arrays must be equal, and the extreme norms are those of the same values."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr,nz", [(16, 16), (29, 61), (30, 62), (93, 29)])
@pytest.mark.parametrize("pad", [0, 5])
def test_readback_moves_bits(oaxis_mod, nr, nz, pad):
    oaxis = oaxis_mod
    p = oaxis.params_from_text("order = four\nidata = schwarzschild\neqsym = .true.\ndr0 = 0.2\ndz0 = 0.2\nNrtotal = %d\n"
                               "Nztotal = %d\nNl0 = 0\n" % (nr, nz))
    rng = np.random.default_rng(nr * nz)
    with oaxis.Spacetime(p) as st:
        n_r, n_z = st.shape(0)
        for name in ("alpha", "trK"):
            a = np.asfortranarray(rng.standard_normal((n_r, n_z)))
            st.upload(name, a, 0)
            out = np.full((n_r + pad, n_z), 7.0, order="F")
            rc = oaxis.lib().oa_download_field(st._h, 0, 0, name.encode(),
                                               out.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), n_r + pad)
            assert rc == 0
            assert np.array_equal(out[:n_r], a) and np.all(out[n_r:] == 7.0)
            norms = st.norms0d(name, 0)
            assert norms["max"] <= a.max() and norms["min"] >= a.min()
            assert norms["max"] in a and norms["min"] in a
