"""GPU: arrays and norms read back through the handle's pinned plane
(save2Ddata.f90, save0Ddata.f90:200-260): every size around the transposing
kernel's 32 x 32 tiles (ghosts included), wider leading dimensions and a
growing plane.  An upload followed by a download moves bits unchanged, so the
arrays must be equal.  The norms are those of the values the kernel reduces
(i in [1, Nr-g], j in [1, Nz-g]): max, min and max|f| exactly, the root mean
square to n 2^-53 (n non-negative terms in any order).  Between norms the plane
holds another array, of larger and then of smaller values, so that a partial
left over from it would show."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check_norms(st, name, a, g):
    s = a[g:a.shape[0] - g, g:a.shape[1] - g]
    n = st.norms0d(name, 0)
    assert n["max"] == s.max() and n["min"] == s.min() and n["nm1"] == np.abs(s).max(), (name, n)
    rms = np.sqrt(np.mean(s * s))
    assert abs(n["nm2"] - rms) <= s.size * 2.0 ** -53 * rms, (name, n["nm2"], rms)


@pytest.mark.parametrize("nr,nz", [(16, 16), (29, 61), (30, 62), (93, 29)])
@pytest.mark.parametrize("pad", [0, 5])
def test_readback_moves_bits(oaxis_mod, nr, nz, pad):
    oaxis = oaxis_mod
    p = oaxis.params_from_text("order = four\nidata = schwarzschild\neqsym = .true.\ndr0 = 0.2\ndz0 = 0.2\nNrtotal = %d\n"
                               "Nztotal = %d\nNl0 = 0\n" % (nr, nz))
    rng = np.random.default_rng(nr * nz)
    with oaxis.Spacetime(p) as st:
        n_r, n_z = st.shape(0)
        held = {}
        for name, scale in (("alpha", 1.0), ("trK", 1.0e6), ("KTA", 1.0e-6)):
            a = np.asfortranarray(scale * rng.standard_normal((n_r, n_z)))
            st.upload(name, a, 0)
            held[name] = a
            out = np.full((n_r + pad, n_z), 7.0, order="F")
            rc = oaxis.lib().oa_download_field(st._h, 0, 0, name.encode(),
                                               out.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), n_r + pad)
            assert rc == 0
            assert np.array_equal(out[:n_r], a) and np.all(out[n_r:] == 7.0)
            check_norms(st, name, a, 3)
        for name in ("trK", "KTA", "alpha", "KTA"):
            check_norms(st, name, held[name], 3)
            assert np.array_equal(st.download("trK", 0), held["trK"])
