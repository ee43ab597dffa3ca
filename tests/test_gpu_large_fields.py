"""F_mu_nu of lattices whose link planes of all directions pass 4 GiB while
those of one direction do not, on sites over the whole range (the first, the
last, and some between) against the oracle, to the 1e-12 of smaller ones."""
import ctypes

import numpy as np
import pytest

import lqcd
import oracle as O
from lqcd import _ffi as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ext", [[216, 216, 216], [48, 48, 48, 72]])
def test_f_mu_nu_past_one_resource(ext):
    d = len(ext)
    print(f"[gpu-case] F_mu_nu past one resource {ext}", flush=True)
    n = int(np.prod(ext))
    assert n * d * 144 > 1 << 32 > n * 144
    st = lqcd.LatticeStateDefault.new_determinist(1.0, 6.0, ext, 3, d, lqcd.F64)
    out = F.DeviceBuffer(n * d * d * 18 * 8)
    lqcd._raise(F.lib().lqcd_field_strength_device(st.handle, F.FIELD_F_MU_NU, out.ptr, n * d * d * 18))
    u = st.link_matrix()
    ol = O.OracleLattice(d, ext)
    got = np.empty((d, d, 18))
    sites = np.concatenate([np.arange(0, 40), np.arange(n - 40, n), np.random.default_rng(1).integers(0, n, 200)])
    for s in sites:
        rc = F.hip_runtime().hipMemcpy(got.ctypes.data_as(ctypes.c_void_p),
                                       ctypes.c_void_p(out.ptr + int(s) * got.nbytes), got.nbytes, 2)
        assert rc == 0
        for i in range(d):
            for j in range(d):
                assert np.max(np.abs(got[i, j] - ol.f_mu_nu(u, int(s), i, j))) <= 1e-12, (int(s), i, j)
