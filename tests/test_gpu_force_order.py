"""The force kernel's workgroup order: lattices walked in slabs (whole
workgroups of 128 sites per slice, slowest extent a multiple of 8) and ones
that are not, the last workgroup full or not, against the oracle's force."""
import numpy as np
import pytest

import lqcd
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ext", [[8, 4, 4, 8], [8, 8, 8, 16], [16, 8, 8], [128, 8], [16, 8, 9], [5, 3, 7, 8], [3, 2]])
@pytest.mark.parametrize("precision", [lqcd.F64, lqcd.F32])
def test_force_of_every_link(ext, precision):
    print(f"[gpu-case] force order {ext} precision={precision}", flush=True)
    ol = O.OracleLattice(len(ext), ext)
    st = lqcd.LatticeStateDefault(lqcd.LatticeCyclic(1.0, ext, len(ext)), 6.0, ol.hot_start(3), precision)
    want = ol.derivative_e(st.link_matrix())   # at the links as they are stored
    got = lqcd.LatticeStateEFSyncDefault(st).derivative_e()
    # 1e-12 of the largest force in f64 arithmetic, 2e-6 in f32
    tol = (1e-12 if precision == lqcd.F64 else 2e-6) * np.max(np.abs(want))
    assert np.max(np.abs(got.reshape(-1) - want.reshape(-1))) <= tol
