"""Force and plaquette sums in every order of the workgroups, on sizes on both
sides of where it changes (test_launch_order.py), against the oracle."""
import numpy as np
import pytest

import lqcd
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ext", [[3, 2], [256, 256], [260, 254], [1024, 1024], [1030, 1020], [2048, 1024],
                                 [32, 32, 64], [34, 44, 46], [128, 128, 64], [104, 104, 98]])
@pytest.mark.parametrize("precision", [lqcd.F64, lqcd.F32])
def test_force_and_plaquette(ext, precision):
    print(f"[gpu-case] launch order {ext} precision={precision}", flush=True)
    ol = O.OracleLattice(len(ext), ext)
    st = lqcd.LatticeStateDefault.new_determinist(1.0, 6.0, ext, 3, len(ext), precision)
    u = st.link_matrix()
    want = ol.derivative_e(u)
    got = lqcd.LatticeStateEFSyncDefault(st).derivative_e()
    # as test_gpu_force_order.py
    tol = (1e-12 if precision == lqcd.F64 else 2e-6) * np.max(np.abs(want))
    assert np.max(np.abs(got.reshape(-1) - want.reshape(-1))) <= tol
    assert abs(st.average_trace_plaquette() - ol.average_trace_plaquette(u)) <= 1e-12
