"""The Gauss projection of small lattices (steps with the transports U^+ E U
carried along) against the oracle's: tiles of 64 sites with and without a
remainder, D = 2 and 4, one workgroup per tile and several tiles per
workgroup, and a lattice on either side of the streamed tiles' size."""
import numpy as np
import pytest

import lqcd
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ext", [[5, 3, 7, 4], [4, 4, 4, 4], [6, 10, 4, 8], [13, 12, 11, 10], [16, 16, 8, 8],
                                 [16, 16, 16, 8], [9, 7], [64, 2], [530, 510]])
@pytest.mark.parametrize("precision", [lqcd.F64, lqcd.F32])
def test_projection_matches_oracle(ext, precision):
    d = len(ext)
    print(f"[gpu-case] gauss transports {ext} precision={precision}", flush=True)
    ol = O.OracleLattice(d, ext)
    st = lqcd.LatticeStateDefault(lqcd.LatticeCyclic(1.0, ext, d), 6.0, ol.hot_start(4), precision)
    ef = lqcd.LatticeStateEFSyncDefault(st, ol.random_efield(5, 0.5 / 6.0))
    u, e = st.link_matrix(), ef.e_field()      # as they are stored
    ef.project_to_gauss(2000)
    rc, want, _ = ol.project_to_gauss(u, e, 2000)
    assert rc == 0
    # at the stop a site's deviation is below 320 eps = 7e-14; one group of
    # steps more or less moves E by about that over (1 - rate): 1e-11 in f64,
    # the rounding of the stored E in f32
    tol = 1e-11 if precision == lqcd.F64 else 1e-7 * np.max(np.abs(want))
    assert np.max(np.abs(ef.e_field() - np.asarray(want).reshape(-1, 8))) <= tol
    if precision == lqcd.F64:
        assert ef.gauss_sum_div() <= 1.01 * 2.220446049250313e-16 * ol.nsite * 320
