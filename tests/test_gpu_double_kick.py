"""The reference scheme's merged kicks: an integration of n kick-drift-kick
steps forms each force once and applies the two kicks of dt/2 that meet there
in one launch.  n steps in one call and n calls of one step (whose kicks are
launches of their own) give the same bits."""
import numpy as np
import pytest

import lqcd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [lqcd.F64, lqcd.F32])
@pytest.mark.parametrize("drift", [lqcd.DRIFT_ADDITIVE, lqcd.DRIFT_EXP])
@pytest.mark.parametrize("variant", [0, 1, 2, 3, 4])
def test_steps_in_one_call_match_single_steps(precision, drift, variant):
    integ = lqcd.SymplecticEulerGpu(drift, lqcd.SCHEME_REFERENCE)
    for ext in ([8, 4, 8, 8], [3, 5, 4], [7, 9]):
        print(f"[gpu-case] double kick {ext} precision={precision} drift={drift} variant={variant}", flush=True)
        sides = []
        for single in (False, True):
            st = lqcd.LatticeStateDefault.new_determinist(1.0, 6.0, ext, 11, len(ext), precision)
            st.set_md_variant(variant)
            ef = lqcd.LatticeStateEFSyncDefault.new_random_e_state(st, 5, 0, project=False)
            if single:
                for _ in range(4):
                    ef.simulate_symplectic(integ, 0.02)
            else:
                ef.simulate_symplectic_n(integ, 0.02, 4)
            sides.append((ef.link_matrix(), ef.e_field()))
        assert np.array_equal(sides[0][0], sides[1][0])
        assert np.array_equal(sides[0][1], sides[1][1])
