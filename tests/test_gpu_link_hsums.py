"""H of lqcd_hmc_trajectory summed inside the per-link MD kernels (f64).

Variants 0 and 1 have one workgroup of sums per (direction, site block); the
lattices leave the last block of 256 sites partly empty, hold exactly one or
two blocks, or one site more.  Against the plaquette kernel's H of the same
states: every link's trace carries about 100 roundings and the blocks are
summed in trees, below 2e-14 of the sum; twice that for the cancellation in
N_plaquettes - sum / 12, rounded up to 1e-13.  Both variants put their
partials in the same order: the same bits.  In f32 the per-link kernels leave
H to the plaquette kernel: the same bits as hamiltonian_total.
"""
import sys

import numpy as np
import pytest

import oracle as O
import lqcd

pytestmark = pytest.mark.gpu


def run(ext, u, e, precision, variant, drift, scheme, graph=False, steps=3):
    dim = len(ext)
    st = lqcd.LatticeStateDefault(lqcd.LatticeCyclic(1.0, ext, dim), 5.8, u, precision)
    st.set_md_variant(variant)
    st.set_md_graph(graph)
    ef = lqcd.LatticeStateEFSyncDefault(st, e)
    before = ef.hamiltonian_total()
    hmc = lqcd.HybridMonteCarloDiagnostic(0.01, steps, lqcd.SymplecticEulerGpu(drift, scheme), 1, project_gauss=False)
    s = hmc.trajectory(st, 0)    # accept word 0: accepted unless p == 0
    assert s.accepted == 1
    return s, before, ef.hamiltonian_total()


@pytest.mark.parametrize("ext", [[16, 16], [257, 2], [8, 8, 8], [5, 3, 17], [4, 4, 4, 4], [5, 3, 7, 5]])
@pytest.mark.parametrize("drift,scheme", [(lqcd.DRIFT_EXP, lqcd.SCHEME_LEAPFROG),
                                          (lqcd.DRIFT_ADDITIVE, lqcd.SCHEME_REFERENCE)])
def test_link_variants_sum_h(ext, drift, scheme):
    print(f"\n[gpu-case] per-link H sums ext={ext} drift={drift} scheme={scheme}", flush=True)
    sys.stdout.flush()
    ol = O.OracleLattice(len(ext), ext)
    u = ol.hot_start(41)
    e = ol.random_efield(42, 0.3)
    seen = []
    for variant in (0, 1):
        for graph in (False, True):
            s, before, after = run(ext, u, e, lqcd.F64, variant, drift, scheme, graph)
            assert abs(s.h_old - before) <= 1e-13 * abs(before)
            assert abs(s.h_new - after) <= 1e-13 * abs(after)
            seen.append((s.h_old, s.h_new))
    assert len(set(seen)) == 1
    u32 = u.astype(np.float32).astype(np.float64)
    e32 = e.astype(np.float32).astype(np.float64)
    for variant in (0, 1):
        s, before, after = run(ext, u32, e32, lqcd.F32, variant, drift, scheme)
        assert (s.h_old, s.h_new) == (before, after)
