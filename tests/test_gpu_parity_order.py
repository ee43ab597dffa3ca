"""f64 sweeps of lattices whose links pass 32 MiB run with the links in parity
order.  The sweeps against the oracle's (every link, same streams), and every
way of reading the links afterwards against a lattice that was given them: the
ones that read either order (normalisation, plaquette, force) bit for bit, and
the ones that put them back in site order first."""
import numpy as np
import pytest

import lqcd
import oracle as O

pytestmark = pytest.mark.gpu

BETA, SEED = 6.0, 77


def reads(st):
    """What the readers of either order give."""
    return st.average_trace_plaquette(), st.hamiltonian_links(), st.su3_distance(), st.wilson_backward()


def check_reads(st):
    """The reads in the order the links are in now, against a fresh lattice
    with the same links; returns them (link_matrix: back in site order)."""
    got = reads(st)
    links = st.link_matrix()
    want = reads(lqcd.LatticeStateDefault(st.lattice(), BETA, links))
    assert got[:3] == want[:3]
    assert np.array_equal(got[3], want[3])
    return links


@pytest.mark.parametrize("ext", [[16, 16, 16, 16], [26, 14, 14, 12], [48, 42, 40]])
def test_sweeps_and_reads_in_parity_order(ext):
    d = len(ext)
    print(f"[gpu-case] parity order {ext}", flush=True)
    ol = O.OracleLattice(d, ext)
    assert ol.nlink * 144 >= 32 << 20
    st = lqcd.LatticeStateDefault.new_determinist(1.0, BETA, ext, SEED, d, lqcd.F64)
    u = st.link_matrix()
    mh = lqcd.MetropolisHastingsSweep(1, 0.2, SEED)
    for n in range(2):
        props, words = ol.device_mh_inputs(SEED, n, 0.2, 1)
        mh.next_element(st)
        u, ref = ol.metropolis_sweep(u, BETA, props, words, O.ORDER_CHECKERBOARD)
        assert mh.number_replace_last() == ref.number_replace_last
    got = check_reads(st)
    assert np.max(np.abs(got - u)) <= 1e-12
    # a cold lattice, heated; each sweep from the device's own links, so that
    # a rounding one sweep leaves is not amplified by the next
    u = ol.cold_start()
    st.set_link_matrix(u)
    sweeps = [lambda u: ol.normalize_link_matrices(ol.heat_bath_sweep(u, BETA, SEED, 0)[0]),
              lambda u: ol.normalize_link_matrices(ol.heat_bath_sweep(u, BETA, SEED, 1)[0]),
              ol.overrelaxation_sweep, ol.overrelaxation_reverse_sweep]
    hb = lqcd.HeatBathSweep(SEED)
    steps = [hb, hb, lqcd.OverrelaxationSweepRotation(), lqcd.OverrelaxationSweepReverse()]
    for step, sweep in zip(steps, sweeps):
        st.monte_carlo_step(step)
        if step is hb:
            st.normalize_link_matrices()
        want = sweep(u)
        u = check_reads(st)
        assert np.max(np.abs(u - want)) <= 1e-10


@pytest.mark.parametrize("ext,times", [([8, 4, 8, 8], [2, 4, 2, 2]), ([12, 14, 20], [4, 3, 2]), ([38, 18], [9, 19])])
def test_sweeps_of_a_tiled_lattice(ext, times):
    """A small lattice (site order) repeated to one that passes 32 MiB (parity
    order): a sweep of the large one is the repeated sweep of the small one, bit for
    bit, as every link sees the same values (host-given proposals, so that
    the streams repeat too)."""
    d = len(ext)
    big = [n * t for n, t in zip(ext, times)]
    print(f"[gpu-case] tiled parity order {big}", flush=True)
    assert np.prod(big) * d * 144 >= 32 << 20 > np.prod(ext) * d * 144

    def tiled(x):
        x = x.reshape(ext[::-1] + [d, -1])
        return np.tile(x, times[::-1] + [1, 1]).reshape(np.prod(big) * d, -1)

    ol = O.OracleLattice(d, ext)
    small = lqcd.LatticeStateDefault(lqcd.LatticeCyclic(1.0, ext, d), BETA, ol.hot_start(SEED))
    large = lqcd.LatticeStateDefault(lqcd.LatticeCyclic(1.0, big, d), BETA, tiled(small.link_matrix()))
    props, words = ol.device_mh_inputs(SEED, 0, 0.2, 1)
    big_words = np.ascontiguousarray(tiled(words.reshape(-1, 1)).reshape(-1))
    mh = lqcd.MetropolisHastingsSweep(1, 0.2, SEED)
    steps = [lambda s, p, w: mh.sweep(s, p, w),
             lambda s, p, w: s.monte_carlo_step(lqcd.OverrelaxationSweepRotation()),
             lambda s, p, w: s.monte_carlo_step(lqcd.OverrelaxationSweepReverse())]
    for step in steps:
        step(small, props, words)
        step(large, tiled(props[0])[None], big_words)
        assert np.array_equal(large.link_matrix(), tiled(small.link_matrix()))


def test_site_order_calls_from_parity_order():
    """Calls that need site order, each straight after a sweep, against the
    same call on a lattice that was given the links."""
    ext = [16, 16, 16, 16]
    print("[gpu-case] site-order calls from parity order", flush=True)
    st = lqcd.LatticeStateDefault.new_determinist(1.0, BETA, ext, SEED, 4, lqcd.F64)
    st.set_md_variant(3)
    integ = lqcd.SymplecticEulerGpu(lqcd.DRIFT_EXP, lqcd.SCHEME_LEAPFROG)
    mh = lqcd.MetropolisHastingsSweep(1, 0.2, SEED)

    def momenta(state):
        return lqcd.LatticeStateEFSyncDefault.new_random_e_state(state, 5, 0, project=False)

    def integrate(state):
        state.set_md_variant(3)
        ef = momenta(state)
        ef.simulate_symplectic_n(integ, 0.01, 3)
        return state.link_matrix(), ef.e_field()

    def trajectory(state):
        state.set_md_variant(3)
        hmc = lqcd.HybridMonteCarloDiagnostic(0.01, 4, integ, 9, project_gauss=False)
        state.monte_carlo_step(hmc)
        return state.link_matrix(), np.array([hmc.last_stats.h_old, hmc.last_stats.h_new])

    calls = [integrate, trajectory,
             lambda s: (s.f_mu_nu_field(), s.magnetic_field_vec_field()),
             lambda s: (momenta(s).gauss(), momenta(s).derivative_u()),
             lambda s: (s.monte_carlo_step(lqcd.MetropolisHastingsDeltaDiagnostic(0.2, 3)).link_matrix(),)]
    for call in calls:
        before = st.link_matrix()
        mh.next_element(st)              # parity order from here
        counter = mh.counter() - 1
        got = call(st)
        again = lqcd.LatticeStateDefault(st.lattice(), BETA, before)
        mh2 = lqcd.MetropolisHastingsSweep(1, 0.2, SEED)
        mh2._counter = counter
        mh2.next_element(again)
        given = lqcd.LatticeStateDefault(st.lattice(), BETA, again.link_matrix())
        for a, b in zip(got, call(given)):
            assert np.max(np.abs(np.asarray(a) - np.asarray(b))) <= 1e-12 * max(1.0, np.max(np.abs(b)))
    # starts over that write every link
    mh.next_element(st)
    lqcd._raise(lqcd._ffi.lib().lqcd_links_random(st.handle, SEED))
    fresh = lqcd.LatticeStateDefault.new_determinist(1.0, BETA, ext, SEED, 4, lqcd.F64)
    assert np.array_equal(st.link_matrix(), fresh.link_matrix())
    mh.next_element(st)
    lqcd._raise(lqcd._ffi.lib().lqcd_links_cold(st.handle))
    assert st.average_trace_plaquette() == 3.0
