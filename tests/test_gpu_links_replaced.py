"""Calls that replace every link of a lattice whose links a sweep left in parity
order: the links are the new ones, and nothing is reordered first."""
import ctypes

import numpy as np
import pytest

import lqcd
import oracle as O
from lqcd import _ffi as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [2, 3, 4])
def test_replaced_links_are_not_reordered_first(d, tmp_path, monkeypatch):
    print(f"[gpu-case] links replaced after a sweep D={d}", flush=True)
    monkeypatch.setenv("LQCD_SWEEP_ORDER", "parity")
    ol = O.OracleLattice(d, [4] * d)
    given = lqcd.LatticeStateDefault(lqcd.LatticeCyclic(1.0, [4] * d, d), 6.0, ol.hot_start(9))
    links = given.link_matrix()
    files = {F.FORMAT_BINCODE: str(tmp_path / "s.bin"), F.FORMAT_JSON: str(tmp_path / "s.json")}
    for fmt, path in files.items():
        given.write(path, fmt)
    st = lqcd.LatticeStateDefault.new_determinist(1.0, 6.0, [4] * d, 5, d)
    random_links = st.link_matrix()
    ctx, beta = st._dev.ctx, ctypes.c_double()
    cold = ol.cold_start().reshape(links.shape)
    for name, replace, want in (
            ("upload", lambda: st.set_link_matrix(links), links),
            ("bincode", lambda: lqcd._raise(F.lib().lqcd_state_read(
                st.handle, files[F.FORMAT_BINCODE].encode(), F.FORMAT_BINCODE, 0, ctypes.byref(beta), None)), links),
            ("json", lambda: lqcd._raise(F.lib().lqcd_state_read(
                st.handle, files[F.FORMAT_JSON].encode(), F.FORMAT_JSON, 0, ctypes.byref(beta), None)), links),
            ("cold", lambda: lqcd._raise(F.lib().lqcd_links_cold(st.handle)), cold),
            ("random", lambda: lqcd._raise(F.lib().lqcd_links_random(st.handle, 5)), random_links)):
        st.monte_carlo_step(lqcd.OverrelaxationSweepRotation())
        ctx.profile_enable(1 << F.KERNEL_REORDER)
        replace()
        got = st.link_matrix()
        assert ctx.profile_read(F.KERNEL_REORDER)[0] == 0, name
        ctx.profile_enable(0)
        assert np.array_equal(got, want), name
    # a refused upload leaves the links that are there
    st.monte_carlo_step(lqcd.OverrelaxationSweepRotation())
    before = st.average_trace_plaquette()
    with pytest.raises(lqcd.StateInitializationError):
        lqcd._raise(F.lib().lqcd_links_upload(st.handle, links.ctypes.data_as(ctypes.c_void_p), links.shape[0] - 1))
    with pytest.raises(lqcd.LqcdError):
        lqcd._raise(F.lib().lqcd_state_read(st.handle, str(tmp_path / "absent").encode(), F.FORMAT_BINCODE, 0,
                                            ctypes.byref(beta), None))
    assert st.average_trace_plaquette() == before
    again = lqcd.LatticeStateDefault(st.lattice(), 6.0, st.link_matrix())
    assert again.average_trace_plaquette() == before
