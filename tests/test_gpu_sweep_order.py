"""Reorderings of the links that programs of sweeps cause, and the sweeps of
one order against the other (LQCD_SWEEP_ORDER), bit for bit."""
import numpy as np
import pytest

import lqcd
import test_gpu_parity_order as parity_order
from lqcd import _ffi as F

pytestmark = pytest.mark.gpu

EXT = [16, 16, 16, 16]   # 36 MiB of f64 links


class Reorders:
    """Number of reorderings since the last look."""

    def __init__(self, st):
        self.ctx = st._dev.ctx
        self.ctx.profile_enable(1 << F.KERNEL_REORDER)

    def __call__(self):
        n, _ = self.ctx.profile_read(F.KERNEL_REORDER)
        self.ctx.profile_enable(1 << F.KERNEL_REORDER)
        return n


def state(seed=5):
    return lqcd.LatticeStateDefault.new_determinist(1.0, 6.0, EXT, seed, 4, lqcd.F64)


def test_reorderings_of_f32_programs():
    """20^4, 44 MiB of f32 links: an update of a heat bath and overrelaxations
    pays, Metropolis sweeps do not."""
    print("[gpu-case] reorderings of f32 programs", flush=True)
    st = lqcd.LatticeStateDefault.new_determinist(1.0, 6.0, [20] * 4, 5, 4, lqcd.F32)
    count = Reorders(st)
    mh, hb, relax = lqcd.MetropolisHastingsSweep(1, 0.2, 3), lqcd.HeatBathSweep(4), lqcd.OverrelaxationSweepRotation()
    for _ in range(10):
        st.monte_carlo_step(mh)
    assert count() == 0
    for _ in range(3):
        st.monte_carlo_step(hb)
        st.normalize_link_matrices()
        for _ in range(4):
            st.monte_carlo_step(relax)
        st.average_trace_plaquette()
    assert count() == 1
    st.link_matrix()
    assert count() == 1
    st.monte_carlo_step(hb)      # the last stretch paid
    assert count() == 1
    st._dev.ctx.profile_enable(0)


def test_reorderings_of_programs():
    print("[gpu-case] reorderings of programs", flush=True)
    st = state()
    count = Reorders(st)
    mh, hb = lqcd.MetropolisHastingsSweep(1, 0.2, 3), lqcd.HeatBathSweep(4)
    # Metropolis sweeps each followed by a call in site order stay in site order
    for _ in range(3):
        st.monte_carlo_step(mh)
        st.magnetic_field_vec_field()
    assert count() == 0
    # a stretch of them goes to parity order once, and back once
    for _ in range(12):
        st.monte_carlo_step(mh)
        st.average_trace_plaquette()
    assert count() == 1
    st.magnetic_field_vec_field()
    assert count() == 1
    # a heat-bath sweep pays for the two by itself
    st = state()
    st.monte_carlo_step(hb)
    assert count() == 1
    st.normalize_link_matrices()
    st.link_matrix()
    assert count() == 1
    st._dev.ctx.profile_enable(0)


@pytest.mark.parametrize("ext", [[2, 2, 2, 2], [6, 4, 2, 8], [16, 16, 8, 8], [4, 6, 2], [34, 4, 6], [2, 4], [66, 18]])
@pytest.mark.parametrize("precision", [lqcd.F64, lqcd.F32])
def test_parity_order_of_any_size_gives_the_bits_of_site_order(ext, precision, monkeypatch):
    print(f"[gpu-case] sweep order {ext} precision={precision}", flush=True)
    parity = precision == lqcd.F64 or len(ext) == 4      # f32: built for D = 4
    links = {}
    for order in ("site", "parity"):
        monkeypatch.setenv("LQCD_SWEEP_ORDER", order)
        st = lqcd.LatticeStateDefault.new_determinist(1.0, 6.0, ext, 5, len(ext), precision)
        out = []
        count = Reorders(st)
        for u in (lqcd.MetropolisHastingsSweep(1, 0.2, 3), lqcd.MetropolisHastingsSweep(3, 0.2, 3),
                  lqcd.OverrelaxationSweepRotation(), lqcd.OverrelaxationSweepReverse(), lqcd.HeatBathSweep(4)):
            st.monte_carlo_step(u)
            assert count() == (parity and order == "parity")
            out += [st.average_trace_plaquette(), st.wilson_backward()]
            st.normalize_link_matrices()
            out.append(st.su3_distance())
            assert count() == 0
            out.append(st.link_matrix())
            assert count() == (parity and order == "parity")
        links[order] = out
        st._dev.ctx.profile_enable(0)
    for a, b in zip(links["site"], links["parity"]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("ext", [[16, 16, 16, 16], [26, 14, 14, 12], [48, 42, 40]])
def test_sweeps_and_reads_pinned_to_parity_order(ext, monkeypatch):
    monkeypatch.setenv("LQCD_SWEEP_ORDER", "parity")
    parity_order.test_sweeps_and_reads_in_parity_order(ext)


def test_site_order_calls_pinned_to_parity_order(monkeypatch):
    monkeypatch.setenv("LQCD_SWEEP_ORDER", "parity")
    parity_order.test_site_order_calls_from_parity_order()
