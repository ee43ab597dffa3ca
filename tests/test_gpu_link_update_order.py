"""Single-link Metropolis updates of a lattice whose links a sweep left in
parity order: the same links, probabilities and decisions as in site order, bit
for bit, without a reordering."""
import numpy as np
import pytest

import lqcd
from lqcd import _ffi as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ext", [[2, 2, 2, 2], [4, 6, 2, 8], [4, 6, 2], [10, 2, 4], [2, 4], [10, 6]])
def test_link_updates_in_parity_order(ext, monkeypatch):
    print(f"[gpu-case] link updates in parity order {ext}", flush=True)
    got = {}
    for order in ("site", "parity"):
        monkeypatch.setenv("LQCD_SWEEP_ORDER", order)
        st = lqcd.LatticeStateDefault.new_determinist(1.0, 6.0, ext, 5, len(ext), lqcd.F64)
        st.monte_carlo_step(lqcd.MetropolisHastingsSweep(1, 0.2, 3))
        st._dev.ctx.profile_enable(1 << F.KERNEL_REORDER)
        mh, steps = lqcd.MetropolisHastingsDeltaDiagnostic(0.3, 11), []
        for _ in range(60):
            st.monte_carlo_step(mh)
            steps.append((mh.prob_replace_last(), mh.has_replace_last()))
        assert st._dev.ctx.profile_read(F.KERNEL_REORDER)[0] == 0
        st._dev.ctx.profile_enable(0)
        got[order] = steps, st.link_matrix()
    assert got["site"][0] == got["parity"][0]
    assert any(a for _, a in got["site"][0]) and not all(a for _, a in got["site"][0])
    assert np.array_equal(got["site"][1], got["parity"][1])
