"""The built library holds no kernel that its dispatch never launches."""
import os

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lattice-qcd-rs_amd", "lqcd",
                   "liblqcd_hip.so")


@pytest.mark.skipif(not os.path.exists(LIB), reason="library not built")
@pytest.mark.parametrize("kernel", ["k_gauss_start", "k_gauss_links"])
def test_transports_are_built_for_the_dimensions_that_take_them(kernel):
    """gauss_uses_transports: not D = 3."""
    data = open(LIB, "rb").read()
    name = f"{len(kernel)}{kernel}ILi%dE".encode()
    assert [d for d in (2, 3, 4) if name % d in data] == [2, 4]
