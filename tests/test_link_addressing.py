"""F_mu_nu reads the links of all directions through one buffer resource where
their planes fit in its 32-bit offsets, and through one per direction where
they do not: the choice on both sides of the limit, against the bytes the
planes take."""
import ctypes

import pytest

from _host_rules import compile_rules

SOURCE = """
#include "limits.hpp"
extern "C" int all_links(int dim, long long npad, int elem) {
    lqcd::Geom g = {};
    g.dim = dim;
    g.nsite = g.npad = npad;
    return lqcd::all_links_addressable(g, elem);
}
extern "C" int direction(long long npad, int elem) { return lqcd::direction_addressable(npad, elem); }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    lib = compile_rules(tmp_path_factory.mktemp("rules"), SOURCE)
    lib.all_links.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_int]
    lib.direction.argtypes = [ctypes.c_longlong, ctypes.c_int]
    return lib


def padded(n):
    return (n + 255) // 256 * 256


@pytest.mark.parametrize("elem", [4, 8])
@pytest.mark.parametrize("dim", [2, 3, 4])
def test_one_resource_holds_every_link_plane(rules, dim, elem):
    # 9 entries of two reals per site and direction
    last = ((1 << 32) - 1) // (dim * 9 * 2 * elem) // 256 * 256
    for npad in (256, last - 256, last, last + 256, 2 * last, 2 * last + 256):
        assert rules.all_links(dim, npad, elem) == (npad * dim * 9 * 2 * elem < 1 << 32), npad
        # a lattice that one resource reaches is one whose directions fit too
        if rules.all_links(dim, npad, elem):
            assert rules.direction(npad, elem)


@pytest.mark.parametrize("ext,elem,one", [([32] * 4, 4, True), ([48, 48, 48, 96], 4, True), ([48, 48, 48, 96], 8, False),
                                          ([256] * 3, 4, True), ([256] * 3, 8, False), ([128] * 3, 8, True),
                                          ([64] * 4, 4, False), ([56, 56, 56, 48], 4, True)])
def test_lattices_around_the_limit(rules, ext, elem, one):
    n = 1
    for x in ext:
        n *= x
    assert rules.direction(padded(n), elem)
    assert rules.all_links(len(ext), padded(n), elem) == one
