"""The order in which the plaquette sums and the force kernel take the blocks of
sites, by dimension and size (launch_order.hpp)."""
import ctypes

import pytest

from _host_rules import compile_rules

SOURCE = """
#include "launch_order.hpp"
using namespace lqcd;
static Geom geom(int dim, const int* ext) {
    Geom g = {};
    g.dim = dim;
    g.nsite = 1;
    for (int d = 0; d < dim; ++d) {
        g.extent[d] = ext[d];
        g.stride[d] = g.nsite;
        g.nsite *= ext[d];
    }
    return g;
}
extern "C" void plaquette(int dim, const int* ext, long long* pg) {
    int64_t P, G;
    plaquette_order(geom(dim, ext), P, G);
    pg[0] = P;
    pg[1] = G;
}
extern "C" void force(int dim, const int* ext, long long* pg) {
    int64_t P, G;
    force_order(geom(dim, ext), 128, P, G);
    pg[0] = P;
    pg[1] = G;
}
"""
STORAGE, XCD = "storage", "contiguous"


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    lib = compile_rules(tmp_path_factory.mktemp("rules"), SOURCE)

    def kind(which, ext, block):
        pg = (ctypes.c_longlong * 2)()
        getattr(lib, which)(len(ext), (ctypes.c_int * len(ext))(*ext), pg)
        if pg[0] <= 0:
            return STORAGE if pg[0] < 0 else XCD
        # slabs: whole workgroups per slice, every slice once
        slice_sites = 1
        for n in ext[:-1]:
            slice_sites *= n
        assert pg[0] * block == slice_sites and pg[1] * 8 == ext[-1]
        return "slabs"

    return lambda ext: (kind("plaquette", ext, 256), kind("force", ext, 128))


@pytest.mark.parametrize("ext,plaquette,force", [
    ([16] * 4, "slabs", "slabs"), ([32] * 4, "slabs", "slabs"), ([15, 13, 11, 17], XCD, XCD),
    ([48, 48, 48, 96], XCD, "slabs"), ([2] * 4, XCD, XCD),
    ([32] * 3, STORAGE, "slabs"), ([64] * 3, XCD, "slabs"), ([100] * 3, XCD, XCD), ([104] * 3, STORAGE, XCD),
    ([128] * 3, STORAGE, "slabs"), ([5, 3, 7], STORAGE, XCD),
    ([256, 256], STORAGE, XCD), ([333, 217], XCD, XCD), ([1024, 1024], XCD, XCD), ([1200, 1200], STORAGE, XCD),
    ([2048, 1024], STORAGE, STORAGE), ([2048, 2048], STORAGE, STORAGE), ([2500, 2500], STORAGE, XCD), ([3, 2], STORAGE, XCD)])
def test_order(order, ext, plaquette, force):
    assert order(ext) == (plaquette, force)
