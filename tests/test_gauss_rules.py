"""Which kernel the Gauss law and its projection take, by size and pinned."""
import ctypes

import pytest

from _host_rules import compile_rules

SOURCE = """
#include "gauss_rules.hpp"
using namespace lqcd;
static Geom geom(int dim, const int* ext) {
    Geom g = {};
    g.dim = dim;
    g.nsite = 1;
    for (int d = 0; d < dim; ++d) {
        g.extent[d] = ext[d];
        g.nsite *= ext[d];
    }
    g.npad = (g.nsite + 255) / 256 * 256;
    return g;
}
extern "C" int transports(int dim, const int* ext) { return gauss_uses_transports(geom(dim, ext)); }
extern "C" void tiles(int dim, const int* ext, int* out) {
    const GaussTiles t = gauss_tiles(geom(dim, ext));
    out[0] = t.a;
    out[1] = t.b;
    out[2] = t.C;
    out[3] = t.nblocks;
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    lib = compile_rules(tmp_path_factory.mktemp("rules"), SOURCE)

    def path(ext):
        """"transports", "walk" or C of the streamed tiles."""
        c, t = (ctypes.c_int * len(ext))(*ext), (ctypes.c_int * 4)()
        if lib.transports(len(ext), c):
            return "transports"
        lib.tiles(len(ext), c, t)
        if t[0] == 0:
            return "walk"
        n = ext[0] * ext[1] * ext[2] * ext[3]
        assert ext[0] * t[0] * t[1] == 256 and ext[1] % t[0] == 0 and ext[2] % t[1] == 0 and ext[3] % t[2] == 0
        assert t[3] * t[2] * 256 == n and t[3] <= 4096
        return t[2]

    return path


# extents: by size; without the transports; the site walk pinned; the transports pinned
CASES = [([8, 16, 8, 4], "transports", 1, "walk", "transports"), ([16, 8, 8, 4], "transports", 1, "walk", "transports"),
         ([8, 8, 4, 4], "transports", 1, "walk", "transports"), ([8] * 4, "transports", 1, "walk", "transports"),
         ([16, 16, 16, 8], 1, 1, "walk", "transports"), ([16] * 4, 1, 1, "walk", "transports"),
         ([16, 16, 16, 32], 2, 2, "walk", "transports"), ([32, 16, 16, 16], 2, 2, "walk", "transports"),
         ([16, 16, 16, 64], 2, 2, "walk", "transports"), ([32, 16, 16, 32], 2, 2, "walk", "transports"),
         ([64, 16, 32, 16], 4, 4, "walk", "transports"), ([16, 16, 16, 128], 4, 4, "walk", "transports"),
         ([32] * 4, 8, 8, "walk", "transports"), ([12, 10, 6, 9], "transports", "walk", "walk", "transports"),
         ([70, 40], "transports", "walk", "walk", "transports"), ([1024, 1024], "walk", "walk", "walk", "transports"),
         ([8] * 3, "walk", "walk", "walk", "walk"), ([48] * 4, "walk", "walk", "walk", "transports")]


@pytest.mark.parametrize("ext,by_size,streamed,walk,transports", CASES)
def test_kernel_of_the_steps(rules, monkeypatch, ext, by_size, streamed, walk, transports):
    for var in ("LQCD_GAUSS_TRANSPORTS", "LQCD_GAUSS_TILES"):
        monkeypatch.delenv(var, raising=False)
    assert rules(ext) == by_size
    monkeypatch.setenv("LQCD_GAUSS_TRANSPORTS", "0")
    assert rules(ext) == streamed
    monkeypatch.setenv("LQCD_GAUSS_TRANSPORTS", "1")
    assert rules(ext) == transports
    monkeypatch.setenv("LQCD_GAUSS_TILES", "0")
    assert rules(ext) == "walk"
    monkeypatch.delenv("LQCD_GAUSS_TRANSPORTS")
    assert rules(ext) == walk
