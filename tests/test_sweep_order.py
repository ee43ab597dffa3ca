"""When f64 sweeps put the links in parity order (sweep_order.hpp): programs of
sweeps and calls in site order, priced with the times measured in either order,
against the same programs in site order throughout."""
import ctypes

import pytest

from _host_rules import compile_rules

SOURCE = """
#include "sweep_order.hpp"
using namespace lqcd;
extern "C" {
double gain(int kind, int f64, int dim, double bytes, int n) {
    return parity_order_gain((SweepKind)kind, f64, dim, (size_t)bytes, n);
}
SweepOrder* make() { return new SweepOrder; }
void drop(SweepOrder* o) { delete o; }
int pays(SweepOrder* o, double g) { return o->pays(g); }
void swept(SweepOrder* o, double g) { o->swept(g); }
void site_call(SweepOrder* o) { o->site_call(); }
}
"""
MH, HB, OR = 0, 1, 2
# extents: us of two reorderings, then site and parity order per sweep of
# (kind, updates)
MEASURED = {
    (16,) * 4: (31, {(MH, 1): (197, 188), (MH, 10): (396, 384), (HB, 1): (281, 247), (OR, 1): (314, 281)}),
    (20,) * 4: (64, {(MH, 1): (350, 291), (MH, 10): (711, 657), (HB, 1): (526, 412), (OR, 1): (586, 496)}),
    (32,) * 4: (536, {(MH, 1): (1587, 1096), (MH, 10): (2571, 2413), (HB, 1): (2635, 1562), (OR, 1): (2556, 1703)}),
    (40,) * 4: (1102, {(MH, 1): (3621, 2543), (MH, 10): (5958, 5601), (HB, 1): (6297, 3497), (OR, 1): (6028, 3978)}),
    (64,) * 3: (85, {(MH, 1): (296, 224), (MH, 10): (569, 511), (HB, 1): (426, 330), (OR, 1): (505, 427)}),
    (128,) * 3: (762, {(MH, 1): (1662, 1267), (MH, 10): (3258, 3163), (HB, 1): (2894, 1741), (OR, 1): (2887, 1970)}),
    (512,) * 2: (56, {(MH, 1): (151, 130), (MH, 10): (344, 316), (HB, 1): (222, 184), (OR, 1): (510, 474)}),
    (2048,) * 2: (939, {(MH, 1): (1631, 1216), (MH, 10): (3726, 3730), (HB, 1): (2391, 1551), (OR, 1): (2452, 2190)}),
}


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    lib = compile_rules(tmp_path_factory.mktemp("rules"), SOURCE)
    lib.gain.restype = ctypes.c_double
    lib.gain.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_double, ctypes.c_int]
    lib.make.restype = ctypes.c_void_p
    for f in ("drop", "site_call"):
        getattr(lib, f).argtypes = [ctypes.c_void_p]
    for f in ("pays", "swept"):
        getattr(lib, f).argtypes = [ctypes.c_void_p, ctypes.c_double]
    return lib


class Program:
    """A lattice of the given extents; cost() is the time against site order."""

    def __init__(self, rules, ext):
        self.rules, self.dim = rules, len(ext)
        self.bytes = 144.0 * self.dim * ext[0] ** self.dim
        self.trip, self.sweeps = MEASURED[ext]
        self.order, self.parity, self.spent, self.reorders = rules.make(), False, 0.0, 0

    def __del__(self):
        self.rules.drop(self.order)

    def reorder(self, parity):
        if self.parity != parity:
            self.spent += self.trip / 2
            self.reorders += 1
            self.parity = parity

    def sweep(self, kind, n):
        gain = self.rules.gain(kind, 1, self.dim, self.bytes, n)
        if self.rules.pays(self.order, gain):
            self.reorder(True)
        self.rules.swept(self.order, gain)
        site, parity = self.sweeps[(kind, n)]
        self.spent += parity - site if self.parity else 0

    def site_call(self):
        self.rules.site_call(self.order)
        self.reorder(False)


@pytest.mark.parametrize("ext", MEASURED)
@pytest.mark.parametrize("k", [1, 2, 3, 5, 20])
@pytest.mark.parametrize("body", [[(MH, 1)], [(MH, 10)], [(HB, 1)], [(OR, 1)], [(HB, 1)] + [(OR, 1)] * 4,
                                  [(OR, 1), (MH, 1)]])
def test_repeated_programs_are_not_slower_than_site_order(rules, ext, k, body):
    """k times the sweeps of `body`, then a call in site order, again and again."""
    p = Program(rules, ext)
    for period in range(12):
        if period == 2:
            assert p.spent <= p.trip
            start = p.spent
        for _ in range(k):
            for kind, n in body:
                p.sweep(kind, n)
        p.site_call()
    assert p.spent <= start


@pytest.mark.parametrize("ext", [e for e in MEASURED if len(e) > 2])
@pytest.mark.parametrize("kind", [MH, HB, OR])
def test_long_runs_go_to_parity_order_once(rules, ext, kind):
    p = Program(rules, ext)
    for _ in range(50):
        p.sweep(kind, 1)
    assert p.parity and p.reorders == 1 and p.spent < 0


def test_fields_that_stay_in_site_order(rules):
    for kind in (MH, HB, OR):
        assert rules.gain(kind, 0, 4, 1e9, 1) == 0
        assert rules.gain(kind, 1, 4, (32 << 20) - 1, 1) == 0
        assert rules.gain(kind, 1, 4, 32 << 20, 1) > 0
