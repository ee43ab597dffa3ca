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
# extents (f64): us of two reorderings, then site and parity order per sweep of
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

MEASURED_F32 = {
    (20,) * 4: (37, {(MH, 1): (277, 268), (MH, 10): (650, 633), (HB, 1): (370, 335), (OR, 1): (428, 401)}),
    (24,) * 4: (67, {(MH, 1): (353, 343), (MH, 10): (888, 874), (HB, 1): (532, 455), (OR, 1): (629, 538)}),
    (32,) * 4: (221, {(MH, 1): (730, 683), (MH, 10): (2122, 2077), (HB, 1): (1199, 986), (OR, 1): (1362, 1197)}),
    (40,) * 4: (503, {(MH, 1): (1935, 1783), (MH, 10): (5258, 5151), (HB, 1): (2791, 2334), (OR, 1): (3177, 2866)}),
    (128,) * 3: (343, {(MH, 1): (938, 899), (MH, 10): (2950, 3042), (HB, 1): (1329, 1235), (OR, 1): (1628, 1580)}),
}
LATTICES = [(ext, 1) for ext in MEASURED] + [(ext, 0) for ext in MEASURED_F32]


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

    def __init__(self, rules, ext, f64):
        self.rules, self.dim, self.f64 = rules, len(ext), f64
        self.bytes = (144.0 if f64 else 72.0) * self.dim * ext[0] ** self.dim
        self.trip, self.sweeps = (MEASURED if f64 else MEASURED_F32)[ext]
        self.order, self.parity, self.spent, self.reorders = rules.make(), False, 0.0, 0

    def __del__(self):
        self.rules.drop(self.order)

    def reorder(self, parity):
        if self.parity != parity:
            self.spent += self.trip / 2
            self.reorders += 1
            self.parity = parity

    def sweep(self, kind, n):
        gain = self.rules.gain(kind, self.f64, self.dim, self.bytes, n)
        if self.rules.pays(self.order, gain):
            self.reorder(True)
        self.rules.swept(self.order, gain)
        site, parity = self.sweeps[(kind, n)]
        self.spent += parity - site if self.parity else 0

    def site_call(self):
        self.rules.site_call(self.order)
        self.reorder(False)


@pytest.mark.parametrize("ext,f64", LATTICES)
@pytest.mark.parametrize("k", [1, 2, 3, 5, 20])
@pytest.mark.parametrize("body", [[(MH, 1)], [(MH, 10)], [(HB, 1)], [(OR, 1)], [(HB, 1)] + [(OR, 1)] * 4,
                                  [(OR, 1), (MH, 1)]])
def test_repeated_programs_are_not_slower_than_site_order(rules, ext, f64, k, body):
    """k times the sweeps of `body`, then a call in site order, again and again."""
    p = Program(rules, ext, f64)
    for period in range(12):
        if period == 2:
            assert p.spent <= p.trip
            start = p.spent
        for _ in range(k):
            for kind, n in body:
                p.sweep(kind, n)
        p.site_call()
    assert p.spent <= start


@pytest.mark.parametrize("ext,f64", [x for x in LATTICES if len(x[0]) > 2])
@pytest.mark.parametrize("kind", [MH, HB, OR])
def test_long_runs_go_to_parity_order_once(rules, ext, f64, kind):
    p = Program(rules, ext, f64)
    for _ in range(50):
        p.sweep(kind, 1)
    if f64 or (len(ext) == 4 and kind != MH):
        assert p.parity and p.reorders == 1 and p.spent < 0
    else:
        assert not p.parity and p.spent == 0


def test_fields_that_stay_in_site_order(rules):
    for kind in (MH, HB, OR):
        for f64 in (0, 1):
            assert rules.gain(kind, f64, 4, (32 << 20) - 1, 1) == 0
        assert rules.gain(kind, 1, 4, 32 << 20, 1) > 0
        assert rules.gain(kind, 0, 3, 1e9, 1) == rules.gain(kind, 0, 2, 1e9, 1) == 0
