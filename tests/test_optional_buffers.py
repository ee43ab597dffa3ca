"""The transports of the Gauss projection: both buffers or, where one cannot be
had, neither, with nothing left allocated (the projection then takes the steps
without them)."""
import pytest

from _host_rules import compile_rules

SOURCE = """
#include "optional_buffers.hpp"
#include <set>
#include <stdlib.h>
// allocation number `fail` (from 0) of two calls fails; bits of the result:
// 1 first call true, 2 second call true, 4 the buffers agree with the second
// result, 8 nothing is allocated that the buffers do not hold
extern "C" int run(int fail) {
    std::set<void*> live;
    int n = 0;
    double* p[2] = {nullptr, nullptr};
    auto alloc = [&](double** q, size_t bytes) {
        if (n++ == fail) {
            *q = (double*)1;
            return false;
        }
        *q = (double*)malloc(bytes);
        live.insert(*q);
        return true;
    };
    auto release = [&](double* q) { live.erase(q); free(q); };
    const bool a = lqcd::both_or_neither(p, 64, alloc, release);
    const bool b = lqcd::both_or_neither(p, 64, alloc, release);
    int r = (a ? 1 : 0) | (b ? 2 : 0);
    if (b ? p[0] && p[1] && p[0] != p[1] : !p[0] && !p[1]) r |= 4;
    if (live.size() == (size_t)(p[0] != nullptr) + (p[1] != nullptr)) r |= 8;
    for (double* q : p) free(q);
    return r;
}
"""


@pytest.mark.parametrize("fail,want", [(-1, 15), (0, 14), (1, 14)])
def test_both_or_neither(tmp_path, fail, want):
    assert compile_rules(tmp_path, SOURCE).run(fail) == want
