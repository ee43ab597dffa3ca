"""The forms of an MD launch: one field chooses the form, and a launch that is
not built in it, or has nothing to write its sums to, is refused."""
import pytest

from _host_rules import compile_rules

SOURCE = """
#include "md_form.hpp"
extern "C" int valid(int form, int drift, int can_sum, int partials) {
    return lqcd::md_form_valid(form, drift, can_sum, partials);
}
"""
NONE, BEFORE, AFTER, TWICE = 0, 1, 2, 3


def test_forms(tmp_path):
    valid = compile_rules(tmp_path, SOURCE).valid
    for drift in (0, 1):
        for can_sum in (0, 1):
            for partials in (0, 1):
                assert valid(NONE, drift, can_sum, partials)
                assert valid(TWICE, drift, can_sum, partials) == drift
                assert valid(BEFORE, drift, can_sum, partials) == (drift and can_sum and partials)
                assert valid(AFTER, drift, can_sum, partials) == (not drift and can_sum and partials)
                assert not valid(-1, drift, can_sum, partials) and not valid(4, drift, can_sum, partials)
