"""LDS that passes values between the lanes of a wavefront, by the text of the kernels: the compiler orders one lane's accesses only, so
wave_lds_order() has to stand between a store and another lane's load (what happens without it depends on the compiler, and is not made
to happen)."""

import os
import re

import pytest

import flydsl_amd

CSRC = os.path.join(os.path.dirname(flydsl_amd.__file__), "csrc")


@pytest.mark.parametrize("file,first,then", [
    # lane 0 of a token's group has stored the winners' weights, all its lanes scale them
    ("moe_gating.hip", r"mine\[k\] = w;", r"mine\[k\] \* f"),
    ("moe_sort.hip", r"mine\[k\] = w;", r"mine\[k\] \* f"),
    # ... before the next pass over the tokens stores the next ones
    ("moe_sort.hip", r"mine\[k\] \* f", r"^}"),
    # the running bases of the scatter: read by every lane, advanced by the first lane of an expert, read again for the next 64 pairs
    ("moe_sort.hip", r"base\[wave\]\[id\[c\]\] \+ __popcll\(below\)", r"base\[wave\]\[id\[c\]\] \+= "),
    ("moe_sort.hip", r"base\[wave\]\[id\[c\]\] \+= ", r"^}"),
])
def test_lanes_that_share_lds_are_ordered(file, first, then):
    text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, file)).read())
    start = re.search(first, text).end()
    end = start + re.search(then, text[start:], re.M).start()
    assert "wave_lds_order();" in text[start:end]
