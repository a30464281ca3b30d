"""What csrc/native.cpp does while the interpreter's lock is given up, by its text (the mistake it guards against ends the process, so it
is not made to happen): nothing but the call into the library, and the lock is taken back on every way out."""

import os
import re

import flydsl_amd

SOURCE = os.path.join(os.path.dirname(flydsl_amd.__file__), "csrc", "native.cpp")


def _without_comments():
    return re.sub(r"//[^\n]*", "", open(SOURCE).read())


def _bodies(text):
    """The argument of every released(...) call."""
    for m in re.finditer(r"return released\(", text):
        depth, i = 1, m.end()
        while depth:
            depth += {"(": 1, ")": -1}.get(text[i], 0)
            i += 1
        yield text[m.end():i - 1]


def test_no_tensor_is_touched_without_the_lock():
    bodies = list(_bodies(_without_comments()))
    assert len(bodies) == 5
    for body in bodies:
        # a tensor's members may throw, materialise a copy-on-write storage or change under another thread
        assert "->" not in body and "data_ptr" not in body and "x_code" not in body and "Py" not in body, body


def test_the_lock_comes_back_when_something_throws():
    # the macros restore the thread state only where the block is left at its end
    assert "Py_BEGIN_ALLOW_THREADS" not in _without_comments()
