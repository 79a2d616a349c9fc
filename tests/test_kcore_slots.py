"""The k-core peeling's rotation of list counts (kcore_slots.hpp), for every
order in which blocks can pass from a barrier into the next phase: between two
barriers no block appends to a count that another may still read or that one
clears, and every count appended to starts at zero."""
import ctypes
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WRAP = r"""
#include "kcore_slots.hpp"
extern "C" {
unsigned slot(unsigned r) { return gpr::kc_slot(r); }
unsigned after_empty(unsigned r) { return gpr::kc_after_empty(r); }
unsigned by_round(unsigned r) { return gpr::kc_cleared_by_round(r); }
unsigned by_pass(unsigned r) { return gpr::kc_cleared_by_pass(r); }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("slots")
    (d / "wrap.cpp").write_text(WRAP)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "graptor_amd", "csrc"), "-o",
                    str(d / "wrap.so"), str(d / "wrap.cpp")], check=True)
    lib = ctypes.CDLL(str(d / "wrap.so"))
    return {name: getattr(lib, name) for name in ("slot", "after_empty", "by_round", "by_pass")}


def run(rules, levels):
    """levels: per pass, the rounds that follow it.  A phase clears one slot and appends to another between the same
    two barriers at whose first every block reads the list that the phase before it filled."""
    count, read, r = [0, 0, 0], None, 0

    def phase(clear, append, some):
        nonlocal read
        assert append != read and clear != read, "a count is written that a block may still read"
        assert append != clear, "a count is cleared while it is appended to"
        assert count[append] == 0, "a list starts with a count left over"
        count[clear], count[append] = 0, int(some)
        read = append    # behind the barrier

    for k, rounds in enumerate(levels):
        if k:
            r = rules["after_empty"](r)
        phase(rules["by_pass"](r), rules["slot"](r), rounds > 0)
        for left in range(rounds - 1, -1, -1):
            phase(rules["by_round"](r), rules["slot"](r + 1), left > 0)
            r += 1


def plans():
    rng = random.Random(7)
    return [[0], [0, 0, 0, 0, 0, 0, 0], [1] * 9, [2] * 9, [3] * 9, [4] * 9] + \
        [[rng.choice((0, 0, 1, 2, 3, 7)) for _ in range(40)] for _ in range(200)]


def test_counts_are_not_written_while_they_may_be_read(rules):
    for p in plans():
        run(rules, p)


def test_the_check_sees_a_pass_that_refills_the_list_just_read(rules):
    with pytest.raises(AssertionError, match="may still read"):
        run(dict(rules, after_empty=lambda r: r), [2, 2, 2])
