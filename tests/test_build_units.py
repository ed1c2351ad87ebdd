"""The solver's translation units: every 7-smooth length of 32 to 1024 has its
kernels once, tuned or in a unit of its own."""

import re

from kwave_amd import build


def smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


def test_one_unit_per_length():
    text = open(build.CSRC + "/kw_kernels.hpp").read()
    tuned = [int(n) for n in re.findall(r"X\((\d+)\)", re.search(r"#define KW_FAST_SIZES.*", text).group(0))]
    lens = build.len_sizes()
    assert sorted(tuned + lens) == [n for n in range(32, 1025) if smooth(n)]
    units = build.solver_units()
    assert [u[2] for u in units if u[0] == build.LEN_SOURCE] == [[f"-DKW_LENGTH={n}"] for n in reversed(lens)]
    assert len({u[1] for u in units}) == len(units)
