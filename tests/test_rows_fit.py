"""Buffers of a bit-exact prompt's rows: grown in powers of two, halved where the
device's memory does not hold them, and none (the tokens then go one step at a time)
where it does not hold two rows.  Compiles csrc/rows_fit.h for the host."""
import os
import subprocess

import pytest

from conftest import PKG, REPO


@pytest.fixture(scope="module")
def fit(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("rows") / "rows_fit_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(PKG, "csrc"),
                    os.path.join(REPO, "tests", "rows_fit_check.cpp"), "-o", out], check=True)

    def run(*args):
        r = subprocess.run([out] + [str(a) for a in args], check=True, capture_output=True, text=True)
        got, *asked = map(int, r.stdout.split())
        return got, asked
    return run


# want, have, most, limit -> rows granted, sizes asked for
@pytest.mark.parametrize("args,got,asked", [
    ((201, 0, 2048, 10 ** 9), 201, [256]),            # grown to the next power of two
    ((201, 256, 2048, 0), 201, []),                   # held already: nothing is asked for
    ((257, 256, 2048, 10 ** 9), 257, [512]),
    ((2048, 0, 2048, 10 ** 9), 2048, [2048]),
    ((2000, 0, 2000, 10 ** 9), 2000, [2000]),         # at most `most`
    ((2048, 512, 2048, 700), 512, [2048, 1024, 512]),  # what memory holds
    ((300, 0, 2048, 300), 256, [512, 256]),
    ((2, 0, 2048, 2), 2, [2]),
    ((600, 0, 2048, 1), 0, [1024, 512, 256, 128, 64, 32, 16, 8, 4, 2]),  # not even two rows
])
def test_rows_fit(fit, args, got, asked):
    assert fit(*args) == (got, asked)
