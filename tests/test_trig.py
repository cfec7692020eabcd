"""The sampling routines' sine and cosine and the fifth power of Schlick's
Fresnel term (bulbit_amd/csrc/bb_trig.h, compiled here with g++) against the
C library in long double.  They are evaluated in double, with an error of at
most about 1.5 units in its last place, and rounded once: the float is the
correctly rounded one unless the exact value lies that close to the middle
between two floats, which is so for about 3 in 2^29 values; then it is the
neighbour."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("trig") / "probe_trig")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-o", exe, os.path.join(HERE, "probe_trig.cpp")],
                   check=True)
    return exe


# the angles of the sampling routines: [0, 2 pi] and [-pi/4, 0), the smallest
# positive floats among them, and the ends of the stated range; the powers of
# what 1 - cos gives
@pytest.mark.parametrize("what,lo,hi,step,negative", [
    ("sincos", "0", "1e-6", 997, False), ("sincos", "1e-6", "6.2831855", 61, False),
    ("sincos", "1.5707", "1.5709", 1, False), ("sincos", "3.1415", "3.1417", 1, False),
    ("sincos", "6.2831", "8", 3, False), ("sincos", "1e-6", "0.7853982", 61, True),
    ("sincos", "0.78539", "8", 101, True),
    ("pow5", "1e-6", "1", 61, False), ("pow5", "1", "2", 61, False), ("pow5", "1e-7", "1e-3", 997, True)])
def test_correctly_rounded(probe, what, lo, hi, step, negative):
    out = subprocess.run([probe, what, lo, hi, str(step)] + (["-"] if negative else []), capture_output=True,
                         text=True, check=True).stdout.split()
    n, off, worst = int(out[0]), int(out[1]), float(out[2])
    assert n > 1000
    assert worst <= 1.0
    assert off <= 2 + n * 3.0 / 2 ** 29 * 4  # four times the share expected, and two more for small samples


def test_zeros(probe):
    # zero of either sign: sin keeps it, cos is 1 (each counted off would be a wrong bit pattern)
    for sign in ([], ["-"]):
        n, off, _ = subprocess.run([probe, "sincos", "0", "0", "1"] + sign, capture_output=True, text=True,
                                   check=True).stdout.split()
        assert (int(n), int(off)) == (2, 0)
