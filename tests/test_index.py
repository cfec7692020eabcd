"""Index arithmetic of the kernels (bulbit_amd/csrc/bb_index.h, compiled here
with g++) up to the largest images and batches that a call accepts, against
the same on Python's integers."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
MOST = 1 << 30  # pixels of an image


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("index") / "probe_index")
    subprocess.run(["g++", "-std=c++17", "-O2", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-o", exe,
                    os.path.join(HERE, "probe_index.cpp")], check=True)

    def run(what, cases):
        text = "".join(what + " " + " ".join(str(x) for x in c) + "\n" for c in cases)
        out = subprocess.run([exe], input=text, capture_output=True, text=True)
        assert out.returncode == 0, out.stderr
        return [tuple(int(x) for x in line.split()) for line in out.stdout.splitlines()]

    return run


def _pixel(width, height, q):
    """strips of 8 columns, row by row within a strip"""
    strip = q // (8 * height)
    r = q - strip * 8 * height
    w = min(8, width - 8 * strip)
    return 8 * strip + r % w, r // w


@pytest.mark.parametrize("width,height", [(1, 1), (1, 9), (5, 4), (7, 33), (8, 8), (9, 3), (16, 2), (65, 33)])
def test_path_order_is_a_permutation(probe, width, height):
    got = probe("pixel", [(width, height, q) for q in range(width * height)])
    assert got == [_pixel(width, height, q) for q in range(width * height)]
    assert sorted(got) == sorted((x, y) for x in range(width) for y in range(height))


# narrow images whose 8-pixel strip would be larger than a 32-bit integer, and the largest of other shapes
@pytest.mark.parametrize("width,height", [(1, 268435455), (1, 268435456), (1, 480_000_000), (1, 536870911), (1, MOST),
                                          (2, MOST // 2), (3, MOST // 3), (7, MOST // 7), (8, MOST // 8),
                                          (9, MOST // 9), (32768, 32768), (MOST, 1)])
def test_path_order_of_the_largest_images(probe, width, height):
    n = width * height
    qs = sorted({q for k in range(33) for q in (n * k // 32 - 1, n * k // 32, n * k // 32 + 1) if 0 <= q < n})
    assert probe("pixel", [(width, height, q) for q in qs]) == [_pixel(width, height, q) for q in qs]


# a batch takes up to 2^31 - 1 rays of two vectors each, an image 2^30 pixels of three floats
def test_places_of_the_last_rays_and_pixels(probe):
    rays = [0, 1, 2 ** 30 - 1, 2 ** 30, 2 ** 31 - 1]
    assert probe("ray", [(i,) for i in rays]) == [(2 * i,) for i in rays]
    pixels = [0, 1, 2 ** 31 // 3, 2 ** 31 // 3 + 1, 2 ** 30 - 1]
    assert probe("film", [(p,) for p in pixels]) == [(3 * p,) for p in pixels]


def test_claims_up_to_the_last_query(probe):
    most = 2 ** 31 - 1
    cases = [(rb, re, n) for end in (128, most) for re in (end - 64, end - 1, end) for rb in range(re - 66, re + 1)
             for n in (0, 1, 31, 63, 64)]
    assert probe("claim", cases) == [(rb + n if rb + n < re else -1, min(rb + n, re)) for rb, re, n in cases]
