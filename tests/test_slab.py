"""The traversal's box tests with margins (bulbit_amd/csrc/bb_slab.h, compiled
here with g++) against the exact one: a box that the exact test passes is never
lost, and the margins are no wider than a fraction of the boxes wherever the
scene lies."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SCENES = ["unit", "moved", "large", "huge", "small", "mixed", "flat"]
RAYS = ["plain", "axis", "far", "length", "any"]


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("slab") / "probe_slab")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fsanitize=undefined,float-cast-overflow",
                    "-fno-sanitize-recover=all", "-o", exe, os.path.join(HERE, "probe_slab.cpp")], check=True)

    def run(*args):
        out = subprocess.run([exe] + [str(a) for a in args], capture_output=True, text=True)
        assert out.returncode == 0, out.stderr
        return [float(x) if args[0] == "grid" else int(x) for x in out.stdout.split()]

    return run


@pytest.mark.parametrize("scene", SCENES)
@pytest.mark.parametrize("rays", RAYS)
def test_no_box_is_lost(probe, scene, rays):
    for seed in range(1, 6):
        tests, passes, with_margin, lost, _ = probe(scene, rays, seed)
        assert tests > 100_000 and passes > 100
        assert lost == 0
        # rays of moderate scenes, distances and lengths keep their margins
        assert with_margin == tests or rays in ("length", "any") or scene in ("large", "huge")


# boxes that only the margin passes make the walk longer: below 1 % of the
# boxes tested, for rays that meet about 1 % of them.  Margins that grew with
# the coordinates instead of the distances passed 8 to 33 % of the boxes of the
# scene far from the origin
@pytest.mark.parametrize("scene", ["unit", "moved", "mixed", "flat"])
@pytest.mark.parametrize("rays", ["plain", "axis", "far"])
def test_margins_are_narrow(probe, scene, rays):
    tests, _, _, _, loose = probe(scene, rays, 7)
    assert loose < 0.01 * tests


# boxes that are accepted but hold nothing: inverted ones (spheres of negative radius) beside ordinary ones and
# alone, and ones that are not finite; the grid's conversions stay in range, and ordinary entries keep their planes
@pytest.mark.parametrize("odd", [(5.0, -5.0), (1e30, -1e30), (0.5, 0.25), ("nan", 1.0), (0.0, "inf"), ("-inf", "nan")])
@pytest.mark.parametrize("all_odd", [False, True])
def test_grid_of_odd_boxes(probe, odd, all_odd):
    boxes = [odd] * 4 if all_odd else [(-1.0, 0.0), odd, (0.25, 2.0), odd]
    p, e, lo, hi = probe("grid", *[x for b in boxes for x in b], 0.5)
    if all_odd or "nan" in odd or "inf" in odd:
        return
    for k in (0, 2):
        low, high = (p + ((int(row) >> (8 * k)) & 255) * 2.0 ** e + 0.5 for row in (lo, hi))
        step = 2.0 ** e
        assert boxes[k][0] - step <= low <= boxes[k][0] and boxes[k][1] <= high <= boxes[k][1] + step
