"""The launch-shape rules (symphas_amd/csrc/shape.hpp), compiled for the host,
against times measured on an MI355X: what a rule picks is no slower than what it
passes over."""
import random
import shutil
import subprocess
from pathlib import Path

import pytest

HOST = Path(__file__).resolve().parent / "host"


@pytest.fixture(scope="module")
def pick(tmp_path_factory):
    """pick(lines): what shape_check prints for them, split."""
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    exe = tmp_path_factory.mktemp("shape") / "shape_check"
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-o", str(exe),
                    str(HOST / "shape_check.cpp")], check=True)

    def run(lines):
        out = subprocess.run([str(exe)], input="\n".join(lines) + "\n", text=True,
                             capture_output=True, check=True).stdout
        return [tuple(int(v) for v in line.split()) for line in out.splitlines()]

    return run


# reference-order step, <15,10,25>: (bytes of a value, sides, us per step with
# one thread per site, as a plane stream), Model B and Allen-Cahn
ONE_SITE = [
    (4, (36, 36, 36), 6.99, 7.56), (4, (40, 40, 40), 7.07, 7.58), (4, (44, 44, 44), 7.19, 7.59),
    (4, (48, 48, 48), 11.51, 7.60), (4, (64, 64, 64), 12.65, 7.90), (4, (24, 24, 100), 11.53, 7.50),
    (4, (100, 24, 24), 7.23, 7.68), (4, (24, 100, 24), 11.52, 7.58), (4, (50, 60, 20), 7.04, 7.74),
    (4, (120, 40, 20), 7.40, 7.76), (4, (24, 60, 60), 12.15, 7.59), (4, (62, 62, 24), 7.09, 7.81),
    (8, (36, 36, 36), 13.82, 8.27), (8, (44, 44, 44), 14.42, 8.36), (8, (64, 64, 64), 26.65, 8.63),
    (8, (100, 24, 24), 14.14, 8.34), (8, (120, 40, 20), 14.68, 8.53), (8, (62, 62, 24), 13.89, 8.49),
    (4, (36, 36, 36), 4.18, 4.87), (4, (44, 44, 44), 4.33, 4.82), (4, (48, 48, 48), 6.37, 4.75),
    (4, (120, 40, 20), 4.43, 4.82), (8, (36, 36, 36), 7.25, 5.20), (8, (120, 40, 20), 7.71, 5.42),
]


def test_one_site_or_stream(pick):
    got = pick([f"one_site {x} {y} {z} {es}" for es, (x, y, z), _, _ in ONE_SITE])
    for (es, n, one_site, stream), (one,) in zip(ONE_SITE, got):
        assert (one_site if one else stream) == min(one_site, stream), (es, n)


# 3D Model B, compact stencil: bytes of a value, sides, times of two steps of
# tall waves in one round (us of 50 steps, one plan alone and of three in turn),
# the rule's shape, its times
RADIUS_TWO = [
    (8, (161, 150, 97), (606, 447), (2, 4, 14), (562, 416)),
    (8, (200, 200, 200), (1190, 1298), (2, 4, 40), (1195, 1300)),
    (8, (103, 194, 243), (827, 763), (2, 4, 25), (828, 770)),
    (8, (256, 256, 256), (2298, 2604), (2, 4, 86), (2307, 2630)),
    (8, (61, 500, 200), (1373, 1384), (2, 4, 50), (1380, 1390)),
    (8, (39, 258, 50), (579, 214), (1, 4, 4), (346, 172)),
    (8, (120, 240, 160), (979, 838), (1, 4, 10), (818, 652)),
    (8, (240, 240, 240), (2146, 2271), (2, 4, 80), (2148, 2281)),
    (8, (300, 280, 260), (3926, 3418), (2, 4, 130), (3946, 3441)),
    (8, (64, 64, 64), (564, 207), (1, 4, 2), (253, 121)),
    (8, (32, 32, 32), (549, 262), (2, 4, 1), (219, 94)),
    (8, (24, 290, 290), (710, 656), (2, 4, 21), (711, 658)),
    (8, (290, 24, 30), (573, 259), (1, 4, 1), (260, 117)),
    (8, (100, 100, 100), (598, 249), (1, 4, 5), (383, 209)),
    (8, (128, 128, 128), (598, 422), (2, 4, 16), (598, 423)),
    (8, (150, 150, 150), (680, 585), (2, 4, 19), (683, 582)),
    (8, (180, 97, 77), (595, 290), (1, 4, 6), (439, 248)),
    (8, (220, 61, 133), (598, 329), (1, 4, 9), (513, 307)),
    (8, (250, 130, 60), (602, 382), (1, 4, 10), (562, 332)),
    (8, (300, 300, 100), (1433, 1486), (2, 4, 50), (1441, 1488)),
    (8, (130, 60, 250), (597, 410), (1, 4, 12), (589, 335)),
    (8, (80, 80, 80), (580, 202), (1, 4, 4), (326, 167)),
    (8, (170, 40, 90), (596, 216), (1, 4, 3), (314, 160)),
    (8, (290, 290, 40), (707, 578), (1, 4, 8), (690, 533)),
    (4, (161, 150, 97), (775, 372), (2, 6, 8), (413, 206)),
    (4, (103, 194, 243), (788, 373), (2, 6, 17), (576, 336)),
    (4, (110, 110, 300), (785, 358), (2, 6, 12), (469, 258)),
    (4, (256, 256, 256), (1195, 1055), (2, 12, 16), (1195, 1057)),
    (4, (61, 500, 200), (1153, 551), (2, 12, 17), (838, 524)),
    (4, (39, 258, 50), (747, 379), (2, 4, 4), (253, 119)),
    (4, (120, 240, 160), (785, 377), (2, 6, 20), (645, 351)),
    (4, (240, 240, 240), (1176, 897), (2, 12, 24), (1066, 857)),
    (4, (300, 280, 260), (1362, 1416), (2, 12, 19), (1359, 1409)),
    (4, (64, 64, 64), (740, 342), (2, 4, 2), (206, 210)),
    (4, (32, 32, 32), (744, 338), (2, 4, 1), (180, 94)),
    (4, (24, 290, 290), (776, 352), (2, 6, 15), (536, 275)),
    (4, (290, 24, 30), (729, 337), (2, 4, 2), (208, 196)),
    (4, (100, 100, 100), (760, 388), (2, 4, 5), (279, 131)),
    (4, (128, 128, 128), (800, 408), (2, 6, 9), (432, 212)),
    (4, (150, 150, 150), (782, 360), (2, 6, 12), (471, 261)),
    (4, (180, 97, 77), (768, 399), (2, 4, 8), (355, 164)),
    (4, (48, 170, 290), (768, 400), (2, 6, 9), (416, 210)),
    (4, (220, 61, 133), (778, 398), (2, 4, 9), (371, 173)),
    (4, (170, 170, 170), (790, 391), (2, 6, 22), (671, 376)),
    (4, (90, 180, 270), (787, 338), (2, 6, 16), (550, 317)),
    (4, (250, 130, 60), (779, 409), (2, 4, 10), (405, 191)),
    (4, (300, 300, 100), (1159, 563), (2, 12, 17), (831, 518)),
    (4, (130, 60, 250), (768, 404), (2, 6, 8), (389, 197)),
    (4, (80, 80, 80), (749, 358), (2, 4, 4), (246, 114)),
    (4, (170, 40, 90), (754, 366), (2, 4, 4), (251, 118)),
    (4, (290, 290, 40), (777, 354), (2, 8, 10), (490, 265)),
    (8, (512, 512, 512), (28770, 19671), (2, 4, 128), (19910, 19829)),
    (8, (640, 480, 200), (11784, 9241), (2, 4, 100), (9585, 9223)),
]


def test_radius_two_is_no_slower_than_one_round(pick):
    got = pick([f"radius_two {x} {y} {z} {es}" for es, (x, y, z), *_ in RADIUS_TWO])
    for (es, n, one, shape, times), picked in zip(RADIUS_TWO, got):
        assert picked == shape, (es, n)
        # 1%: two runs of one shape differ by as much
        assert times[0] <= 1.01 * one[0] and times[1] <= 1.01 * one[1], (es, n)


# batches of equal instances: number, side, radius, us per launch of four steps
# by item height
BATCHES = [
    (64, 256, 1, {8: 12.05, 10: 12.16, 13: 12.46, 16: 11.91, 24: 13.12, 26: 12.39, 32: 14.05,
                  64: 15.44, 128: 25.78}),
    (4, 1024, 2, {21: 15.58, 23: 16.26, 24: 16.69, 32: 18.45, 43: 16.29, 45: 15.66, 64: 18.78,
                  128: 30.59}),
    (1000, 128, 2, {24: 57.38, 32: 51.05, 64: 44.86, 86: 44.95, 96: 43.46, 128: 45.33}),
    (1, 512, 2, {4: 5.43, 6: 5.90, 8: 6.24, 16: 8.47, 32: 11.22, 64: 16.69}),
]


def test_batch_heights_split_the_sides(pick):
    got = pick([f"batch {n} " + f"{side} {side} {r} " * n for n, side, r, _ in BATCHES])
    for (n, side, r, us), (rows,) in zip(BATCHES, got):
        assert rows in {-(-side // m) for m in range(1, side)}, (n, side)
        assert us[rows] <= 1.05 * min(us.values()), (n, side)
    # sides of no listed height, and sides below the least height
    (a,), (b,) = pick(["batch 3 100 300 2 220 220 1 150 100 2", "batch 2 8 3 2 6 3 1"])
    assert any(a in {-(-y // m) for m in range(1, y)} for y in (300, 220, 100)) and b == 4


def test_batch_cost_is_that_of_the_lists(pick):
    # mixed sides, one instance that is split, two instances, one
    rng = random.Random(3)
    batches = [[(2 * rng.randrange(2, 260), rng.randrange(3, 520), rng.randrange(1, 3))
                for _ in range(n)] for n in (120, 40, 2, 1)]
    batches.append([(2048, 1500, 2)] + [(128, 128, 1)] * 30)
    lines = [f"launch_cost {k} {rows} {len(b)} " + " ".join(f"{x} {y} {r}" for x, y, r in b)
             for b in batches for k in (1, 2, 3, 4) for rows in (4, 17, 64, 103, 512)]
    assert all(by_count == by_list for by_count, by_list in pick(lines))
