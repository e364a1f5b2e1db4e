"""The launch-shape rules (symphas_amd/csrc/shape.hpp), compiled for the host,
against times measured on an MI355X: what a rule picks is no slower than what it
passes over."""
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
