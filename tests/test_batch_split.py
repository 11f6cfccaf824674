"""The rule that splits a batch between the one-launch fit and the many-mesh
solver (its_amd/csrc/batch_split.hpp), on the CPU."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "its_amd", "csrc")
# octrees of one many-mesh solve: 12 bits of a block table entry
MOST = (1 << int(re.search(r"kMeshBits = (\d+)", open(os.path.join(CSRC, "lscg_batch.hpp")).read())[1])) - 1


@pytest.fixture(scope="module")
def split(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("split") / "batch_split_driver")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, "-o", exe,
                    os.path.join(ROOT, "tests", "batch_split_driver.cpp")], check=True)

    def run(cand, big=(), most=MOST):
        args = [most, len(big)] + [v for m in list(big) + list(cand) for v in m]
        return int(subprocess.run([exe] + [str(v) for v in args], check=True, capture_output=True, text=True).stdout)

    return run


@pytest.mark.parametrize("count", [1, 4095, 4096, 5000, 6000, 12000])
@pytest.mark.parametrize("mesh", [(160, 3), (14110, 7)])
@pytest.mark.parametrize("big", [0, 5])
def test_split_fits_the_many_mesh_solver(split, count, mesh, big):
    """However many meshes there are, no more go to the many-mesh solver than
    it takes."""
    one = split([mesh] * count, [(100_000, 8)] * big)
    assert 0 <= one <= count
    assert count - one + big <= MOST


def test_split_of_too_many_large_meshes(split):
    """With the many-mesh solver full already, none is added."""
    assert split([(160, 3)] * 7, [(100_000, 8)] * 40, most=40) == 7
    assert split([(160, 3)] * 7, [(100_000, 8)] * 41, most=40) == 7
    assert split([(160, 3), (60_000, 7)], [(100_000, 8)] * 39, most=40) == 1


def test_split_moves_what_holds_the_launch_up(split):
    """6 meshes of 7,165 to 55,852 unknowns: the largest would take 6 ms on its
    workgroup, the many-mesh solver's launches about 2; the small ones stay."""
    assert split([(7165, 6), (14110, 7), (20000, 7), (31101, 7), (40000, 7), (55852, 7)]) == 2
    assert split([(160, 3), (3668, 5)]) == 2
    assert split([(56062, 7)] * 2) == 0 and split([(14176, 6)] * 4) == 0
    assert split([(56062, 7)] * 128) == 0   # beside each other both slow down


@pytest.mark.parametrize("mesh", [(160, 3), (854, 4), (3694, 5), (14110, 7)])
@pytest.mark.parametrize("count", [256, 600, 1000, 2000])
def test_split_leaves_a_full_chip_alone(split, mesh, count):
    """Where the one launch has a workgroup for every CU, nothing runs beside it:
    many meshes of one small size stay together (moving 88 of 600 meshes of 854
    unknowns doubled the fit's time)."""
    assert split([mesh] * count) == count
