"""Launch arithmetic shared by the kernels that stride over their grid (CPU)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("launch") / "launch_driver")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "its_amd", "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "launch_driver.cpp")], check=True)
    return exe


def test_strided_blocks_stay_below_the_limit(driver):
    """A launch dimension holds fewer than 2^32 work items, whatever the number
    of items; below that there is a block for each share."""
    cases = [(n, per, threads) for n in (0, 1, 15, 16, 17, 1 << 20, (1 << 29) + 5, (1 << 30) - 16, 1 << 30,
                                         (1 << 32) - 1, 1 << 32, 27 << 28, 1 << 36)
             for per, threads in ((16, 64), (64, 512), (256, 256))]
    out = subprocess.run([driver] + [str(v) for c in cases for v in c], check=True, capture_output=True, text=True)
    for (n, per, threads), blocks in zip(cases, map(int, out.stdout.split())):
        want = max(1, -(-n // per))
        assert blocks >= 1 and blocks * threads < 1 << 32, (n, per, threads)
        assert blocks == want if want * threads < 1 << 32 else (blocks + 1) * threads >= 1 << 32, (n, per, threads)
