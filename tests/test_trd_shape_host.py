"""The tridiagonalisation's launch shape (dft-zig_amd/csrc/trd_shape.h, host arithmetic, built with g++):
on a whole MI355X (256 CUs) and its partitions of 128, 64 and 32 CUs every size up to 1,024, 1,024, 704
and 512 rows has an instance that holds it, with all its workgroups resident at once."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = tmp_path_factory.mktemp("trd") / "trd_shape_driver"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", str(ROOT / "dft-zig_amd" / "csrc"),
                    str(ROOT / "tests" / "trd_shape_driver.cpp"), "-o", str(exe)], check=True, capture_output=True)
    return lambda cases: [tuple(map(int, l.split())) for l in subprocess.run(
        [str(exe)], input="\n".join("%d %d %d" % c for c in cases), capture_output=True, text=True, check=True).stdout.splitlines()]


@pytest.mark.parametrize("cus,most", [(256, 1024), (128, 1024), (64, 704), (32, 512)])
@pytest.mark.parametrize("cols", [0, 4, 8, 16])
def test_every_size_has_an_instance(driver, cus, most, cols):
    cases = [(m, cus, cols) for m in range(1, most + 1)]
    for (m, _, _), (nq, cw, groups) in zip(cases, driver(cases)):
        assert 0 < m <= 64 * nq and groups <= cus and (groups - 1) * 4 * cw < m <= groups * 4 * cw, (m, nq, cw, groups)
        assert 4 * cw >= cols or m > 704  # no instance of four columns a wavefront there


def test_one_column_a_wavefront_on_the_whole_device(driver):
    assert all(cw == 1 for _, cw, _ in driver([(m, 256, 0) for m in range(1, 1025)]))
    assert driver([(513, 32, 0), (1025, 256, 0)]) == [(0, 0, 0), (0, 0, 0)]
