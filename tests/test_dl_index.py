"""The direct-LDS DGEMM kernels' index arithmetic on the CPU: the header that the
kernels include (cosma_amd/csrc/dl_index.hpp) compiled for the host."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("dl_index") / "dl_index_test")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(ROOT, "cosma_amd", "csrc"),
                    "-o", out, os.path.join(ROOT, "tests", "cpp", "dl_index_test.cpp")], check=True)
    return out


def run(exe, what):
    r = subprocess.run([exe, what], capture_output=True, text=True, timeout=300)
    bad = [line for line in r.stdout.splitlines() if line.startswith("FAIL")]
    assert r.returncode == 0 and not bad, (r.returncode, bad[:10], r.stderr[-2000:])
    return r.stdout


def test_every_group_m_walks_every_tile_once(exe):
    """cosma_amd_dgemm_set_tuning takes any group_m >= 0; the kernel's 32-bit walk is right for all of them."""
    assert run(exe, "raster").count("ok raster") == 8 * 14


def test_loads_end_inside_the_operand(exe):
    """For odd and even extents, every k up to three steps and the tightest leading dimension, as A and as B; the
    over-read that the steps would make of an odd row-contiguous operand without holding back its last k is seen."""
    out = run(exe, "loads")
    assert [out.count(s) for s in ("ok loads inside", "ok loads complete", "ok over-read seen")] == [10, 10, 10]
