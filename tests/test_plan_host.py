"""The pipelined GEMMs' plan and tile numbering (mlx-runner_amd/csrc/gemm_plan.h), on the host: the calls
that the GPU tests run reach the tiles they name, and the blocks of a call cover its tiles."""
import shutil
import subprocess
from pathlib import Path

import pytest

import gemm_shapes as G

HERE = Path(__file__).resolve().parent
KINDS = {"dense": G.DENSE, "nvfp4": G.NVFP4, "mxfp8": G.MXFP8, "nvfp4-mlp": G.NVFP4_MLP, "mxfp8-mlp": G.MXFP8_MLP}


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not found")
    out = tmp_path_factory.mktemp("plan") / "plan"
    subprocess.run([gxx, "-std=c++17", "-O1", "-I", str(HERE.parent / "mlx-runner_amd/csrc"),
                    str(HERE / "host_plan/plan.cpp"), "-o", str(out)], check=True, timeout=300)
    return out


@pytest.mark.parametrize("kind", list(KINDS))
def test_listed_calls_reach_their_tiles(driver, kind):
    lines = "".join("%s %d %d %d\n" % (kind, M, N, K) for M, N, K, _, _ in KINDS[kind])
    r = subprocess.run([str(driver)], input=lines, text=True, capture_output=True, check=True, timeout=60)
    got = list(zip([(M, N, K) for M, N, K, _, _ in KINDS[kind]], r.stdout.splitlines()))
    assert got == [((M, N, K), ("%s %s" % (t, s)).strip()) for M, N, K, t, s in KINDS[kind]]


def test_blocks_cover_every_tile(driver):
    r = subprocess.run([str(driver), "numbering"], text=True, capture_output=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
