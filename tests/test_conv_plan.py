"""The boxes that the convolutions run on (conv_plan in mf-lbm-cuda_amd/csrc/conv_plan.h), on the
CPU: large grids have one, it covers the grid and fits LDS, and a block's box coordinates are exact
at every index."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "mf-lbm-cuda_amd", "csrc")


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("conv_plan") / "conv_plan_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-D__host__=", "-D__device__=", "-D__forceinline__=inline", "-I" + CSRC,
                    os.path.join(HERE, "conv_plan_check.cpp"), "-o", out], check=True, timeout=120)
    return out


def plan(harness, *args):
    r = subprocess.run([harness, *map(str, args)], timeout=60, capture_output=True, text=True)
    return r.returncode, r.stdout.strip()


@pytest.mark.parametrize("shape,cin,cout", [
    ((256, 256, 256), 48, 16), ((256, 256, 256), 16, 48), ((256, 256, 256), 96, 32), ((256, 256, 256), 192, 64),
    ((192, 192, 192), 192, 64), ((192, 192, 192), 128, 128), ((320, 320, 320), 32, 32), ((512, 512, 512), 16, 16),
    ((800, 1000, 900), 8, 16), ((3, 5, 10000000), 8, 8), ((7, 30000000, 1), 8, 8), ((20000000, 3, 5), 8, 8),
    ((1, 1, 1), 8, 8), ((33, 34, 35), 16, 48), ((64, 64, 64), 48, 16),
    ((128, 128, 128), 320, 64), ((128, 128, 128), 320, 160), ((96, 96, 96), 384, 64), ((64, 64, 64), 448, 192),
    ((32, 32, 32), 576, 64), ((20, 20, 20), 560, 128), ((8, 8, 8), 1056, 128)])
def test_grids_have_a_box(harness, shape, cin, cout):
    rc, box = plan(harness, *shape, cin, cout)
    assert rc == 0, box


@pytest.mark.parametrize("shape,cin,cout", [((32, 32, 32), 800, 64), ((24, 24, 24), 720, 64), ((64, 64, 64), 600, 128), ((12, 12, 12), 1056, 128), ((3, 2, 5), 1104, 8)])
def test_deep_inputs_are_left_to_the_gathering_kernel(harness, shape, cin, cout):
    assert plan(harness, *shape, cin, cout)[0] == 1


def test_planes_beyond_a_descriptor_have_none(harness):
    """2 GiB and more a plane: the gathering kernel's"""
    assert plan(harness, 2, 8192, 8192, 16, 16)[0] == 1
    assert plan(harness, 2, 8192, 8192, 8, 16)[0] == 0


def test_kept_plans(harness):
    """a size is searched for once while it keeps its place, and gets the plan of a search"""
    assert subprocess.run([harness, "kept"], timeout=60).returncode == 0
