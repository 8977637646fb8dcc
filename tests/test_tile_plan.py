"""How a call of n steps is cut into launches (lbm_amd/csrc/tile_plan.h), host
code only: the launches' steps are of allowed lengths and add up to n for every
short call and for the longest a 32-bit count can ask for.  No reference
counterpart."""
import os
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(__file__), "cpp")


@pytest.fixture(scope="module")
def tool(tmp_path_factory):
    exe = tmp_path_factory.mktemp("plan") / "tile_plan_check"
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", "-Wextra", "-Werror", os.path.join(CPP, "tile_plan_check.cpp"),
                    "-o", str(exe)], check=True, timeout=120)

    def run(*args):
        return subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=60)
    return run


@pytest.mark.parametrize("nx,ny", [(3, 3), (400, 160), (1021, 777), (8192, 4096)])
def test_every_short_call(tool, nx, ny):
    r = tool(nx, ny, *range(1, 400))
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout[-300:]


@pytest.mark.parametrize("nx,ny", [(64, 16), (8192, 4096)])
@pytest.mark.parametrize("back", range(1, 12))
def test_the_longest_calls(tool, nx, ny, back):
    r = tool(nx, ny, 2 ** 32 - back)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), (r.returncode, r.stdout[-300:])
