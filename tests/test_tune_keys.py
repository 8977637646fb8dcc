"""The autotune cache's keys (lbm_amd/csrc/tune_cache.h): shape classes, and a
generation that keeps choices made among other kernels from being hits; entries
of calls too short to time every variant answer only such calls."""
import json
import os
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(__file__), "cpp")


@pytest.fixture(scope="module")
def tool(tmp_path_factory):
    exe = tmp_path_factory.mktemp("keys") / "tune_key_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", os.path.join(CPP, "tune_key_check.cpp"),
                    "-o", str(exe)], check=True, timeout=120)

    def run(*args):
        return subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, check=True,
                              timeout=60).stdout.strip()
    return run


def test_keys_hold_class_and_generation(tool):
    assert tool("grid", "gfx950:x/256cu", 300, 160, "f32", "ref", 10) == "gfx950:x/256cu/grid/512x256/f32/ref/v10/g2"
    assert tool("grid", "a b", 4096, 4097, "f16e", "zg", 10) == "a_b/grid/4096x8192/f16e/zg/v10/g2"
    assert tool("batch", "gfx950/256cu", 3, 100000, "f32", "ref", 8) == "gfx950/256cu/batch/4d/1Mcells/f32/ref/v8/g2"
    assert tool("batch", "d", 512, 3 << 20, "f16s", "zg", 8) == "d/batch/512d/4Mcells/f16s/zg/v8/g2"
    assert tool("batch", "d", 1, (1 << 20) + 1, "f32", "ref", 8) == "d/batch/1d/2Mcells/f32/ref/v8/g2"
    assert tool("batch", "d", 1, 1 << 60, "f32", "ref", 8) == "d/batch/1d/1073741824Mcells/f32/ref/v8/g2"


@pytest.mark.parametrize("variant,entry_steps,steps,want", [
    (0, 20, 20, 1), (9, 3, 100, 1), (9, 20, 2, 1), (3, 2, 2, 1), (3, 1, 2, 1),
    (3, 2, 3, 0), (3, 1, 20, 0), (10, 20, 20, 0), (-1, 20, 20, 0)])
def test_which_entries_answer(tool, variant, entry_steps, steps, want):
    assert tool("answers", variant, entry_steps, steps, 3, 10) == str(want)


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [False, True])
def test_stale_and_short_entries_are_misses(tmp_path, batch):
    """A file of another generation is tuned anew; a two-step call's entry answers
    two-step calls, which keep the default path, and is replaced by a longer call's."""
    from lbm_amd import LBM, Batch
    print(f"case: stale and short cache entries, batch {batch}", flush=True)

    def make():
        return Batch([(400, 160, 1.6, 0.05), (96, 64, 1.5, 0.04)]) if batch else LBM(1.6, 400, 160)
    path = tmp_path / "tune.json"
    a = make()
    assert not a.autotune_cached(str(path), 6)[1]
    a.close()
    (key, entry), = json.loads(path.read_text()).items()
    path.write_text(json.dumps({key[:key.rindex("/g")]: dict(entry, variant=0)}))  # as before generations
    a = make()
    assert not a.autotune_cached(str(path), 6)[1]
    a.close()
    path.unlink()
    a, b = make(), make()
    untuned = a.launches(60)
    best, hit = a.autotune_cached(str(path), 2)
    assert not hit and a.launches(60) == untuned < 60
    assert b.autotune_cached(str(path), 2) == (best, True)
    assert b.launches(60) == untuned and b.variant == best
    best, hit = b.autotune_cached(str(path), 6)
    assert not hit and json.loads(path.read_text())[key]["steps"] == 6
    assert a.autotune_cached(str(path), 2) == (best, True) and a.variant == best
    a.close()
    b.close()
