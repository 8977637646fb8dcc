"""Large host copies (lbm_amd/csrc/staging.h) on the CPU, over a stand-in for the
runtime whose copies run as late as they may: every byte of every piece, chunks
reused many times and by a second call, partial last chunks, calls in which a
thread cannot be made or a copy fails.  No reference counterpart."""
import os
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(__file__), "cpp")
MB = 1 << 20


@pytest.fixture(scope="module")
def tool(tmp_path_factory):
    exe = tmp_path_factory.mktemp("staging") / "staging_check"
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", "-Wextra", "-Werror", "-pthread", "-I",
                    os.path.join(CPP, "host_hip"), os.path.join(CPP, "staging_check.cpp"), "-o", str(exe)],
                   check=True, timeout=120)

    def run(*args):
        r = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=60)
        return r.returncode, r.stdout.strip()
    return run


def counts(sizes, calls=1):
    """What the calls of these pieces launch: one kernel a chunk, no copy of the runtime's."""
    return f"chunks=1 copies=0 launches={calls * sum((n + MB - 1) // MB for n in sizes)}"


@pytest.mark.parametrize("way,sizes,chunked", [
    ("out", [4 * MB - 1], False), ("out", [4 * MB], True), ("out", [20 * MB + 1, 3, MB], True),
    ("in", [8 * MB - 1], False), ("in", [8 * MB], True), ("in", [3 * MB - 5, 6 * MB + 7, 17], True),
    ("in", [33 * MB + 4093], True), ("out", [1] * 7 + [41 * MB - 9], True)])
def test_every_byte_arrives(tool, way, sizes, chunked):
    want = counts(sizes, 2) if chunked else f"chunks=0 copies={2 * len(sizes)} launches=0"
    assert tool("copy", way, *sizes) == (0, "ok " + want)


@pytest.mark.parametrize("way", ["out", "in"])
def test_unaligned_device_memory(tool, way):
    """The kernel takes 4-byte aligned addresses; the runtime copies the other chunks."""
    assert tool("odd", way, 13 * MB + 11) == (0, "ok chunks=1 copies=14 launches=0")


@pytest.mark.parametrize("way", ["out", "in"])
def test_pinned_memory_goes_straight(tool, way):
    """The runtime copies a caller's pinned buffer itself: no chunks, no error left behind."""
    assert tool("pinned", way, 13 * MB + 11) == (0, "ok chunks=0 copies=1 launches=0")


@pytest.mark.parametrize("way", ["out", "in"])
@pytest.mark.parametrize("nth", [0, 1, 2])
def test_a_thread_that_cannot_be_made(tool, way, nth):
    """Its share is copied by the calling thread; the process goes on."""
    assert tool("nothread", way, 13 * MB + 11, nth) == (0, "ok " + counts([13 * MB + 11], 2))


@pytest.mark.parametrize("way", ["out", "in"])
@pytest.mark.parametrize("nth", [0, 5, 18])
def test_a_failed_launch_is_reported_and_the_next_call_is_whole(tool, way, nth):
    rc, text = tool("error", way, 20 * MB + 1, nth)
    assert rc == 0 and text.startswith("ok chunks=1 copies=0 ")
