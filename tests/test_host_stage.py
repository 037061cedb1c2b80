"""Staged transfers to the host where memory is refused, on the CPU: the transfer code is compiled against a
runtime of the test's own (host_stage.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SOURCE = os.path.join(HERE, "..", "mithra_amd", "csrc", "gpu")
OK, NOMEM = 0, -4


@pytest.fixture(scope="module")
def lines(tmp_path_factory):
    d = tmp_path_factory.mktemp("stage")
    (d / "hip").mkdir()
    shutil.copy(os.path.join(HERE, "hip_host_stub.h"), d / "hip" / "hip_runtime.h")
    exe = str(d / "stage")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-I", str(d), "-I", SOURCE,
                    os.path.join(HERE, "host_stage.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=120).stdout
    return [(w[0], *map(int, w[1:])) for w in (line.split() for line in out.splitlines())]


def of(lines, name):
    return [line[1:] for line in lines if line[0] == name]


SIZES = [0, 1, 744, 745, 5957, 5958, 100001]


@pytest.mark.parametrize("name", ["first", "pinned", "refused", "little", "granted", "full"])
def test_transfer_comes_through(lines, name):
    """With pinned memory, without any, with a device that grants 50 kB at most, with pinned memory granted
    again after a refusal, whose error no later launch may report, and with pinned memory alone."""
    assert sorted({line[0] for line in of(lines, name)}) == SIZES
    for n, status, good, *_ in of(lines, name):
        assert (status, good) == (OK, 1), (name, n)


def test_nothing_granted(lines):
    for n, status, good, puts, *held in of(lines, "none"):
        assert (status, puts, held) == (OK if n == 0 else NOMEM, 0, [0, 0])


def test_failing_chunk_ends_the_transfer(lines):
    for n, status, good, puts, *_ in of(lines, "failing"):
        assert (status != OK, puts) == ((n > 0), min(n, 1))


def test_memory_is_bounded_and_given_back(lines):
    for _, _, _, _, *held in of(lines, "left"):
        assert held == [0, 0]
    for name, most in (("refused", 512 << 10), ("little", 50000)):
        for *_, pinned, device in of(lines, name):
            assert pinned == 0 and device <= most
    assert max(line[4] for line in of(lines, "pinned")) <= 4 << 20


def test_a_first_small_transfer_pins_nothing(lines):
    """744 records are 64 kB: as many as an owner's first transfer takes without pinned memory."""
    assert [line[4] > 0 for line in of(lines, "first")] == [n > 744 for n in SIZES]
    assert [line[4] > 0 for line in of(lines, "pinned")] == [n > 0 for n in SIZES]


def test_no_more_chunks_than_asked(lines):
    for n, status, good, puts, *_ in of(lines, "three"):
        assert (status, good) == (OK, 1) and puts <= 3
