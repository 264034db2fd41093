"""The engine's host rules (tmc_amd/csrc/dmc_plan.h), compiled for the CPU."""
import itertools
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "plan_probe")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "plan_probe.cpp")], check=True)

    def run(*args):
        return subprocess.run([exe, *map(str, args)], capture_output=True, text=True, check=True).stdout.strip()
    return run


# axes up to 2^24 points: shapes whose axes ran into each other when they were
# packed into 21 bits each, and batches that differ in the order of their axes
SHAPES = [(2, 2, 10485759), (2, 6, 2097151), (6, 2, 2097151), (2, 2097154, 2), (3, 2, 2), (2, 3, 2), (2, 2, 3),
          (2, 2, 1 << 24), (2, 10, 2), (4, 1 << 21, 2), (5, 2, 2), (2, 2, 2, 3, 3, 3), (3, 3, 3, 2, 2, 2),
          (2, 2, 2, 3, 3, 3, 2, 2, 2)]


def test_shapes_have_keys_of_their_own(probe):
    keys = {s: probe("key", *s) for s in SHAPES}
    for a, b in itertools.combinations(SHAPES, 2):
        assert keys[a] != keys[b], (a, b)
    assert probe("key", 2, 2, 3) == keys[(2, 2, 3)]


@pytest.mark.parametrize("volumes,shift", [
    # one volume: the limits of the group sizes
    ([(1, 1)], 0), ([(1, 8191)], 0), ([(1, 8192)], 2), ([(1, 65535)], 2), ([(1, 65536)], 4),
    # many small ones: whole groups of 16, 8, 4, 2 and 1 within an eighth
    ([(8000, 30)], 4), ([(10000, 8)], 3), ([(10000, 25)], 2), ([(8000, 9)], 1), ([(70000, 1)], 0),
    # a large one among them carries their padding
    ([(100, 1), (1, 65536)], 4), ([(1000, 1), (1, 65536)], 3)])
def test_groups_pad_little(probe, volumes, shift):
    total = sum(n * rs for n, rs in volumes)
    got, padded = map(int, probe("groups", *itertools.chain(*volumes)).split())
    assert got == shift
    assert total <= padded <= total + total // 8


@pytest.mark.parametrize("args,blocks", [
    ((0, 256, 0, 32768), 1), ((256, 256, 0, 32768), 1), ((257, 256, 0, 32768), 2), ((1 << 30, 256, 0, 32768), 32768),
    # a kernel's own limit never lifts the caller's cap
    ((1 << 30, 256, 4096, 32768), 4096), ((1 << 30, 256, 4096, 64), 64), ((1000, 256, 4096, 64), 4)])
def test_blocks_of_a_launch(probe, args, blocks):
    assert int(probe("blocks", *args)) == blocks
