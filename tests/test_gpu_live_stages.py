"""Simplifications on the live mesh against the same stages run one by one with
a compaction and a generic halfedge build each (an engine created with
TMC_GENERIC_ROWS=1): every flag combination, on smooth, noisy and two-valued
fields (regular merges, irregular ones, 3-face and non-manifold edges), with
few blocks (a block's face list fills and is flushed many times) and with many
(most blocks have no face), alone and in a batch (per-volume counts)."""
import os

import numpy as np
import pytest

from meshcheck import assert_same

pytestmark = pytest.mark.gpu

import tmc_amd  # noqa: E402
from tmc_amd import (SIMPLIFY_3333, SIMPLIFY_3X3Y_COLOR, SIMPLIFY_3X3Y_ISOLATED, SIMPLIFY_ALL,  # noqa: E402
                     TRIANGLES, workloads)

KEYS = ("v", "n", "quads", "tris", "he", "he_v", "bnd")
FLAGS = [SIMPLIFY_3X3Y_COLOR, SIMPLIFY_3X3Y_ISOLATED, SIMPLIFY_3333, SIMPLIFY_3X3Y_COLOR | SIMPLIFY_3333,
         SIMPLIFY_3X3Y_COLOR | SIMPLIFY_3X3Y_ISOLATED, SIMPLIFY_ALL]


@pytest.fixture(scope="module")
def engines():
    os.environ["TMC_GENERIC_ROWS"] = "1"
    try:
        staged = tmc_amd.Engine(0)
    finally:
        del os.environ["TMC_GENERIC_ROWS"]
    live = tmc_amd.Engine(0)
    yield live, staged
    live.close()
    staged.close()


def _two_valued(shape, seed):
    """Thick random blocks: many valence-3 corners, pinched edges."""
    rng = np.random.default_rng(seed)
    f = rng.random([(n + 1) // 2 for n in shape]) < 0.45
    f = f.repeat(2, 0).repeat(2, 1).repeat(2, 2)[:shape[0], :shape[1], :shape[2]]
    return f.astype(np.float32), tmc_amd.Grid.make(shape), 0.5


FIELDS = {"schwarz_100": lambda: workloads.schwarz((100, 97, 103), seed=8),
          "blobs_80": lambda: workloads.blobs((80, 72, 76), seed=3),
          "genus2_64": lambda: workloads.genus2(64),
          "two_valued": lambda: _two_valued((31, 40, 37), 5),
          "tiny": lambda: _two_valued((5, 4, 6), 2)}


@pytest.mark.parametrize("name", FIELDS)
def test_live_stages_match_staged_pass(engines, name):
    live, staged = engines
    f, g, iso = FIELDS[name]()
    usual = live.launch
    try:
        for flags in FLAGS:
            m = staged.extract(f, iso, g, flags=flags | TRIANGLES)
            exp, esum = staged.download(), m.summary()
            for cap in (64, 32768):
                print(f"[gpu] live stages {name} flags {flags} blocks {cap}", flush=True)
                live.launch = {"grid_cap": cap}
                m = live.extract(f, iso, g, flags=flags | TRIANGLES)
                got = live.download()
                for k in KEYS:
                    assert_same(got[k], exp[k], f"{name} flags {flags} blocks {cap}: {k}")
                assert m.summary() == esum
    finally:
        live.launch = usual


def test_live_stages_in_a_batch(engines):
    live, staged = engines
    vols = [(f, iso, g) for f, g, iso in (make() for make in FIELDS.values())]
    print("[gpu] live stages in a batch", flush=True)
    sums = [[m.summary() for m in e.extract_batch(vols, flags=SIMPLIFY_ALL | TRIANGLES)] for e in engines]
    for i in range(len(vols)):
        got, exp = live.download_batch(i), staged.download_batch(i)
        for k in KEYS:
            assert_same(got[k], exp[k], f"volume {i}: {k}")
        assert sums[0][i] == sums[1][i], f"volume {i}"
