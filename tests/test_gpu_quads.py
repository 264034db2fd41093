"""Quadrilaterals with their halfedges straight from the cells, against the
oracle bit for bit: rows that end at, before and after a segment's end (a
neighbour cell in the next segment), grids of one cell layer, blocks of the
kernel that end inside, and fields whose faces have three and four halfedges
on a vertex pair; with and without the simplifications (boundary arrivals),
alone and in a batch (per-volume counts)."""
import numpy as np
import pytest

from meshcheck import assert_same

pytestmark = pytest.mark.gpu

import tmc_amd  # noqa: E402
from tmc_amd import SIMPLIFY_ALL, TRIANGLES  # noqa: E402

SHAPES = [(4, 4, 256), (4, 5, 257), (5, 4, 258), (4, 4, 513), (3, 3, 3), (2, 9, 9), (9, 2, 9), (9, 9, 2), (13, 12, 11)]
KEYS = ("v", "n", "quads", "he", "he_v", "bnd")


def _field(shape, kind):
    rng = np.random.default_rng(shape[0] * 1000 + shape[1] * 100 + shape[2] + kind)
    if kind == 0:
        return rng.standard_normal(shape).astype(np.float32), 0.1      # every face configuration
    if kind == 1:
        return rng.integers(-1, 2, shape).astype(np.float64), 0.0      # ties
    f = rng.standard_normal(shape)
    return np.round(f * 2) / 2 + 0.05, 0.0


def _oracle(oracle, f, iso, g, flags):
    s = np.asarray(f, np.float64).ravel()
    return oracle.dualmc(g, s, oracle.gradient(g, s), iso, flags=flags | 8)


@pytest.mark.parametrize("flags", [0, SIMPLIFY_ALL], ids=["plain", "simplified"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_quads_match_oracle(engine, oracle, shape, flags):
    g = tmc_amd.Grid.make(shape, (0.1, 0.2, 0.3), (0.5, 0.25, 0.75))
    for kind in range(3):
        f, iso = _field(shape, kind)
        print(f"[gpu] quads {shape} field {kind} flags {flags}", flush=True)
        exp = _oracle(oracle, f, iso, g, flags)
        m = engine.extract(f, iso, g, flags=flags | TRIANGLES)
        got = engine.download()
        for k in KEYS:
            assert_same(got[k], exp[k], f"{shape} field {kind}: {k}")
        assert m.nonmanifold_edges == exp["nonmanifold"]


@pytest.mark.parametrize("flags", [0, SIMPLIFY_ALL], ids=["plain", "simplified"])
def test_quads_in_a_batch(engine, flags):
    vols = [(np.asarray(_field(s, i % 2)[0], np.float32), 0.1, None) for i, s in enumerate(SHAPES)]
    ms = engine.extract_batch(vols, flags=flags | TRIANGLES)
    sums = [m.summary() for m in ms]
    got = [engine.download_batch(i) for i in range(len(vols))]
    for i, (f, iso, _) in enumerate(vols):
        print(f"[gpu] batch volume {i} {f.shape} flags {flags}", flush=True)
        m = engine.extract(f, iso, flags=flags | TRIANGLES)
        exp = engine.download()
        for k in KEYS:
            assert_same(got[i][k], exp[k], f"volume {i}: {k}")
        for k in ("nv", "nq", "nonmanifold_edges", "edge_errors", "nbnd", "nv_cells", "nq_cells"):
            assert sums[i][k] == getattr(m, k), f"volume {i}: {k}"
