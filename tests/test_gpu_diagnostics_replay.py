"""Mesh diagnostics after replayed passes on the GPU, with and without
simplifications: the halfedge rows that they read are made for the mesh at hand,
whatever the passes before left."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import tmc_amd  # noqa: E402
from tmc_amd import SIMPLIFY_ALL, TRIANGLES, workloads  # noqa: E402


def test_diagnostics_after_replays():
    from oracle import diagnostics as D
    f, g, iso = workloads.blobs((24, 30, 27), seed=6)
    eng = tmc_amd.Engine(0)
    try:
        for flags in (TRIANGLES, SIMPLIFY_ALL | TRIANGLES, TRIANGLES):
            for i in range(8):
                m = eng.extract(f, iso, g, flags=flags)
            print(f"[gpu] diagnostics, flags {flags}, pass mode {m.pass_mode}", flush=True)
            assert m.pass_mode == 2
            d = eng.download(halfedges=False)
            for _ in range(2):
                assert np.array_equal(eng.edges(), D.mesh_edges(d["quads"]))
                h, beyond = eng.valence_histogram()
                eh, eb = D.valence_histogram(len(d["v"]), d["quads"])
                assert np.array_equal(h, eh) and beyond == eb
    finally:
        eng.close()
