"""Passes that the live mesh cannot express, on the GPU.

In a slab one cell thick two merging faces can meet at a vertex without sharing
an edge that pairs them, so that one removes the vertex that the other merges
into: its new name then depends on the numbering after a compaction, and the
pass is run again stage by stage.  Small slabs that do so (noise in steps of a
half, cut out of large ones) against the oracle, the staged engine, themselves in
a batch and through the no-alloc call; and the usual fields of the live stages,
which must not take this way."""
import os

import numpy as np
import pytest

from meshcheck import assert_same
from test_gpu_live_stages import FIELDS

pytestmark = pytest.mark.gpu

import tmc_amd  # noqa: E402
from tmc_amd import SIMPLIFY_3X3Y_ISOLATED, SIMPLIFY_ALL, STAGE_TIMING, TRIANGLES, workloads  # noqa: E402

KEYS = ("v", "n", "quads", "tris", "he", "he_v", "bnd")
SLABS = {
    "6x6": [[[2, -1, 3, -2, 1, -1], [0, 0, -1, 1, 4, 0], [4, -1, -1, 2, 0, -3], [0, 1, -1, 1, 0, -1],
             [-2, -2, -4, -3, -1, -1], [0, 1, 0, 0, -1, 1]],
            [[-2, -2, 1, -1, 0, 2], [1, -1, -1, 0, 0, 0], [-1, 2, 2, -2, 4, -1], [-3, 0, -2, 0, -1, -3],
             [-1, -3, 1, 1, 1, 2], [0, -4, -1, -2, -1, 0]]],
    "6x8": [[[-2, 0, 2, 1, 0, 2, 2, -2], [1, 3, 5, 0, 1, -4, 4, -2], [-2, -1, -2, 0, -2, -1, 0, 4],
             [-1, 0, 1, 0, 1, 2, -1, 0], [2, -1, 0, 2, -3, 0, 0, 3], [0, -5, -3, -4, -2, 2, 3, 1]],
            [[4, 1, -2, 1, -1, 2, -1, 0], [-2, -1, 2, -2, 0, -3, 0, 0], [-2, 0, 4, 1, 1, -2, 0, -1],
             [-1, -2, -1, -1, 0, -2, 1, 0], [4, 1, -5, -2, 1, -3, -2, 3], [-1, 1, 2, -1, -2, -3, -1, 0]]]}
ISO = 0.1


def _slab(name, tiles=1):
    f = np.concatenate([np.array(SLABS[name], np.float32) / 2] * tiles, 1)
    return f, tmc_amd.Grid.make(f.shape), ISO


def _staged_engine():
    os.environ["TMC_GENERIC_ROWS"] = "1"
    try:
        return tmc_amd.Engine(0)
    finally:
        del os.environ["TMC_GENERIC_ROWS"]


def _ran_staged(eng, f, iso, g, flags):
    """Whether the extraction ended with the stage-by-stage pass (which pairs
    halfedges through rows) rather than on the live mesh."""
    eng.extract(f, iso, g, flags=flags | STAGE_TIMING)
    names = eng.stage_times()
    assert ("k_he_twins" in names) != ("k_stage_merge" in names), sorted(names)
    return "k_he_twins" in names


@pytest.mark.parametrize("name", SLABS)
def test_slab_is_run_stage_by_stage(oracle, name):
    f, g, iso = _slab(name)
    s = f.astype(np.float64).ravel()
    exp = oracle.dualmc(g, s, oracle.gradient(g, s), iso, True)
    eng, staged = tmc_amd.Engine(0), _staged_engine()
    try:
        for flags in (SIMPLIFY_ALL | TRIANGLES, SIMPLIFY_3X3Y_ISOLATED | TRIANGLES):
            print(f"[gpu] slab {name} flags {flags}", flush=True)
            em = staged.extract(f, iso, g, flags=flags)
            ed = staged.download()
            for i in range(8):   # the later passes are replayed
                m = eng.extract(f, iso, g, flags=flags)
                got = eng.download()
                for k in KEYS:
                    assert_same(got[k], ed[k], f"pass {i}: {k}")
                    if flags == SIMPLIFY_ALL | TRIANGLES and k != "tris":
                        assert_same(got[k], exp[k], f"pass {i}: {k}, oracle")
                assert m.summary() == em.summary()
                # the first pass runs twice, the next ones know the shape
                assert m.host_syncs == (2 if i == 0 else 1) + (m.nbnd > 0), f"pass {i}"
            assert m.pass_mode == 2
            assert _ran_staged(eng, f, iso, g, flags)
            # another field of the shape goes back to the live mesh
            z = np.linspace(-1, 1, f.size, dtype=np.float32).reshape(f.shape)
            eng.extract(z, iso, g, flags=flags)
            assert not _ran_staged(eng, z, iso, g, flags)
    finally:
        eng.close()
        staged.close()


def test_slabs_in_a_batch():
    """A member of a batch equals the volume alone, whatever comes before it.
    (Many slabs in a row remove enough vertices for ids of the old numbering
    that the mesh no longer has.)"""
    usual = [workloads.genus2(20), workloads.blobs((12, 14, 13), seed=2)]
    vols = [(f, iso, g) for f, g, iso in (usual[0], _slab("6x6"), usual[1], _slab("6x8"), _slab("6x6", 12),
                                           _slab("6x8", 40), _slab("6x6"))]
    eng = tmc_amd.Engine(0)
    try:
        for flags in (SIMPLIFY_ALL | TRIANGLES, SIMPLIFY_3X3Y_ISOLATED | TRIANGLES):
            print(f"[gpu] slabs in a batch, flags {flags}", flush=True)
            exp = []
            for f, iso, g in vols:
                m = eng.extract(f, iso, g, flags=flags)
                exp.append((m.summary(), eng.download()))
            if flags == SIMPLIFY_3X3Y_ISOLATED | TRIANGLES:
                assert any(d["quads"].max() >= len(d["v"]) for _, d in exp)
            for rep in range(3):
                ms = eng.extract_batch(vols, flags=flags)
                for i, (es, ed) in enumerate(exp):
                    got = eng.download_batch(i)
                    for k in KEYS:
                        assert_same(got[k], ed[k], f"flags {flags} pass {rep} volume {i}: {k}")
                    s = ms[i].summary()
                    assert all(s[k] == es[k] for k in s if k not in ("invalid_refs", "valence_zero")), (i, s, es)
    finally:
        eng.close()


def test_capacities_and_rerun_together():
    """A new context learns the cells' sizes, then the records', and that the
    pass has to be run stage by stage, within its three attempts."""
    flags = SIMPLIFY_ALL | TRIANGLES
    f = np.random.default_rng(8).standard_normal((3, 3, 100000)).astype(np.float32)
    vols = [(f, ISO, tmc_amd.Grid.make(f.shape))] + [(s, iso, g) for s, g, iso in (_slab("6x8"), _slab("6x6", 12))]
    eng, ref = tmc_amd.Engine(0), tmc_amd.Engine(0)
    try:
        print("[gpu] capacities and rerun together", flush=True)
        ms = eng.extract_batch(vols, flags=flags)
        assert ms[0].host_syncs == 3 + 1   # the last for the records
        for i, (v, iso, g) in enumerate(vols):
            ref.extract(v, iso, g, flags=flags)
            exp, got = ref.download(), eng.download_batch(i)
            for k in KEYS:
                assert_same(got[k], exp[k], f"volume {i}: {k}")
    finally:
        eng.close()
        ref.close()


def test_slab_without_allocation():
    flags = SIMPLIFY_ALL | TRIANGLES
    f, g, iso = _slab("6x8")
    eng = tmc_amd.Engine(0)
    cap = 4096
    sizes = [24 * cap, 24 * cap, 16 * cap, 24 * cap, 16 * cap, 4 * cap, 4 * cap]
    bufs = [eng.alloc(s) for s in sizes]
    o = tmc_amd.OutBuffers()
    o.positions, o.normals, o.quads, o.tris, o.twins, o.he_flags, o.he_v = (b.ptr.value for b in bufs)
    o.cap_v = o.cap_q = cap
    try:
        dev = eng.alloc(f.nbytes).upload(f)
        for i in range(2):
            m, _ = eng.extract_noalloc(dev, iso, g, o, flags=flags)
            quads = eng.copy_to_host(np.empty((m.nq, 4), np.int32), m.d_quads)
            v = eng.copy_to_host(np.empty((m.nv, 3), np.float64), m.d_positions)
            em = eng.extract(f, iso, g, flags=flags)
            ed = eng.download()
            assert m.nq == em.nq and m.nv == em.nv
            assert_same(quads, ed["quads"], "quads")
            assert_same(v, ed["v"], "v")
        dev.free()
    finally:
        for b in bufs:
            b.free()
        eng.close()


@pytest.mark.parametrize("name", FIELDS)
def test_usual_fields_stay_on_the_live_mesh(name):
    f, g, iso = FIELDS[name]()
    print(f"[gpu] live path {name}", flush=True)
    eng = tmc_amd.Engine(0)
    try:
        for flags in (SIMPLIFY_ALL, SIMPLIFY_3X3Y_ISOLATED):
            assert not _ran_staged(eng, f, iso, g, flags)
    finally:
        eng.close()
