"""Batches of very small volumes on the GPU: groups of 1, 2, 4 and 8 (row,
segment)s in passes large enough for 16, members against the volume alone, and
the memory such a pass holds."""
import numpy as np
import pytest

from meshcheck import assert_same

pytestmark = pytest.mark.gpu

import tmc_amd  # noqa: E402
from tmc_amd import FIELD_ON_DEVICE, SIMPLIFY_ALL, TRIANGLES  # noqa: E402

FLAGS = SIMPLIFY_ALL | TRIANGLES
# volumes, shape: 1, 9, 12, 25 and 8 (row, segment)s each
BATCHES = [(70000, (2, 2, 2)), (8000, (4, 4, 4)), (6000, (5, 4, 3)), (3000, (6, 6, 4)), (10000, (3, 5, 5))]


@pytest.mark.parametrize("count,shape", BATCHES, ids=lambda x: "x".join(map(str, np.atleast_1d(x))))
def test_batch_of_small_volumes(engine, count, shape):
    rng = np.random.default_rng(count)
    f = rng.standard_normal((count,) + shape).astype(np.float32)
    print(f"[gpu] {count} volumes of {shape}", flush=True)
    eng = tmc_amd.Engine(0)
    try:
        buf = eng.alloc(f.nbytes).upload(f)
        g = tmc_amd.Grid.make(shape)
        vols = [(buf.ptr.value + i * f[0].nbytes, 0.1, g) for i in range(count)]
        meshes = eng.extract_batch(vols, flags=FLAGS | FIELD_ON_DEVICE)
        for i in [0, 1, 7, count // 2, count - 2, count - 1]:
            m = engine.extract(f[i], 0.1, g, flags=FLAGS)
            exp, got = engine.download(), eng.download_batch(i)
            assert meshes[i].nq == m.nq and meshes[i].active_cells == m.active_cells
            for k in ("v", "n", "quads", "tris", "he", "he_v", "bnd"):
                assert_same(got[k], exp[k], f"volume {i}:{k}")
        if shape == (2, 2, 2):
            # no quadrilaterals: the lists of the rows, 1 KB each, and the
            # cells' records; padded to 16 rows a volume they alone held 1.1 GB
            assert eng.context_bytes() < 250e6
        buf.free()
    finally:
        eng.close()
