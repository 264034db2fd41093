"""The field sweep of passes of 2^28 points and more (8 cell rows a wave instead
of 4) on the GPU, for doubles and for ragged rows: a batch of one volume many
times over against the volume alone."""
import numpy as np
import pytest

from meshcheck import assert_same

pytestmark = pytest.mark.gpu

import tmc_amd  # noqa: E402
from tmc_amd import FIELD_ON_DEVICE, SIMPLIFY_ALL, workloads  # noqa: E402


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("shape", [(133, 131, 132), (130, 133, 131), (70, 66, 517)], ids=lambda s: "x".join(map(str, s)))
def test_many_points_match_alone(dtype, shape):
    f, g, iso = workloads.schwarz(shape, seed=4)
    f = (f + 0.05 * np.random.default_rng(4).standard_normal(f.shape)).astype(dtype)
    count = (1 << 28) // f.size + 1
    eng = tmc_amd.Engine(0)
    try:
        buf = eng.alloc(f.nbytes).upload(f)
        eng.extract(buf, iso, g, flags=SIMPLIFY_ALL, dtype=dtype)
        exp = eng.download()
        print(f"[gpu] {count} volumes of {shape} {np.dtype(dtype).name}", flush=True)
        eng.extract_batch([(buf.ptr.value, iso, g)] * count, flags=SIMPLIFY_ALL | FIELD_ON_DEVICE, dtype=dtype)
        for i in (0, count // 2, count - 1):
            got = eng.download_batch(i)
            for k in ("v", "n", "quads", "he", "he_v", "bnd"):
                assert_same(got[k], exp[k], f"{shape} volume {i}: {k}")
        buf.free()
    finally:
        eng.close()
