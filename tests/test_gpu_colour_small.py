"""Face colouring by one block and by a launch per level, on the GPU: meshes on
either side of the one-block size, dense in faces, against the oracle, bit for
bit (which faces merge depends on the colours)."""
import numpy as np
import pytest

from meshcheck import assert_same

pytestmark = pytest.mark.gpu

import tmc_amd  # noqa: E402
from tmc_amd import SIMPLIFY_ALL  # noqa: E402

# room for the faces: 4,096 (its smallest) .. 32,768 (one block's most, 32^3)
# and above (34^3)
SHAPES = [(3, 4, 5), (11, 12, 13), (17, 16, 15), (24, 25, 26), (32, 32, 32), (34, 34, 34)]


@pytest.mark.parametrize("noise", [0.3, 3.0])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_colouring_matches_oracle(engine, oracle, shape, noise):
    rng = np.random.default_rng(sum(shape))
    k, j, i = np.meshgrid(*[np.linspace(-4, 4, n) for n in shape], indexing="ij")
    f = (np.cos(k) + np.cos(j) + np.cos(i) + noise * rng.standard_normal(shape)).astype(np.float32)
    g = tmc_amd.Grid.make(shape, (0.1, 0.2, 0.3), (0.5, 0.25, 0.75))
    s = f.astype(np.float64).ravel()
    print(f"[gpu] colouring {shape} noise {noise}", flush=True)
    exp = oracle.dualmc(g, s, oracle.gradient(g, s), 0.05, True)
    for _ in range(4):   # the later passes are replayed
        engine.extract(f, 0.05, g, flags=SIMPLIFY_ALL)
        got = engine.download()
        for key in ("v", "n", "quads", "he", "he_v"):
            assert_same(got[key], exp[key], f"{shape}:{key}")
