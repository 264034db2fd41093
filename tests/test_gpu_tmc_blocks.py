"""TMC cells taken in blocks on the GPU: noise (a third of the cells ambiguous,
every edge owner and grid side met), cell counts at the edges of a block and of
the lists of ambiguous cells -- against the oracle, bit for
bit."""
import numpy as np
import pytest

from meshcheck import assert_same

pytestmark = pytest.mark.gpu

import tmc_amd  # noqa: E402

# (nz, ny, nx): cells 1; 255 / 256 / 257 (all active in noise, nearly);
# one row, column and line of cells; 1.9 million (waves that flush their list)
SHAPES = [(2, 2, 2), (4, 6, 18), (5, 9, 9), (2, 2, 258), (2, 300, 2), (300, 2, 2), (20, 21, 22), (100, 130, 150)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_blocks_match_oracle(engine, oracle, shape):
    f = np.random.default_rng(sum(shape)).standard_normal(shape)
    if f.size < 1 << 20:
        f[0] = np.where(np.arange(shape[1])[:, None] % 2 == np.arange(shape[2]) % 2, 1.0, -1.0) * np.abs(f[0])
    g = tmc_amd.Grid.make(shape, (0.1, 0.2, 0.3), (0.5, 0.25, 0.75))
    print(f"[gpu] tmc blocks {shape}", flush=True)
    exp = oracle.tmc(g, f.ravel(), 0.05)
    got = engine.tmc(f, 0.05, g)
    for k in ("v", "n", "tris"):
        assert_same(got[k], exp[k], f"{shape}: {k}")
