"""3-face edges (getBndVertices and the halfedges that they override) on the GPU:
few of them, as many as a context starts with room for, and more, which are
applied by a launch per step -- against the oracle, bit for bit, on the first
pass and on later ones, which are replayed."""
import numpy as np
import pytest

from meshcheck import assert_same

pytestmark = pytest.mark.gpu

import tmc_amd  # noqa: E402
from tmc_amd import SIMPLIFY_ALL  # noqa: E402


@pytest.mark.parametrize("simplify", [True, False])
@pytest.mark.parametrize("n,most", [(600, 1024), (12500, None), (40000, None)])
def test_records_match_oracle(oracle, n, most, simplify):
    shape = (3, 3, n)
    f = np.random.default_rng(n).standard_normal(shape).astype(np.float32)
    g = tmc_amd.Grid.make(shape, (0.1, 0.2, 0.3), (0.5, 0.25, 0.75))
    s = f.astype(np.float64).ravel()
    exp = oracle.dualmc(g, s, oracle.gradient(g, s), 0.1, simplify)
    eng = tmc_amd.Engine(0)
    try:
        for i in range(8):
            m = eng.extract(f, 0.1, g, flags=SIMPLIFY_ALL if simplify else 0)
            got = eng.download()
            print(f"[gpu] {shape} simplify {simplify} pass {i} mode {m.pass_mode}: {m.nbnd // 2} records", flush=True)
            assert (m.nbnd // 2 <= most) if most else m.nbnd // 2 > 900
            for k in ("v", "n", "quads", "he", "he_v", "bnd"):
                assert_same(got[k], exp[k], f"{shape} pass {i}:{k}")
        assert m.pass_mode == 2
    finally:
        eng.close()
