"""Cell records in groups of (row, segment)s on the GPU: volumes on either
side of the group sizes' limits, rows of several segments, groups that end in
padding, and a batch whose volumes end inside a group -- against the oracle,
bit for bit (DMC) and against each volume alone (batch, TMC by the oracle)."""
import numpy as np
import pytest

from meshcheck import assert_same

pytestmark = pytest.mark.gpu

import tmc_amd  # noqa: E402
from tmc_amd import SIMPLIFY_ALL, TRIANGLES  # noqa: E402

# (nz, ny, nx): (row, segment)s 1; 24; 8,190 / 8,192 (groups of 1 / 4); 16,376
# in two segments; 65,535 / 65,536 (groups of 4 / 16)
SHAPES = [(2, 2, 2), (3, 5, 700), (91, 92, 9), (65, 129, 9), (93, 90, 270), (256, 258, 7), (257, 257, 7)]


def _field(shape, seed):
    """A plane with noise: flat segments, ambiguous cells, empty rows."""
    rng = np.random.default_rng(seed)
    k, j, i = np.meshgrid(*[np.linspace(-1, 1, n) for n in shape], indexing="ij")
    f = (k + 0.3 * j + 0.1 * i + 0.02 * rng.standard_normal(shape)).astype(np.float32)
    f[: min(4, shape[0])] += 0.5 * rng.standard_normal((min(4, shape[0]),) + shape[1:]).astype(np.float32)
    return f


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_groups_match_oracle(engine, oracle, shape):
    f = _field(shape, sum(shape))
    g = tmc_amd.Grid.make(shape, (0.1, 0.2, 0.3), (0.5, 0.25, 0.75))
    s = f.astype(np.float64).ravel()
    print(f"[gpu] groups {shape}", flush=True)
    exp = oracle.dualmc(g, s, oracle.gradient(g, s), 0.05, True)
    engine.extract(f, 0.05, g, flags=SIMPLIFY_ALL | TRIANGLES)
    got = engine.download()
    for k in ("v", "n", "quads", "he", "he_v"):
        assert_same(got[k], exp[k], f"{shape}:{k}")
    texp = oracle.tmc(g, s, 0.05)
    tgot = engine.tmc(f, 0.05, g)
    for k in ("v", "n", "tris"):
        assert_same(tgot[k], texp[k], f"{shape}: tmc {k}")


def test_groups_in_a_batch(engine):
    vols = [(_field(s, i), 0.05, None) for i, s in enumerate(SHAPES[1:5] * 2)]
    engine.extract_batch(vols, flags=SIMPLIFY_ALL | TRIANGLES)
    got = [engine.download_batch(i) for i in range(len(vols))]
    for i, (f, iso, _) in enumerate(vols):
        print(f"[gpu] batch volume {i} {f.shape}", flush=True)
        engine.extract(f, iso, flags=SIMPLIFY_ALL | TRIANGLES)
        exp = engine.download()
        for k in ("v", "n", "quads", "tris", "he", "he_v", "bnd"):
            assert_same(got[i][k], exp[k], f"volume {i}:{k}")
