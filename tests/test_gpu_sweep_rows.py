"""Rows that are not whole vectors, on the GPU: every remainder of nx, rows
shorter than a vector, rows that end at and after a segment, and a field that
ends with its buffer -- against the oracle, bit for bit, with noise on every
point so that a point read from its neighbour's place shows."""
import numpy as np
import pytest
import torch

from meshcheck import assert_same

pytestmark = pytest.mark.gpu

import tmc_amd  # noqa: E402
from tmc_amd import SIMPLIFY_ALL  # noqa: E402

SHAPES = [(2, 2, 2), (2, 2, 3), (3, 4, 4), (4, 3, 5), (5, 20, 6), (4, 18, 7), (3, 17, 9), (6, 33, 255), (5, 17, 257),
          (3, 18, 258), (4, 16, 259), (2, 3, 513)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_ragged_rows_match_oracle(engine, oracle, shape, dtype):
    rng = np.random.default_rng(sum(shape))
    f = rng.standard_normal(shape).astype(dtype)
    g = tmc_amd.Grid.make(shape, (0.1, 0.2, 0.3), (0.5, 0.25, 0.75))
    s = f.astype(np.float64).ravel()
    exp = oracle.tmc(g, s, 0.05)
    # one element into its buffer, and ending with it
    buf = torch.empty(f.size + 1, dtype=torch.from_numpy(f).dtype, device="cuda")
    buf[1:] = torch.from_numpy(f).ravel().cuda()
    torch.cuda.synchronize()
    for at in (f, buf.data_ptr() + f.itemsize):
        print(f"[gpu] rows {shape} {np.dtype(dtype).name} {'host' if at is f else at % 32}", flush=True)
        got = engine.tmc(at, 0.05, g, shape=shape, dtype=dtype)
        for k in ("v", "n", "tris"):
            assert_same(got[k], exp[k], f"{shape}: {k}")


def test_ragged_batch_rows(engine, oracle):
    """One volume of rows shorter than a vector puts the whole batch on clamped
    loads; without it the others take vectors."""
    vols = [(np.random.default_rng(n).standard_normal((4, 9, n)).astype(np.float32), 0.05, None) for n in (5, 260, 257, 3)]
    for n in (4, 3):
        print(f"[gpu] batch of {n}", flush=True)
        engine.extract_batch(vols[:n], flags=SIMPLIFY_ALL)
        got = [engine.download_batch(i) for i in range(n)]
        for i in range(n):
            g = tmc_amd.Grid.make(vols[i][0].shape)
            s = vols[i][0].astype(np.float64).ravel()
            exp = oracle.dualmc(g, s, oracle.gradient(g, s), 0.05, True)
            for k in ("v", "n", "quads", "he", "he_v"):
                assert_same(got[i][k], exp[k], f"batch of {n}, volume {i}: {k}")
