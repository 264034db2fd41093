"""Face lists of the simplifications that outgrow a block's buffer, on the GPU.

With 64 blocks a block's share of these meshes is several turns, and it holds
more than the 1,024 entries above which the buffer is flushed in mid-walk:
140^3 noise has 174,599 candidates and 103,649 merges in the colour stage, the
130x120x140 field of two values 600,000 candidates, 140,000 patterns and 180,000
rewritten faces in the 3333 stage.  Against the staged engine, bit for bit."""
import os

import numpy as np
import pytest

from meshcheck import assert_same

pytestmark = pytest.mark.gpu

import tmc_amd  # noqa: E402
from tmc_amd import SIMPLIFY_3X3Y_COLOR, SIMPLIFY_ALL, STAGE_TIMING  # noqa: E402


def _field(kind, shape):
    rng = np.random.default_rng(3)
    f = rng.standard_normal(shape) if kind == "noise" else (rng.random(shape) < 0.3) - 0.5
    return f.astype(np.float32)


@pytest.mark.parametrize("kind,shape,flags", [("noise", (140, 140, 140), SIMPLIFY_3X3Y_COLOR),
                                              ("two_values", (130, 120, 140), SIMPLIFY_ALL)])
def test_lists_flushed_in_mid_walk(kind, shape, flags):
    f, g = _field(kind, shape), tmc_amd.Grid.make(shape)
    os.environ["TMC_GENERIC_ROWS"] = "1"
    try:
        staged = tmc_amd.Engine(0)
    finally:
        del os.environ["TMC_GENERIC_ROWS"]
    live = tmc_amd.Engine(0)
    try:
        em = staged.extract(f, 0.1, g, flags=flags)
        exp = staged.download()
        for cap in (64, 32768):
            live.launch = {"grid_cap": cap}
            print(f"[gpu] long lists {kind} {shape}, {cap} blocks", flush=True)
            m = live.extract(f, 0.1, g, flags=flags | STAGE_TIMING)
            assert "k_he_twins" not in live.stage_times()   # not rerun stage by stage
            got = live.download()
            assert m.summary() == em.summary()
            for k in ("v", "n", "quads", "he", "he_v", "bnd"):
                assert_same(got[k], exp[k], f"{kind} {cap} blocks: {k}")
    finally:
        live.close()
        staged.close()
