"""GPU checks of the vocoder's resblock groups run in step: the three resblocks'
activations and convs of a stage go three to a launch (launch_gemm_group), with
tiles chosen by the rows, and their mean is taken by a kernel of its own.

A group's output must equal, bit for bit, the mean of its resblocks run one by
one: the tiles and the launch change no sum's order, and the mean is
((0 + v0 / 3) + v1 / 3) + v2 / 3 in fp32 either way.  Row counts sit at the edges
of the tile rules (64-row tiles of the 768- and 384-channel stages: up to 40, 64,
90, 100 tiles; the pipelined 128-row tiles from 128 to 256, whose convs run one
by one, and beyond), odd counts and one row among them.
"""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx_bvg(mit2, tensors):
    c = mit2.Context({**tensors, **mit2.synthetic_bigvgan_tensors()}, device=0)
    yield c
    c.close()


CASES = [(0, t) for t in (1, 17, 320, 384, 385, 640, 641, 960, 1024, 1025, 2752, 5504)]
CASES += [(1, t) for t in (64, 832, 833, 1345, 1921, 2112, 5441)]
CASES += [(2, 65), (2, 16385), (3, 127), (4, 255), (4, 33001), (5, 511)]


@pytest.mark.parametrize("mode", ["f32", "f16"])
@pytest.mark.parametrize("stage,rows", CASES)
def test_group_is_the_mean_of_its_resblocks(ctx_bvg, mode, stage, rows):
    C = 768 >> stage
    x = np.random.default_rng(100 * stage + rows).standard_normal((rows, C)).astype(np.float32)
    print(f"group stage={stage} rows={rows} {mode}", flush=True)
    ctx_bvg.set_precision("vocoder", mode)
    try:
        got = ctx_bvg.bigvgan_stage("group", stage, x)
        v = [ctx_bvg.bigvgan_stage("resblock", 3 * stage + r, x) for r in range(3)]
    finally:
        ctx_bvg.set_precision("vocoder", "f32")
    third = np.float32(3.0)
    want = ((np.float32(0) + v[0] / third) + v[1] / third) + v[2] / third
    assert got.shape == want.shape and np.isfinite(want).all()
    assert np.array_equal(got.view(np.uint32), want.astype(np.float32).view(np.uint32))
