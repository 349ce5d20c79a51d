"""GPU checks of the vocoder's resblock groups run in step: the three resblocks'
activations and convs of a stage go three to a launch (launch_gemm_group), with
tiles chosen by the rows, and their mean is taken by a kernel of its own.

A group's output must equal, bit for bit, the mean of its resblocks run one by
one: the tiles and the launch change no sum's order, and the mean is
((0 + v0 / 3) + v1 / 3) + v2 / 3 in fp32 either way.  Row counts sit at the edges
of the tile rules (64-row tiles of the 768- and 384-channel stages: up to 32, 64,
100 tiles; the pipelined 128-row tiles from 128 to 256, whose convs run one by
one, and beyond), at counts between them, odd ones and one row among them.

A row's bits do not depend on the call's length either: the rows of a short call
that its end does not reach equal a longer call's, in each stage and in the
waveform.
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


CASES = [(0, t) for t in (1, 17, 320, 321, 384, 385, 640, 641, 960, 1024, 1025, 2752, 5504)]
CASES += [(1, t) for t in (64, 640, 641, 832, 833, 1345, 1921, 2112, 5441)]
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


# Rows that a group's output row depends on, to either side: six activations of 6
# and, for k = 11, convs of 5 (1 + 3 + 5) and 3 x 5.
GROUP_REACH = 36 + 45 + 15


@pytest.mark.parametrize("mode", ["f32", "f16"])
@pytest.mark.parametrize("stage,rows", [(0, 128), (0, 244), (0, 384), (0, 640), (0, 960), (1, 244), (1, 832), (1, 1921)])
def test_group_rows_do_not_depend_on_the_length(ctx_bvg, mode, stage, rows):
    C = 768 >> stage
    x = np.random.default_rng(7 * rows + stage).standard_normal((5504, C)).astype(np.float32)
    print(f"group rows stage={stage} rows={rows} {mode}", flush=True)
    ctx_bvg.set_precision("vocoder", mode)
    try:
        short, long = (ctx_bvg.bigvgan_stage("group", stage, x[:n]) for n in (rows, len(x)))
    finally:
        ctx_bvg.set_precision("vocoder", "f32")
    n = rows - GROUP_REACH
    assert np.array_equal(short[:n].view(np.uint32), long[:n].view(np.uint32))


@pytest.mark.parametrize("mode", ["f32", "f16"])
@pytest.mark.parametrize("frames", [48, 61, 90, 120, 180])
def test_waveform_does_not_depend_on_the_length(ctx_bvg, mode, frames):
    """The stages' reach in frames: conv_pre 3, the upsamplers and groups of the
    stages at 4, 16, 32, 64, 128 and 256 rows a frame (96 + 2) / 4 + (96 + 2) / 16
    + ... and the last activation and conv: under 45."""
    mel = (np.random.default_rng(frames).standard_normal((400, 80)) * 2.0 - 5.0).astype(np.float32)
    print(f"waveform frames={frames} {mode}", flush=True)
    ctx_bvg.set_precision("vocoder", mode)
    try:
        short, long = (ctx_bvg.bigvgan(mel[:n]) for n in (frames, 400))
    finally:
        ctx_bvg.set_precision("vocoder", "f32")
    n = 256 * (frames - 45)
    assert np.array_equal(short[:n].view(np.uint32), long[:n].view(np.uint32))
