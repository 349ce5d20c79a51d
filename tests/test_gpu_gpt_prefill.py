"""GPU checks of the GPT decoder's prefill, which pushes the prefix through each
layer as matrix-core products of split f16 pairs (launch_gemm_rows) with its own
LayerNorm and attention kernels.

The reference is the same call with MIT2CFM_GPT_ROW_PREFILL=1: one row at a time
through the decode step's fp32 kernels, which test_gpu_gpt.py holds to the
oracle.  Both forms sum in fp32 (a split pair holds a value to 2^-23, or 2^-36
below 2^-13, and the weights are exact in f16), so they differ by the order of fp32 sums: logits of
magnitude about 1 over sums of 1,280 and 5,120 terms, a few 1e-6 measured; the
bar is test_gpu_gpt.py's 1e-5 for the same comparison.

Row counts (the prefix and the row decoded with it) sit at the edges of the
16-query attention blocks, the 32- and 64-row tiles and each rule of the tile
choice, and past the 1,024-row chunk, so that a second chunk attends to the
first one's keys.
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import gpt_paths

pytestmark = pytest.mark.gpu

W = 1280


@pytest.fixture(scope="module")
def gpt2_t(mit2):
    return mit2.synthetic_gpt_tensors(layers=2)


@pytest.fixture(scope="module")
def ctx2(mit2, tensors, gpt2_t):
    c = mit2.Context({**tensors, **gpt2_t}, device=0)
    yield c
    c.close()


def _rows(n, seed):
    return (np.random.default_rng(seed).standard_normal((n, W)) * 0.05).astype(np.float32)


def _both(ctx, rows, monkeypatch, fits=True):
    """The call as row products and plain; `fits`: its values fit f16, so the
    first must not have fallen back to the second (else it must have)."""
    plain = {"plain_prefills": 1} if len(rows) > 1 else {}
    monkeypatch.delenv("MIT2CFM_GPT_ROW_PREFILL", raising=False)
    got, how = gpt_paths(ctx, lambda: ctx.gpt_cached_decode(rows, len(rows) - 1))
    assert how == ({"row_prefills": 1} if fits else {"row_prefills": 1, "range_reruns": 1, **plain})
    monkeypatch.setenv("MIT2CFM_GPT_ROW_PREFILL", "1")
    ref, how = gpt_paths(ctx, lambda: ctx.gpt_cached_decode(rows, len(rows) - 1))
    assert how == plain
    return got, ref


@pytest.mark.parametrize("M", [1, 2, 15, 16, 17, 33, 64, 65, 129, 193, 321, 450, 641, 1024, 1025, 1100])
def test_prefill_equals_row_prefill(ctx2, monkeypatch, M):
    rows = _rows(M, M)
    print(f"prefill M={M}", flush=True)
    got, ref = _both(ctx2, rows, monkeypatch)
    errs = [float(np.abs(a - b).max()) for a, b in zip(got[:3], ref[:3])]
    print(f"  ln_f {errs[0]:.2e} final_norm {errs[1]:.2e} logits {errs[2]:.2e}", flush=True)
    assert max(errs) <= 1e-5 and got[3] == ref[3]


def test_a_row_does_not_depend_on_the_prefix_length(mit2, tensors):
    """The tiles and K groups of the products follow the row count; a row's bits
    do not.  One layer whose last row attends to itself alone: keys are 8 x the
    queries' weights, and the rows before it are its negative, hundreds of units
    of score below, probability exactly 0.  So its value, projection and MLP are
    the same sums whatever stands before it."""
    t = dict(mit2.synthetic_gpt_tensors(layers=1))
    w = np.array(t["gpt.gpt.h.0.attn.c_attn.weight"], np.float32).reshape(W, 3 * W)
    b = np.array(t["gpt.gpt.h.0.attn.c_attn.bias"], np.float32)
    w[:, :W] *= 8
    w[:, W : 2 * W] = w[:, :W]
    b[: 2 * W] = 0
    t["gpt.gpt.h.0.attn.c_attn.weight"], t["gpt.gpt.h.0.attn.c_attn.bias"] = w, b
    x = _rows(1, 77)
    c = mit2.Context({**tensors, **t}, device=0)
    try:
        ref = None
        for M in (1, 2, 16, 33, 64, 65, 128, 129, 193, 213, 257, 385, 450, 833, 1024, 1025, 1100):
            print(f"row bits M={M}", flush=True)
            rows = np.concatenate([np.repeat(-x, M - 1, 0), x])
            got, how = gpt_paths(c, lambda: c.gpt_cached_decode(rows, M - 1))
            assert how == {"row_prefills": 1}
            ref = got if ref is None else ref
            for a, r in zip(got[:3], ref[:3]):
                assert np.isfinite(a).all() and np.array_equal(a, r)
    finally:
        c.close()


def test_prefill_caches_serve_the_decode(ctx2, monkeypatch):
    """Tokens decoded after the prefill read the caches it wrote."""
    prefix = _rows(97, 5)
    monkeypatch.delenv("MIT2CFM_GPT_ROW_PREFILL", raising=False)
    got, how = gpt_paths(ctx2, lambda: ctx2.gpt_kv_greedy(prefix, 20))
    assert how == {"row_prefills": 1, "resident_steps": 20}
    monkeypatch.setenv("MIT2CFM_GPT_ROW_PREFILL", "1")
    ref = ctx2.gpt_kv_greedy(prefix, 20)
    assert got["predicted"].tolist() == ref["predicted"].tolist()
    assert np.abs(got["last_logits"] - ref["last_logits"]).max() <= 1e-5


@pytest.mark.parametrize("where", ["gelu", "layernorm", "value"])
def test_values_past_f16_take_the_row_prefill(mit2, tensors, gpt2_t, monkeypatch, where):
    """A value that does not fit f16 (a c_fc output of 1e5; a LayerNorm output
    of 1e5; attention outputs of 1e5) is seen, and the call runs again through
    the fp32 row prefill: the same bits as asking for it."""
    t = dict(gpt2_t)
    if where == "gelu":
        b = np.array(t["gpt.gpt.h.1.mlp.c_fc.bias"], np.float32)
        b[7] = 1e5
        t["gpt.gpt.h.1.mlp.c_fc.bias"] = b
    elif where == "layernorm":
        b = np.array(t["gpt.gpt.h.0.ln_2.bias"], np.float32)
        b[1279] = -1e5
        t["gpt.gpt.h.0.ln_2.bias"] = b
    else:
        b = np.array(t["gpt.gpt.h.0.attn.c_attn.bias"], np.float32)
        b[2 * W + 70] = 1e5
        t["gpt.gpt.h.0.attn.c_attn.bias"] = b
    c = mit2.Context({**tensors, **t}, device=0)
    try:
        got, ref = _both(c, _rows(21, 9), monkeypatch, fits=False)
        for a, b in zip(got[:3], ref[:3]):
            assert np.isfinite(a).all() and np.array_equal(a, b)
        assert got[3] == ref[3]
        monkeypatch.delenv("MIT2CFM_GPT_ROW_PREFILL", raising=False)
        g, how = gpt_paths(c, lambda: c.gpt_kv_greedy(_rows(21, 9), 12))
        assert how["range_reruns"] == 1 and how["plain_prefills"] == 1 and how["plain_steps"] == 12
        monkeypatch.setenv("MIT2CFM_GPT_ROW_PREFILL", "1")
        r = c.gpt_kv_greedy(_rows(21, 9), 12)
        assert g["predicted"].tolist() == r["predicted"].tolist()
        assert np.array_equal(g["last_logits"], r["last_logits"])
    finally:
        c.close()


@pytest.mark.parametrize("P", [7, 8, 9, 160, 300])
def test_past_f16_the_prefix_goes_in_chunks(mit2, tensors, gpt2_t, monkeypatch, P):
    """The fp32 prefill of such a call takes eight rows a pass over the weights:
    the bits of one row at a time, in about a quarter of its time (measured
    40.6 against 140 ms at 213 rows of 24 layers; the bar leaves a factor of 2)."""
    t = dict(gpt2_t)
    b = np.array(t["gpt.gpt.h.0.mlp.c_fc.bias"], np.float32)
    b[7] = 1e5
    t["gpt.gpt.h.0.mlp.c_fc.bias"] = b
    c = mit2.Context({**tensors, **t}, device=0)
    try:
        x = _rows(P, P)
        got = [c.gpt_kv_greedy(x, 3) for _ in range(3)]
        monkeypatch.setenv("MIT2CFM_GPT_ROW_PREFILL", "1")
        ref = [c.gpt_kv_greedy(x, 3) for _ in range(3)]
        for g in got:
            assert g["predicted"].tolist() == ref[0]["predicted"].tolist()
            assert np.array_equal(g["last_logits"], ref[0]["last_logits"])
        ms = [min(r["prefill_ms"] for r in rs) for rs in (got, ref)]  # (the first with its attempt)
        print(f"P={P}: chunks {ms[0]:.2f} ms, rows {ms[1]:.2f} ms", flush=True)
        assert P < 100 or ms[0] < 0.55 * ms[1]
    finally:
        c.close()


def small_values(gpt2_t, where, spare=False):
    """Weights whose layer-1 inputs of one product are all about 2^-16 (fp32 biases
    and LayerNorm weights; that product's weights are raised, so they matter), or
    all but one of them (`spare`)."""
    t = dict(gpt2_t)

    def arr(name, shape):
        t["gpt.gpt.h.1." + name] = a = np.array(t["gpt.gpt.h.1." + name], np.float32).reshape(shape)
        return a

    noise = (np.random.default_rng(6).uniform(0.5, 1.0, 5120) * 2.0**-16).astype(np.float32)
    if where == "layernorm":
        arr("ln_2.weight", -1)[:] = 0
        v, w = arr("ln_2.bias", -1), arr("mlp.c_fc.weight", (W, 5120))
    elif where == "value":
        arr("attn.c_attn.weight", (W, 3 * W))[:, 2 * W :] = 0
        v, w = arr("attn.c_attn.bias", -1)[2 * W :], arr("attn.c_proj.weight", (W, W))
    else:
        arr("mlp.c_fc.weight", (W, 5120))[:] = 0
        v, w = arr("mlp.c_fc.bias", -1), arr("mlp.c_proj.weight", (5120, W))
    v[:] = noise[: v.size]
    if spare:
        v[3] = 0.5
    w *= 2.0**12
    return t


@pytest.mark.parametrize("where", ["layernorm", "value", "gelu"])
@pytest.mark.parametrize("spare", [False, True])
def test_rows_below_a_pairs_full_precision(mit2, tensors, gpt2_t, monkeypatch, where, spare):
    """A pair holds values below 2^-13 to 2^-36 only.  A product whose input row
    is all that small runs plain (the same bits as asking for it); one with a
    single larger value keeps its row products, which then hold the row to 2^-23
    of that value."""
    c = mit2.Context({**tensors, **small_values(gpt2_t, where, spare)}, device=0)
    try:
        for M in (2, 70, 300):
            print(f"small {where} spare={spare} M={M}", flush=True)
            got, ref = _both(c, _rows(M, 9), monkeypatch, fits=spare)
            for a, b in zip(got[:3], ref[:3]):
                assert np.isfinite(a).all()
                assert np.abs(a - b).max() <= 1e-5 if spare else np.array_equal(a, b)
    finally:
        c.close()
