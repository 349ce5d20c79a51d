"""GPU checks of the GPT decode step as one resident kernel (gpt_token.hip).

The reference is the same call on a context created with MIT2CFM_GPT_RESIDENT=0,
whose steps are separate fp32 launches that test_gpu_gpt.py holds to the oracle.
The resident kernel's products are split f16 pairs on the matrix cores (a pair
holds a value to 2^-23, or 2^-36 below 2^-13, the weights are exact in f16) with fp32 sums, so the two
differ by the order of fp32 sums of up to 5,120 terms: logits of magnitude about
1 agree to a few 1e-6, and the bar is test_gpu_gpt.py's 1e-5 for such pairs.

A head's keys are split over four workgroups (row r to workgroup r % 4), each of
which holds 208 of its rows in LDS and reads the rest from memory, so cache
lengths run over every remainder of 4, from empty, and across 832.
"""
from __future__ import annotations

import threading
import time

import numpy as np
import pytest

from conftest import gpt_paths
from test_gpu_gpt_prefill import small_values

pytestmark = pytest.mark.gpu

W = 1280
SAMPLING = dict(temperature=0.8, top_k=30, top_p=0.8, repetition_penalty=10.0)


def _tensors(mit2, tensors, layers):
    t = {**tensors, **mit2.synthetic_gpt_tensors(layers=layers)}
    b = np.array(t["gpt.mel_head.bias"], np.float32)
    b[mit2.GPT_STOP_TOKEN] -= 20.0  # no early stop
    t["gpt.mel_head.bias"] = b
    return t


def _plain(mit2, t, monkeypatch):
    monkeypatch.setenv("MIT2CFM_GPT_RESIDENT", "0")
    c = mit2.Context(t, device=0)
    monkeypatch.delenv("MIT2CFM_GPT_RESIDENT")
    return c


@pytest.fixture(scope="module")
def pair2(mit2, tensors):
    t = _tensors(mit2, tensors, 2)
    mp = pytest.MonkeyPatch()
    a, b = mit2.Context(t, device=0), _plain(mit2, t, mp)
    mp.undo()
    yield a, b
    a.close()
    b.close()


def _rows(n, seed):
    return (np.random.default_rng(seed).standard_normal((n, W)) * 0.05).astype(np.float32)


def _pair(a, b, steps, P, call):
    """`call` on the resident context and on the plain one, each on its own path."""
    prefill = {"row_prefills": 1} if P else {}
    ra, how = gpt_paths(a, lambda: call(a))
    assert how == {"resident_steps": steps, **prefill}
    rb, how = gpt_paths(b, lambda: call(b))
    assert how == {"plain_steps": steps, **prefill}
    return ra, rb


def _same(a, b):
    assert a["predicted"].tolist() == b["predicted"].tolist()
    assert a["input_tokens"].tolist() == b["input_tokens"].tolist()
    err = float(np.abs(a["last_logits"] - b["last_logits"]).max())
    print(f"  logits max-abs {err:.2e}", flush=True)
    assert err <= 1e-5


@pytest.mark.parametrize("P,steps", [(0, 1), (0, 9), (1, 3), (2, 1), (3, 8), (65, 17), (827, 1), (828, 12), (1100, 3)])
def test_greedy_equals_separate_launches(pair2, P, steps):
    print(f"resident greedy P={P} steps={steps}", flush=True)
    x = _rows(P, P)
    _same(*_pair(*pair2, steps, P, lambda c: c.gpt_kv_greedy(x, steps, True)))


@pytest.mark.parametrize("layers", [1, 3])
def test_layer_counts(mit2, tensors, monkeypatch, layers):
    t = _tensors(mit2, tensors, layers)
    a, b = mit2.Context(t, device=0), _plain(mit2, t, monkeypatch)
    try:
        print(f"resident greedy layers={layers}", flush=True)
        _same(*_pair(a, b, 9, 7, lambda c: c.gpt_kv_greedy(_rows(7, 1), 9)))
    finally:
        a.close()
        b.close()


def test_sampled_equals_separate_launches(pair2):
    x = _rows(33, 2)
    _same(*_pair(*pair2, 20, 33, lambda c: c.gpt_kv_sample(x, 20, 11, hf_generate_positions=True,
                                                           history=[1] * 33 + [8192], **SAMPLING)))


def test_repeats_to_the_bit(pair2):
    """The order of every sum is fixed, whichever workgroup comes first."""
    x = _rows(40, 3)
    a = pair2[0].gpt_kv_greedy(x, 30)
    for _ in range(5):
        b, how = gpt_paths(pair2[0], lambda: pair2[0].gpt_kv_greedy(x, 30))
        assert how == {"row_prefills": 1, "resident_steps": 30}
        assert a["predicted"].tolist() == b["predicted"].tolist()
        assert np.array_equal(a["last_logits"], b["last_logits"])


def test_contexts_on_threads_take_turns(mit2, tensors):
    """Two contexts decode at once from two threads: their resident kernels run
    one after the other, and each gives what it gives alone."""
    t = _tensors(mit2, tensors, 2)
    ctx = [mit2.Context(t, device=0) for _ in range(2)]
    try:
        want = [c.gpt_kv_greedy(_rows(20 + i, i), 60) for i, c in enumerate(ctx)]
        got = [[], []]

        def work(i):
            for _ in range(4):
                got[i].append(ctx[i].gpt_kv_greedy(_rows(20 + i, i), 60))

        threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
        for th in threads:
            th.start()
        for th in threads:
            th.join()
        for i in range(2):
            assert len(got[i]) == 4
            for g in got[i]:
                assert g["predicted"].tolist() == want[i]["predicted"].tolist()
                assert np.array_equal(g["last_logits"], want[i]["last_logits"])
            n = ctx[i].gpt_counts()
            assert n["resident_steps"] == 5 * 60 and n["plain_steps"] == n["wait_reruns"] == n["range_reruns"] == 0
    finally:
        for c in ctx:
            c.close()


def test_other_work_beside_a_decode(mit2, tensors):
    """Mel decodes on a second context while the resident kernel, which holds the
    whole GPU, makes codes on the first: both give what they give alone, no step
    is taken plain, and the mel decodes get their part of the GPU (measured 1.6 of
    their time alone; 26 when the steps followed each other without a pause)."""
    t = _tensors(mit2, tensors, 24)
    a, b = mit2.Context(t, device=0), mit2.Context(tensors, device=0)
    try:
        rng = np.random.default_rng(8)
        args = [rng.standard_normal(s).astype(np.float32) for s in ((128, 80), (38, 80), (128, 512), (192,))]
        x = _rows(150, 9)
        mel = lambda: b.decode(*args, 12, 0.7)

        def seconds(n=10):
            t0 = time.perf_counter()
            for _ in range(n):
                assert np.array_equal(mel(), mel0)
            return (time.perf_counter() - t0) / n

        mel0, codes0 = mel(), a.gpt_kv_greedy(x, 400)
        alone = seconds()
        before, stop, got = a.gpt_counts(), threading.Event(), []

        def work():
            while not stop.is_set():
                got.append(a.gpt_kv_greedy(x, 400))

        th = threading.Thread(target=work)
        th.start()
        try:
            beside = seconds(30)
        finally:
            stop.set()
            th.join()
        print(f"mel decode alone {1e3 * alone:.2f} ms, beside codes {1e3 * beside:.2f} ms", flush=True)
        for g in got:
            assert g["predicted"].tolist() == codes0["predicted"].tolist()
            assert np.array_equal(g["last_logits"], codes0["last_logits"])
        n = a.gpt_counts()
        assert n["resident_steps"] - before["resident_steps"] == 400 * len(got)
        assert n["plain_steps"] == n["wait_reruns"] == n["range_reruns"] == 0
        assert beside <= 4 * alone
    finally:
        a.close()
        b.close()


def test_a_wait_that_runs_out_falls_back(mit2, tensors, monkeypatch):
    """With a limit of one poll the kernel gives up at its first wait and ends;
    the call decodes with the separate launches: their bits."""
    t = _tensors(mit2, tensors, 2)
    b = _plain(mit2, t, monkeypatch)
    monkeypatch.setenv("MIT2CFM_GPT_SPIN_LIMIT", "1")
    a = mit2.Context(t, device=0)
    try:
        x = _rows(25, 4)
        ra, how = gpt_paths(a, lambda: a.gpt_kv_greedy(x, 12))
        assert how == {"row_prefills": 1, "wait_reruns": 1, "plain_steps": 12}
        rb = b.gpt_kv_greedy(x, 12)
        assert ra["predicted"].tolist() == rb["predicted"].tolist()
        assert np.array_equal(ra["last_logits"], rb["last_logits"])
        # the resident kernel is tried again after 1, 2, 4 .. plain calls
        rb = b.gpt_kv_sample(x, 12, 5, **SAMPLING)
        for gave_up in (0, 1, 0, 0, 1, 0, 0, 0, 0, 1, 0):
            ra, how = gpt_paths(a, lambda: a.gpt_kv_sample(x, 12, 5, **SAMPLING))
            assert how == {"row_prefills": 1, "plain_steps": 12, **({"wait_reruns": 1} if gave_up else {})}
            assert ra["predicted"].tolist() == rb["predicted"].tolist()
            assert np.array_equal(ra["last_logits"], rb["last_logits"])
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("where", ["gelu", "layernorm"])
def test_decode_values_past_f16(mit2, tensors, monkeypatch, where):
    """A decode step whose values do not fit f16 (nothing of the prefix does,
    as there is none) runs again through the fp32 launches: their bits."""
    t = _tensors(mit2, tensors, 2)
    name, at, v = {"gelu": ("gpt.gpt.h.1.mlp.c_fc.bias", 5119, 1e5),
                   "layernorm": ("gpt.final_norm.bias", 3, -1e5)}[where]
    bias = np.array(t[name], np.float32)
    bias[at] = v
    t[name] = bias
    a, b = mit2.Context(t, device=0), _plain(mit2, t, monkeypatch)
    try:
        for _ in range(2):
            ra, how = gpt_paths(a, lambda: a.gpt_kv_greedy(_rows(0, 0), 10))
            assert how == {"range_reruns": 1, "plain_steps": 10}
            rb = b.gpt_kv_greedy(_rows(0, 0), 10)
            assert ra["predicted"].tolist() == rb["predicted"].tolist()
            assert np.isfinite(ra["last_logits"]).all()
            assert np.array_equal(ra["last_logits"], rb["last_logits"])
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("where", ["layernorm", "value", "gelu"])
@pytest.mark.parametrize("spare", [False, True])
def test_steps_below_a_pairs_full_precision(mit2, tensors, monkeypatch, where, spare):
    """As test_rows_below_a_pairs_full_precision, for the token steps."""
    t = small_values(_tensors(mit2, tensors, 2), where, spare)
    a, b = mit2.Context(t, device=0), _plain(mit2, t, monkeypatch)
    try:
        ra, how = gpt_paths(a, lambda: a.gpt_kv_greedy(_rows(0, 0), 6))
        assert how == ({"resident_steps": 6} if spare else {"range_reruns": 1, "plain_steps": 6})
        _same(ra, b.gpt_kv_greedy(_rows(0, 0), 6))
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("P,fails", [(0, 0), (0, 5), (19, 8), (3, 100)])
def test_the_step_that_fails_is_taken_again(mit2, tensors, monkeypatch, P, fails):
    """One position whose first LayerNorm output does not fit f16 (it meets zero
    weights, so the result is as finite as the others): the steps before it keep
    their form, it and the rest run plain, greedy and sampled, with the sorts of
    the sampler that no NaN may enter."""
    t = _tensors(mit2, tensors, 2)
    emb, pos, g, w = (np.array(t["gpt." + n], np.float32) for n in
                      ("mel_embedding.weight", "mel_pos_embedding.emb.weight", "gpt.h.0.ln_1.weight",
                       "gpt.h.0.attn.c_attn.weight"))
    emb, pos, w = emb.reshape(-1, W), pos.reshape(-1, W), w.reshape(W, 3 * W)
    emb[:, 7] = pos[:, 7] = w[7] = 0
    pos[fails, 7], g[7] = 1.0, 1e5
    t.update({"gpt.mel_embedding.weight": emb, "gpt.mel_pos_embedding.emb.weight": pos, "gpt.gpt.h.0.ln_1.weight": g,
              "gpt.gpt.h.0.attn.c_attn.weight": w})
    x = _rows(P, 50 + P)
    x[:, 7] = 0
    steps = fails + 11
    a, b = mit2.Context(t, device=0), _plain(mit2, t, monkeypatch)
    try:
        want = {"range_reruns": 1, "plain_steps": 11}
        want |= {"row_prefills": 1} if P else {}
        want |= {"resident_steps": fails} if fails else {}
        for call in (lambda c: c.gpt_kv_greedy(x, steps),
                     lambda c: c.gpt_kv_sample(x, steps, 3, **SAMPLING),
                     lambda c: c.gpt_kv_sample(x, steps, 4, temperature=1.1, top_k=2000, top_p=0.9)):
            ra, how = gpt_paths(a, lambda: call(a))
            assert how == want
            _same(ra, call(b))
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("top_k,top_p", [(1, 0.5), (2, 1.0), (30, 0.8), (30, 1.0), (30, 0.05), (63, 0.9), (64, 0.9),
                                         (65, 0.9), (200, 0.99)])
def test_sampler_survivor_counts(pair2, orc, mit2, top_k, top_p):
    """The sampler's wave form (up to 64 survivors) and the general form next to
    it, against the oracle's processors on the same logits: the same tokens kept
    and, drawn from them, the same code."""
    x = _rows(15, 100 + top_k)
    cfg = dict(temperature=0.9, top_k=top_k, top_p=top_p, repetition_penalty=1.5)
    g = orc.GPT(_tensors(mit2, {}, 2))
    for seed in range(3):
        got = pair2[1].gpt_kv_sample(x, 6, seed, **cfg)
        ref = g.kv_sample(x, 6, seed, **cfg)
        assert got["predicted"].tolist() == ref["predicted"].tolist()
        a, b = got["last_processed_logits"], ref["last_processed_logits"]
        assert np.array_equal(np.isfinite(a), np.isfinite(b))
