"""The work that is timed and compared: what a speech-synthesis program asks of this library.

Each case is one call (or one request) through the public Python binding,
`mit2cfm.Context`, on a resident model:

  condition  condition_device: length regulator + prompt merge, semantic codes -> decode condition
  decode     decode_device: one request's CFG Euler decode of the mel, buffers on the GPU
  batch      decode_batched_device: several right-padded requests at once
  vocoder    bigvgan_device: mel -> waveform
  acoustic   acoustic_device: condition, seeded noise, decode and vocoder in one call
  prefill    gpt_cached_decode: a prefix through the GPT stack, then one row decoded against it
  greedy     gpt_kv_greedy: prefix + greedy mel codes
  sample     gpt_kv_sample: prefix + sampled mel codes (IndexTTS2's generation settings)

Sizes are those of bench.py, the tests and the reference's published segment;
`draw` spreads over the same ranges.  The models have the real architecture
with the library's synthetic weights (one per process, as a server keeps
them); inputs come from the seed.  `exact` restates every path in float64
torch, from the weights and the mathematics alone.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "index-tts2-metal_amd"))
import mit2cfm  # noqa: E402

DEV = "cuda:0"
SAMPLING = dict(temperature=0.8, top_k=30, top_p=0.8, repetition_penalty=10.0)


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the first short chunk of a streamed answer: the smallest call, where launches count
        dict(name="condition_24", kind="condition", codes=24, prompt=64, precision="f32"),
        # the condition of a full synthesis segment behind a long voice prompt
        dict(name="condition_553", kind="condition", codes=553, prompt=629, precision="f32"),
        # a short utterance at few steps: launch-bound
        dict(name="decode_128", kind="decode", tokens=128, prompt=38, steps=12, cfg=0.7),
        # the headline request
        dict(name="decode_860", kind="decode", tokens=860, prompt=258, steps=25, cfg=0.7),
        # long-form speech
        dict(name="decode_3000", kind="decode", tokens=3000, prompt=900, steps=25, cfg=0.7),
        # batched serving: eight requests of mixed lengths, padded to the longest
        dict(name="batch_8", kind="batch", nreq=8, t_max=1348, steps=16, cfg=0.7, padding="compute"),
        # a short chunk's waveform in the fast mode, an odd length
        dict(name="vocoder_61_f16", kind="vocoder", tokens=61, precision="f16"),
        # the headline request's waveform, fp32-level arithmetic (the default)
        dict(name="vocoder_860", kind="vocoder", tokens=860, precision="f32"),
        # codes to waveform in one call: the reference's published steady-state segment
        dict(name="acoustic_553", kind="acoustic", codes=553, prompt=629, steps=16, cfg=0.7),
        # a conditioning + text prefix through the GPT, no codes yet (time to the first code)
        dict(name="gpt_prefill_213", kind="prefill", prefix=213),
        # the mel codes of a full segment
        dict(name="gpt_greedy_150_553", kind="greedy", prefix=150, codes=553),
        # a short sentence with the generation settings the synthesis path uses
        dict(name="gpt_sample_57_96", kind="sample", prefix=57, codes=96),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["condition", "decode", "decode", "batch", "vocoder", "acoustic", "prefill", "greedy", "sample"])
    if kind == "condition":
        return dict(kind=kind, codes=log(8, 900), prompt=rng.randint(0, 640), precision=rng.choice(["f32", "f32", "f16"]))
    if kind == "decode":
        t = log(48, 2999)
        return dict(kind=kind, tokens=t, prompt=rng.randint(0, t // 2), steps=rng.randint(6, 25),
                    cfg=rng.choice([0.7, 0.7, 0.0]))
    if kind == "batch":
        return dict(kind=kind, nreq=rng.randint(2, 8), t_max=log(100, 1347), steps=rng.randint(6, 16), cfg=0.7,
                    padding=rng.choice(["compute", "skip"]))
    if kind == "vocoder":
        return dict(kind=kind, tokens=log(12, 1600), precision=rng.choice(["f32", "f32", "f16"]))
    if kind == "acoustic":
        return dict(kind=kind, codes=log(30, 552), prompt=rng.randint(60, 640), steps=rng.randint(8, 25), cfg=0.7)
    if kind == "prefill":
        return dict(kind=kind, prefix=log(5, 640))
    if kind == "greedy":
        return dict(kind=kind, prefix=log(16, 300), codes=log(16, 400))
    return dict(kind=kind, prefix=log(16, 300), codes=log(16, 400))


# ------------------------------------------------------------------ resident models
_models: dict = {}


def _tensors(part: str) -> dict:
    """The synthetic weights of one part of the model, as host arrays."""
    if part not in _models:
        sets = {"estimator": (mit2cfm.SYNTH_ESTIMATOR, 20240605), "regulator": (mit2cfm.SYNTH_LENGTH_REGULATOR, 20240606),
                "vocoder": (mit2cfm.SYNTH_BIGVGAN, 20240607), "gpt": (mit2cfm.SYNTH_GPT, 20240608)}
        set_id, seed = sets[part]
        t = mit2cfm.synthetic_set(set_id, seed, 0.02)
        if part == "gpt":
            # A trained decoder stops at the end of the sentence, random weights anywhere:
            # the stop token is kept from winning, so that a call makes the codes it asks for.
            t["gpt.mel_head.bias"][mit2cfm.GPT_STOP_TOKEN] -= 20.0
        _models[part] = t
    return _models[part]


def _context(kind: str) -> mit2cfm.Context:
    key = "gpt context" if kind in ("prefill", "greedy", "sample") else "acoustic context"
    if key not in _models:
        parts = ["estimator", "gpt"] if key == "gpt context" else ["estimator", "regulator", "vocoder"]
        _models[key] = mit2cfm.Context({k: v for p in parts for k, v in _tensors(p).items()}, device=0)
    return _models[key]


def _frames(codes: int) -> int:
    return int(np.floor(np.float32(codes) * np.float32(1.72)))


def _lengths(case):
    """The requests' lengths and prompt lengths of a padded batch: the longest fills t_max."""
    n, t_max = case["nreq"], case["t_max"]
    tokens = [max(2, round(t_max * (1.0 - 0.55 * ((5 * r) % n) / n))) for r in range(n)]
    return tokens, [int(t * 0.3) for t in tokens]


# ------------------------------------------------------------------ inputs
def _inputs(case, seed):
    """Host-independent inputs of a case, on the GPU (the GPT's prefix rows on the host, where its calls take them)."""
    g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=DEV)

    def mel(*shape):  # log-mel values
        return normal(*shape) * 2.0 - 5.0

    kind = case["kind"]
    if kind == "condition":
        return dict(s_infer=normal(case["codes"], 1024), prompt_cond=normal(max(case["prompt"], 1), 512))
    if kind == "decode":
        t, p = case["tokens"], case["prompt"]
        return dict(x0=normal(t, 80), prompt=mel(max(p, 1), 80), cond=normal(t, 512), style=normal(192))
    if kind == "batch":
        n, t = case["nreq"], case["t_max"]
        d = dict(x0=normal(n, t, 80), prompt=mel(n, t, 80), cond=normal(n, t, 512), style=normal(n, 192))
        for r, (tok, p) in enumerate(zip(*_lengths(case))):
            d["x0"][r, tok:] = 0
            d["cond"][r, tok:] = 0
            d["prompt"][r, p:] = 0
        return d
    if kind == "vocoder":
        return dict(mel=mel(case["tokens"], 80))
    if kind == "acoustic":
        p = case["prompt"]
        return dict(s_infer=normal(case["codes"], 1024), prompt_cond=normal(p, 512), prompt_mel=mel(p, 80),
                    style=normal(192), seed=seed)
    rows = case["prefix"] + (1 if kind == "prefill" else 0)
    return dict(prefix=(normal(rows, 1280) * 0.05).cpu().numpy(), seed=seed)


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    s["ctx"] = ctx = _context(case["kind"])
    kind = case["kind"]
    if kind == "condition":
        ctx.set_precision("length_regulator", case["precision"])
        s["out"] = torch.empty(case["prompt"] + _frames(case["codes"]), 512, device=DEV)
    elif kind == "decode":
        s["out"] = torch.empty(case["tokens"], 80, device=DEV)
    elif kind == "batch":
        ctx.set_padding(case["padding"])
        s["tokens"], s["prompts"] = (np.array(v, np.uint32) for v in _lengths(case))
        s["out"] = torch.zeros(case["nreq"], case["t_max"], 80, device=DEV)
    elif kind == "vocoder":
        ctx.set_precision("vocoder", case["precision"])
        s["out"] = torch.empty(256 * case["tokens"], device=DEV)
    elif kind == "acoustic":
        ctx.set_precision("length_regulator", "f32")
        ctx.set_precision("vocoder", "f32")
        n = _frames(case["codes"])
        s["out"], s["mel_out"] = torch.empty(256 * n, device=DEV), torch.empty(case["prompt"] + n, 80, device=DEV)
    torch.cuda.synchronize()  # the context works on a stream of its own
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "condition":
        ctx.condition_device(s["s_infer"].data_ptr(), case["codes"], s["prompt_cond"].data_ptr(), case["prompt"],
                             s["out"].data_ptr())
        return s["out"]
    if kind == "decode":
        ctx.decode_device(s["x0"].data_ptr(), s["prompt"].data_ptr(), s["cond"].data_ptr(), s["style"].data_ptr(),
                          case["tokens"], case["prompt"], case["steps"], case["cfg"], s["out"].data_ptr())
        return s["out"]
    if kind == "batch":
        ctx.decode_batched_device(s["tokens"], s["prompts"], s["x0"].data_ptr(), s["prompt"].data_ptr(),
                                  s["cond"].data_ptr(), s["style"].data_ptr(), case["t_max"], case["steps"],
                                  case["cfg"], s["out"].data_ptr())
        # with skipped padding the rows past a request's length are unspecified
        return [s["out"][r, :t] for r, t in enumerate(s["tokens"].tolist())] if case["padding"] == "skip" else s["out"]
    if kind == "vocoder":
        ctx.bigvgan_device(s["mel"].data_ptr(), case["tokens"], s["out"].data_ptr())
        return s["out"]
    if kind == "acoustic":
        ctx.acoustic_device(s["s_infer"].data_ptr(), case["codes"], s["prompt_cond"].data_ptr(),
                            s["prompt_mel"].data_ptr(), case["prompt"], s["style"].data_ptr(), s["seed"], 1.0,
                            case["steps"], case["cfg"], s["out"].data_ptr(), s["mel_out"].data_ptr())
        return {"wav": s["out"], "mel": s["mel_out"]}
    if kind == "prefill":
        ln_f, final_norm, logits, argmax = ctx.gpt_cached_decode(s["prefix"], case["prefix"])
        return {"ln_f": ln_f, "final_norm": final_norm, "logits": logits, "argmax": argmax}
    if kind == "greedy":
        r = ctx.gpt_kv_greedy(s["prefix"], case["codes"], hf_generate_positions=True)
        return {"codes": r["predicted"].astype(np.int64), "logits": r["last_logits"]}
    r = ctx.gpt_kv_sample(s["prefix"], case["codes"], s["seed"], hf_generate_positions=True,
                          history=[1] * case["prefix"] + [mit2cfm.GPT_START_TOKEN], **SAMPLING)
    return {"codes": r["predicted"].astype(np.int64), "logits": r["last_logits"], "processed": r["last_processed_logits"]}


# ------------------------------------------------------------------ work and tolerance
def _decode_work(rows_valid, steps, cfg, nreq, rows):
    """Estimator FLOPs (GEMMs and attention of every step) and bytes: the f16 weights once, inputs and output."""
    branches = 2 if cfg > 0 else 1
    per_row = 13 * 2 * (512 * 1536 + 512 * 512 + 512 * 3072 + 1536 * 512) + 6 * 2 * 1024 * 512  # blocks, skip-ins
    per_row += 2 * 80 * 512 + 2 * 592 * 512 + 2 * 2 * 512 * 512  # merge (mel columns), skip_linear, conv1, res_projection
    per_row += 8 * 2 * 2560 * 1024 + 7 * 2 * 512 * 1024 + 2 * 512 * 512 + 2 * 512 * 512 + 2 * 512 * 80  # WaveNet, final
    attn = 13 * 4 * 512 * sum(t * t for t in rows_valid)
    flops = steps * branches * (per_row * sum(rows_valid) + attn)
    weights = 2 * 80e6  # without the time conditioning's projections, whose products are kept per step count
    return flops, weights + 4.0 * rows * (80 * 3 + 512) + 4.0 * nreq * 192


def _condition_work(codes, prompt):
    n = _frames(codes)
    flops = 2.0 * codes * 512 * 1024 + 4 * 2.0 * n * 512 * 1536 + 2.0 * n * 512 * 512
    nbytes = 2.0 * (512 * 1024 + 4 * 512 * 1536 + 512 * 512) + 4.0 * (codes * 1024 + prompt * 512 + (prompt + n) * 512)
    return flops, nbytes


def _vocoder_work(tokens):
    weights = 2.0 * 112.2e6  # f16 conv weights of the real architecture
    return mit2cfm.bigvgan_flops(tokens), weights + 4.0 * tokens * (80 + 256)


_GPT_LAYER = 1280 * 3840 + 1280 * 1280 + 2 * 1280 * 5120
_GPT_HEAD = 8194 * 1280


def _gpt_work(prefix, codes):
    # (codes = 0: the prefix and one more row against it, all known at the start)
    if codes == 0:
        flops = 2.0 * 24 * _GPT_LAYER * (prefix + 1) + 2.0 * _GPT_HEAD + 24 * 2.0 * 1280 * (prefix + 1) * (prefix + 2)
        return flops, 2.0 * (24 * _GPT_LAYER + _GPT_HEAD) + 4.0 * (prefix + 1) * 1280
    flops = 2.0 * 24 * _GPT_LAYER * (prefix + codes) + 2.0 * _GPT_HEAD * codes
    ctx = prefix + codes
    flops += 24 * 4.0 * 1280 * (ctx * (ctx + 1) / 2)
    # the weights once for the prefix (its rows together) and once a code: each code waits for the one before,
    # and they don't fit a cache; a code also reads the keys and values before it
    nbytes = 2.0 * 24 * _GPT_LAYER + codes * 2.0 * (24 * _GPT_LAYER + _GPT_HEAD)
    nbytes += 24 * 2 * 1280 * 4.0 * sum(prefix + k for k in range(codes)) + prefix * 1280 * 4.0
    return flops, nbytes


def work(case):
    kind = case["kind"]
    if kind == "condition":
        f, b = _condition_work(case["codes"], case["prompt"])
    elif kind == "decode":
        f, b = _decode_work([case["tokens"]], case["steps"], case["cfg"], 1, case["tokens"])
    elif kind == "batch":
        rows = case["nreq"] * case["t_max"]
        if case["padding"] == "compute":
            valid = [case["t_max"]] * case["nreq"]
        else:
            valid = _lengths(case)[0]
        f, b = _decode_work(valid, case["steps"], case["cfg"], case["nreq"], rows)
    elif kind == "vocoder":
        f, b = _vocoder_work(case["tokens"])
    elif kind == "acoustic":
        n, p = _frames(case["codes"]), case["prompt"]
        parts = [_condition_work(case["codes"], p), _decode_work([p + n], case["steps"], case["cfg"], 1, p + n), _vocoder_work(n)]
        f, b = (sum(v) for v in zip(*parts))
    else:
        f, b = _gpt_work(case["prefix"], case.get("codes", 0))
    return {"flops": f, "bytes": b}


def tolerance(case):
    """About four times the error measured against `exact` (the f16 modes: f16 operands; the estimator: f16 operands
    inside steps whose sum moves the mel by little; the GPT and the f32 modes: fp32 sums)."""
    kind = case["kind"]
    if kind == "condition":
        return {"rel": 2e-3} if case["precision"] == "f16" else {"rel": 2e-6}  # f16 operands; measured 1.6e-7 to 2.3e-7
    if kind in ("decode", "batch"):
        return {"rel": 1.2e-5}  # measured 2.4e-6 to 2.9e-6
    if kind == "vocoder":
        return {"rel": 5e-3} if case["precision"] == "f16" else {"rel": 2e-5}  # measured 9e-4; 4.5e-6
    if kind == "acoustic":
        return {"rel": 3e-5}  # measured 2.5e-6 (mel), 5.7e-6 (waveform)
    return {"rel": 4e-6, "differ": 0.0}  # measured 3.5e-7 to 3.7e-7


# ------------------------------------------------------------------ float64 restatements
F64 = torch.float64


def _w64(part):
    """A part's weights in float64 on the GPU."""
    key = part + " f64"
    if key not in _models:
        _models[key] = {k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV).to(F64) for k, v in _tensors(part).items()}
    return _models[key]


def _lin(x, w, b=None):
    y = x @ w.t()
    return y if b is None else y + b


def _wn(w, name):
    """A weight-normed weight, normalised over all but its first axis."""
    g, v = w[name + ".weight_g"], w[name + ".weight_v"]
    flat = v.reshape(v.shape[0], -1)
    return (flat * (g.reshape(-1, 1) / flat.norm(dim=1, keepdim=True))).reshape(v.shape)


def _conv(x, w, b, dilation=1):
    """Zero-padded 'same' conv, x [T][in], w [out][in][k]."""
    k = w.shape[2]
    pad = (k - 1) * dilation // 2
    xp = torch.nn.functional.pad(x, (0, 0, pad, pad))
    y = sum(xp[i * dilation : i * dilation + x.shape[0]] @ w[:, :, i].t().contiguous() for i in range(k))
    return y if b is None else y + b


def _regulator64(s_infer, n):
    w = {k[len(mit2cfm.LR_PREFIX):]: v for k, v in _w64("regulator").items()}
    x = _lin(s_infer.to(F64), w["content_in_proj.weight"], w["content_in_proj.bias"])
    scale = np.float32(x.shape[0]) / np.float32(n)
    src = np.minimum(np.floor(np.arange(n, dtype=np.float32) * scale).astype(np.int64), x.shape[0] - 1)
    x = x[torch.from_numpy(src).to(DEV)]
    for i in (0, 3, 6, 9):
        x = _conv(x, w["model.%d.weight" % i], w["model.%d.bias" % i])
        x = (x - x.mean()) / torch.sqrt(x.var(unbiased=False) + 1e-5) * w["model.%d.weight" % (i + 1)] + w["model.%d.bias" % (i + 1)]
        x = x * torch.tanh(torch.nn.functional.softplus(x, threshold=700.0))
    return _lin(x, w["model.12.weight"][:, :, 0], w["model.12.bias"])


def _condition64(s_infer, codes, prompt_cond, prompt):
    n = _frames(codes)
    return torch.cat([prompt_cond[:prompt].to(F64), _regulator64(s_infer, n)])


class _Estimator64:
    """The DiT estimator (input merge, 13 AdaRMSNorm blocks, WaveNet, AdaLN final layer) in float64."""

    def __init__(self):
        self.w = {k[len(mit2cfm.PREFIX):]: v for k, v in _w64("estimator").items()}
        w = self.w
        self.norm = {k[: -len(".weight_g")]: _wn(w, k[: -len(".weight_g")]) for k in w if k.endswith(".weight_g")}

    def embed(self, t, which):
        w, p = self.w, "t_embedder" if which == 1 else "t_embedder2"
        a = 1000.0 * t * w[p + ".freqs"]
        e = torch.cat([torch.cos(a), torch.sin(a)])
        h = torch.nn.functional.silu(_lin(e, w[p + ".mlp.0.weight"], w[p + ".mlp.0.bias"]))
        return _lin(h, w[p + ".mlp.2.weight"], w[p + ".mlp.2.bias"])

    def adaptive(self, x, t1, p):
        w = self.w
        wb = _lin(t1, w[p + ".project_layer.weight"], w[p + ".project_layer.bias"])
        return wb[:512] * (x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w[p + ".norm.weight"]) + wb[512:]

    def attention(self, x, keep, p):
        t = x.shape[0]
        q, k, v = _lin(x, self.w[p + ".wqkv.weight"]).split(512, dim=-1)
        ang = torch.arange(t, dtype=F64, device=DEV)[:, None] * 10000.0 ** (-torch.arange(0, 64, 2, dtype=F64, device=DEV) / 64.0)
        cos, sin = torch.cos(ang)[:, None], torch.sin(ang)[:, None]

        def rope(z):
            z = z.reshape(t, 8, 32, 2)
            a, b = z[..., 0], z[..., 1]
            return torch.stack([a * cos - b * sin, b * cos + a * sin], -1).reshape(t, 8, 64)

        q, k, v = rope(q), rope(k), v.reshape(t, 8, 64)
        out = torch.empty(t, 8, 64, dtype=F64, device=DEV)
        for h in range(8):
            s = q[:, h].contiguous() @ k[:, h].t().contiguous() / 8.0
            s = s.masked_fill(~keep[None], -math.inf)
            out[:, h] = torch.softmax(s, -1) @ v[:, h].contiguous()
        return _lin(out.reshape(t, 512), self.w[p + ".wo.weight"])

    def forward(self, x, px, cond, style, t, keep):
        w, t1, t2 = self.w, self.embed(t, 1), self.embed(t, 2)
        rows = x.shape[0]
        cp = _lin(cond, w["cond_projection.weight"], w["cond_projection.bias"])
        h = _lin(torch.cat([x, px, cp, style.expand(rows, 192)], -1), w["cond_x_merge_linear.weight"], w["cond_x_merge_linear.bias"])
        saved = []
        for layer in range(13):
            p = "transformer.layers.%d" % layer
            if layer > 6:
                h = _lin(torch.cat([h, saved.pop()], -1), w[p + ".skip_in_linear.weight"], w[p + ".skip_in_linear.bias"])
            h = h + self.attention(self.adaptive(h, t1, p + ".attention_norm"), keep, p + ".attention")
            z = self.adaptive(h, t1, p + ".ffn_norm")
            f = p + ".feed_forward"
            h = h + _lin(torch.nn.functional.silu(_lin(z, w[f + ".w1.weight"])) * _lin(z, w[f + ".w3.weight"]), w[f + ".w2.weight"])
            if layer < 6:
                saved.append(h)
        h = self.adaptive(h, t1, "transformer.norm")
        h = _lin(torch.cat([h, x], -1), w["skip_linear.weight"], w["skip_linear.bias"])
        y, res = _lin(h, w["conv1.weight"], w["conv1.bias"]), _lin(h, w["res_projection.weight"], w["res_projection.bias"])
        m = keep.to(F64)[:, None]
        cl = "wavenet.cond_layer.conv.conv"
        g = _lin(t2, self.norm[cl][:, :, 0], w[cl + ".bias"])
        at = torch.arange(-2, rows + 2, device=DEV).abs()  # reflected positions
        at = torch.where(at >= rows, 2 * (rows - 1) - at, at).clamp(0, rows - 1)
        out = torch.zeros_like(y)
        for layer in range(8):
            ip, rp = "wavenet.in_layers.%d.conv.conv" % layer, "wavenet.res_skip_layers.%d.conv.conv" % layer
            yp = y[at]
            z = sum(yp[i : i + rows] @ self.norm[ip][:, :, i].t().contiguous() for i in range(5)) + w[ip + ".bias"] + g[1024 * layer : 1024 * (layer + 1)]
            z = _lin(torch.tanh(z[:, :512]) * torch.sigmoid(z[:, 512:]), self.norm[rp][:, :, 0], w[rp + ".bias"])
            if layer < 7:
                y = (y + z[:, :512]) * m
                out = out + z[:, 512:]
            else:
                out = out + z
        h = out * m + res
        ss = _lin(torch.nn.functional.silu(t1), w["final_layer.adaLN_modulation.1.weight"], w["final_layer.adaLN_modulation.1.bias"])
        h = (h - h.mean(-1, keepdim=True)) / torch.sqrt(h.var(-1, unbiased=False, keepdim=True) + 1e-6) * (1.0 + ss[512:]) + ss[:512]
        h = _lin(h, self.norm["final_layer.linear"], w["final_layer.linear.bias"])
        return _lin(h, w["conv2.weight"][:, :, 0], w["conv2.bias"])

    def euler(self, x0, prompt, cond, style, valid, p, steps, cfg):
        x, cond, style = x0.to(F64).clone(), cond.to(F64), style.to(F64)
        keep = torch.arange(x.shape[0], device=DEV) < valid
        px = torch.zeros_like(x)
        px[:p] = prompt[:p]
        x[:p] = 0
        t, dt = np.float32(0), np.float32(1) / np.float32(steps)
        for _ in range(steps):
            d = self.forward(x, px, cond, style, float(t), keep)
            if cfg > 0:
                null = self.forward(x, torch.zeros_like(px), torch.zeros_like(cond), torch.zeros_like(style), float(t), keep)
                d = (1.0 + cfg) * d - cfg * null
            x = x + float(dt) * d
            x[:p] = 0
            t = np.float32(t + dt)
        return x


def _estimator64():
    if "estimator64" not in _models:
        _models["estimator64"] = _Estimator64()
    return _models["estimator64"]


def _snake64(x, w, p):
    """BigVGAN's alias-free activation: 2x upsample, SnakeBeta, low-pass and downsample, x [T][C]."""
    up, down = w[p + ".upsample.filter"].reshape(-1), w[p + ".downsample.lowpass.filter"].reshape(-1)
    t = x.shape[0]
    xp = x[torch.arange(-6, t + 6, device=DEV).clamp(0, t - 1)]  # row r holds x[clamp(r - 6)]
    u = torch.empty(2 * t, x.shape[1], dtype=F64, device=DEV)
    # upsampled position 2v + o takes filter taps k with 2v + o + 15 - k even, at x[(2v + o + 15 - k) / 2 - 5]
    for o in (0, 1):
        u[o::2] = 2.0 * sum(up[k] * xp[(o + 15 - k) // 2 - 5 + 6 : (o + 15 - k) // 2 - 5 + 6 + t] for k in range(12) if (o + 15 - k) % 2 == 0)
    alpha, beta = torch.exp(w[p + ".act.alpha"]), torch.exp(w[p + ".act.beta"])
    u = u + torch.sin(u * alpha) ** 2 / (beta + 1e-9)
    at = torch.arange(-5, 2 * t + 6, device=DEV).clamp(0, 2 * t - 1)
    u = u[at]
    return sum(down[k] * u[k : k + 2 * t : 2] for k in range(12))


def _vocoder64(mel):
    w = _w64("vocoder")
    x = _conv(mel.to(F64), _wn(w, "bigvgan.conv_pre"), w["bigvgan.conv_pre.bias"])
    for g, (name, _, cout, k, stride, pad) in enumerate(mit2cfm.BIGVGAN_UPSAMPLERS):
        wt = _wn(w, name)
        t = x.shape[0]
        full = torch.zeros((t - 1) * stride + k, cout, dtype=F64, device=DEV)
        for i in range(k):
            full[i : i + (t - 1) * stride + 1 : stride] += x @ wt[:, :, i].contiguous()
        x = full[pad : pad + t * stride] + w[name + ".bias"]
        total = 0
        for i in range(3):
            p, y = "bigvgan.resblocks.%d" % (3 * g + i), x
            for j, d in enumerate((1, 3, 5)):
                z = _snake64(y, w, "%s.activations.%d" % (p, 2 * j))
                z = _conv(z, _wn(w, "%s.convs1.%d" % (p, j)), w["%s.convs1.%d.bias" % (p, j)], d)
                z = _snake64(z, w, "%s.activations.%d" % (p, 2 * j + 1))
                y = y + _conv(z, _wn(w, "%s.convs2.%d" % (p, j)), w["%s.convs2.%d.bias" % (p, j)])
            total = total + y
        x = total / 3.0
    x = _conv(_snake64(x, w, "bigvgan.activation_post"), _wn(w, "bigvgan.conv_post"), None)
    return x.reshape(-1).clamp(-1.0, 1.0)


def _noise64(n, seed):
    """The library's seeded Gaussian noise: splitmix64 uniforms (rounded to float32) through Box-Muller."""
    k = np.arange(1, 2 * ((n + 1) // 2) + 1, dtype=np.uint64)
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + k * np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    u = (((z >> np.uint64(11)).astype(np.float64) + 0.5) * 2.0**-53).astype(np.float32)
    r, a = np.sqrt(-2.0 * np.log(u[0::2].astype(np.float64))), 2.0 * np.pi * u[1::2].astype(np.float64)
    out = np.stack([r * np.cos(a), r * np.sin(a)], -1).reshape(-1)[:n]
    return torch.from_numpy(out).to(DEV)


class _Gpt64:
    """The GPT-2 stack with its key/value cache in float64."""

    def __init__(self, rows):
        self.w = _w64("gpt")
        self.k = torch.zeros(24, 20, rows, 64, dtype=F64, device=DEV)
        self.v = torch.zeros_like(self.k)
        self.n = 0

    def norm(self, x, p):
        m = x.mean(-1, keepdim=True)
        return (x - m) / torch.sqrt(((x - m) ** 2).mean(-1, keepdim=True) + 1e-5) * self.w[p + ".weight"] + self.w[p + ".bias"]

    def rows(self, x):
        """Appends x's rows to the cache; returns their hidden states."""
        w, m, n0 = self.w, x.shape[0], self.n
        n1 = n0 + m
        later = torch.arange(n1, device=DEV)[None] > torch.arange(n0, n1, device=DEV)[:, None]
        for l in range(24):
            p = "gpt.gpt.h.%d" % l
            qkv = self.norm(x, p + ".ln_1") @ w[p + ".attn.c_attn.weight"] + w[p + ".attn.c_attn.bias"]
            q, k, v = (z.reshape(m, 20, 64).transpose(0, 1) for z in qkv.split(1280, -1))
            self.k[l, :, n0:n1], self.v[l, :, n0:n1] = k, v
            s = torch.matmul(q.contiguous(), self.k[l, :, :n1].transpose(1, 2).contiguous()) / 8.0
            a = torch.softmax(s.masked_fill(later[None], -math.inf), -1)
            a = torch.matmul(a, self.v[l, :, :n1].contiguous()).transpose(0, 1).reshape(m, 1280)
            x = x + a @ w[p + ".attn.c_proj.weight"] + w[p + ".attn.c_proj.bias"]
            f = self.norm(x, p + ".ln_2") @ w[p + ".mlp.c_fc.weight"] + w[p + ".mlp.c_fc.bias"]
            f = 0.5 * f * (1.0 + torch.tanh(0.7978845608028654 * (f + 0.044715 * f**3)))
            x = x + f @ w[p + ".mlp.c_proj.weight"] + w[p + ".mlp.c_proj.bias"]
        self.n = n1
        return x

    def head(self, x):
        ln_f = self.norm(x, "gpt.gpt.ln_f")
        fn = self.norm(ln_f, "gpt.final_norm")
        return ln_f, fn, fn @ self.w["gpt.mel_head.weight"].t() + self.w["gpt.mel_head.bias"]


def _sample64(logits, history, rng):
    """The sampling processors and one draw, as float64: the chosen code, the processed scores, the generator's state."""
    s = logits.copy()
    seen = np.unique([t for t in history if t < s.size])
    s[seen] = np.where(s[seen] < 0, s[seen] * SAMPLING["repetition_penalty"], s[seen] / SAMPLING["repetition_penalty"])
    s /= SAMPLING["temperature"]
    s[s < np.sort(s)[-SAMPLING["top_k"]]] = -np.inf
    order = np.lexsort((np.arange(s.size), s))
    p = np.exp(s[order] - s.max())
    drop = order[:-1][np.cumsum(p / p.sum())[:-1] <= 1.0 - SAMPLING["top_p"]]
    s[drop] = -np.inf
    mask = (1 << 64) - 1
    rng = (rng + 0x9E3779B97F4A7C15) & mask
    z = ((rng ^ (rng >> 30)) * 0xBF58476D1CE4E5B9) & mask
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
    z ^= z >> 31
    p = np.exp(s - s.max())
    target = (z >> 11) * 2.0**-53 * p.sum()
    return int(np.nonzero(np.cumsum(p) > target)[0][0]), s, rng


def _generate64(case, s):
    g = _Gpt64(case["prefix"] + case["codes"])
    if case["prefix"]:
        g.rows(torch.from_numpy(s["prefix"]).to(DEV).to(F64))
    emb, pos = g.w["gpt.mel_embedding.weight"], g.w["gpt.mel_pos_embedding.emb.weight"]
    history, rng = [1] * case["prefix"] + [mit2cfm.GPT_START_TOKEN], s["seed"]
    token = mit2cfm.GPT_START_TOKEN
    for step in range(case["codes"]):
        _, _, logits = g.head(g.rows((emb[token] + pos[step + 1 if step else 0])[None]))
        if case["kind"] == "greedy":
            token, processed = int(logits[0].argmax()), None
        else:
            token, processed, rng = _sample64(logits[0].cpu().numpy(), history, rng)
            history.append(token)
    return logits[0], processed


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "condition":
        return _condition64(s["s_infer"], case["codes"], s["prompt_cond"], case["prompt"])
    if kind == "decode":
        return _estimator64().euler(s["x0"], s["prompt"], s["cond"], s["style"], case["tokens"], case["prompt"], case["steps"], case["cfg"])
    if kind == "batch":
        tokens, prompts = _lengths(case)
        x = [_estimator64().euler(s["x0"][r], s["prompt"][r], s["cond"][r], s["style"][r], tokens[r], prompts[r], case["steps"], case["cfg"])
             for r in range(case["nreq"])]
        return [v[:t] for v, t in zip(x, tokens)] if case["padding"] == "skip" else torch.stack(x)
    if kind == "vocoder":
        return _vocoder64(s["mel"])
    if kind == "acoustic":
        p, n = case["prompt"], _frames(case["codes"])
        cond = _condition64(s["s_infer"], case["codes"], s["prompt_cond"], p)
        mel = _estimator64().euler(_noise64((p + n) * 80, s["seed"]).reshape(p + n, 80), s["prompt_mel"], cond, s["style"], p + n, p, case["steps"], case["cfg"])
        return {"wav": _vocoder64(mel[p:]), "mel": mel}
    if kind == "prefill":
        g = _Gpt64(case["prefix"] + 1)
        x = g.rows(torch.from_numpy(s["prefix"]).to(DEV).to(F64))
        ln_f, fn, logits = g.head(x[-1:])
        return {"ln_f": ln_f[0], "final_norm": fn[0], "logits": logits[0], "argmax": None}
    # a code that a rounding decides the other way changes all that follow: the logits of short runs only
    if case["codes"] > 200:
        return None
    logits, processed = _generate64(case, s)
    return {"codes": None, "logits": logits, "processed": processed} if kind == "sample" else {"codes": None, "logits": logits}
