"""Timed cases of the mixer library: what a program that serves the 4B model has it do.

Every case goes through `qora_mixer.Context`, the library's Python binding, on device tensors
that torch owns.  Kinds (`case["kind"]`):

  dn_step        one DeltaNet mixer decode step for `batch` sequences
  gqa_step       one GQA mixer decode step for `batch` sequences over the f16 KV cache
  layer_step     one whole decode layer of one sequence: norm + Q4 projections, mixer, MLP
  head           final norm + lm_head and the next token's sampling
  layer_prefill  one whole layer over a prompt of `tokens` tokens
  model_step     a decode token through the whole model, a captured graph replayed
  model_prefill  a prompt through the whole model, up to the last token's logits

Shapes are the 4B model's (hidden 2560, intermediate 9216, 24 DeltaNet + 8 attention layers,
vocabulary 248320); what varies is what varies in use: batch, context, prompt length,
sampling settings.
"""
from __future__ import annotations

import importlib.util
import math
import sys
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parents[1]
DEV = "cuda"
HIDDEN, INTER, VOCAB = 2560, 9216, 248320
LAYERS, ATTN_EVERY = 32, 4
MAX_BATCH, MAX_KV_BATCH, MAX_CONTEXT, MAX_PROMPT = 256, 64, 32769, 8192
F64 = torch.float64

DN_PROJ = {"in_proj_qkv": (HIDDEN, 8192), "in_proj_z": (HIDDEN, 4096), "in_proj_a": (HIDDEN, 32),
           "in_proj_b": (HIDDEN, 32), "out_proj": (4096, HIDDEN)}
ATTN_PROJ = {"q_proj": (HIDDEN, 8192), "k_proj": (HIDDEN, 1024), "v_proj": (HIDDEN, 1024), "o_proj": (4096, HIDDEN)}
MLP_PROJ = {"gate_proj": (HIDDEN, INTER), "up_proj": (HIDDEN, INTER), "down_proj": (INTER, HIDDEN)}


# ---- the cases -----------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: the recurrent mixer of one chat, one token
        {"name": "dn_step_b1", "kind": "dn_step", "batch": 1, "conv": False},
        # a serving batch, raw projections in (conv1d + SiLU run in the call)
        {"name": "dn_step_b64", "kind": "dn_step", "batch": 64, "conv": True},
        # one chat, a few pages of context
        {"name": "gqa_step_b1", "kind": "gqa_step", "batch": 1, "pos": 4096, "ragged": False},
        # the benchmark's serving step: 64 sequences at 32K context
        {"name": "gqa_step_b64_32k", "kind": "gqa_step", "batch": 64, "pos": 32768, "ragged": False},
        # a decode layer of one chat: projections, mixer, MLP
        {"name": "dn_layer_step", "kind": "layer_step", "layer": "dn", "pos": 0},
        # the end of every decode step: logits over the vocabulary, then the next token
        {"name": "head", "kind": "head", "vocab": VOCAB, "top_k": 20, "generated": 1000},
        # a one-line question through a recurrent layer
        {"name": "dn_layer_t45", "kind": "layer_prefill", "layer": "dn", "tokens": 45},
        # a long document through a recurrent layer
        {"name": "dn_layer_t4096", "kind": "layer_prefill", "layer": "dn", "tokens": 4096},
        # a page of text through an attention layer
        {"name": "attn_layer_t700", "kind": "layer_prefill", "layer": "attn", "tokens": 700},
        # the longest prompt through an attention layer
        {"name": "attn_layer_t8192", "kind": "layer_prefill", "layer": "attn", "tokens": 8192},
        # one token of a chat through the whole model
        {"name": "model_step", "kind": "model_step", "pos": 2000},
        # an ordinary prompt through the whole model
        {"name": "model_prefill_t300", "kind": "model_prefill", "tokens": 300},
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, even over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["dn_step", "gqa_step", "gqa_step", "layer_step", "head", "layer_prefill", "layer_prefill",
                       "layer_prefill", "model_step", "model_prefill"])
    if kind == "dn_step":
        return {"kind": kind, "batch": _spread(rng, 1, MAX_BATCH), "conv": rng.random() < 0.5}
    if kind == "gqa_step":
        return {"kind": kind, "batch": _spread(rng, 1, MAX_KV_BATCH), "pos": _spread(rng, 8, 32768),
                "ragged": rng.random() < 0.5}
    if kind == "layer_step":
        return {"kind": kind, "layer": "attn", "pos": _spread(rng, 8, 32768)}
    if kind == "head":
        return {"kind": kind, "vocab": _spread(rng, 8000, VOCAB), "top_k": _spread(rng, 1, 100),
                "generated": rng.randrange(0, 2000)}
    if kind == "layer_prefill":
        layer = rng.choice(["dn", "attn"])
        return {"kind": kind, "layer": layer, "tokens": _spread(rng, 2, 4096 if layer == "dn" else MAX_PROMPT)}
    if kind == "model_step":
        return {"kind": kind, "pos": _spread(rng, 8, 8192)}
    return {"kind": kind, "tokens": _spread(rng, 2, 400)}


# ---- the library ---------------------------------------------------------------------------
_made = {}


def _binding():
    if "qora_mixer" not in sys.modules:
        spec = importlib.util.spec_from_file_location("qora_mixer", ROOT / "qora-llm-4b_amd" / "qora_mixer.py")
        mod = importlib.util.module_from_spec(spec)
        sys.modules["qora_mixer"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["qora_mixer"]


def _context():
    """One context for the process, on a torch stream, reserved for the largest case."""
    if "ctx" not in _made:
        M = _binding()
        ctx = M.Context(0)
        _made["stream"] = torch.cuda.Stream()
        ctx.stream = _made["stream"].cuda_stream
        ctx.reserve(MAX_BATCH, MAX_CONTEXT, MAX_PROMPT)
        _made["ctx"] = ctx
    return _made["ctx"], _made["stream"]


# ---- inputs --------------------------------------------------------------------------------
class _Gen:
    """Seeded device tensors; every draw is another part of the same stream of numbers."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def normal(self, shape, std=1.0, mean=0.0, dtype=torch.float32):
        t = torch.randn(shape, generator=self.g, device=DEV, dtype=dtype)
        return t.mul_(std).add_(mean) if (std, mean) != (1.0, 0.0) else t

    def uniform(self, shape, lo, hi):
        return torch.rand(shape, generator=self.g, device=DEV).mul_(hi - lo).add_(lo)

    def ids(self, count, below):
        return torch.randint(0, below, (count,), generator=self.g, device=DEV, dtype=torch.int32)

    def q4(self, k, n, std=0.02):
        """A quantized N(0, std) weight in the file's layout: per 32 columns absmax / 7 in f16, codes 1 .. 15."""
        w = self.normal((k, n // 32, 32), std)
        scale = (w.abs().amax(-1) / 7).half()
        q = (w / scale.float().unsqueeze(-1)).round_().clamp_(-8, 7).add_(8).to(torch.uint8).view(k, n)
        return q[:, 0::2] | (q[:, 1::2] << 4), scale


def _dequant(weight):
    packed, scale = weight
    q = torch.stack([packed & 15, packed >> 4], -1).view(packed.shape[0], -1).to(F64) - 8
    return q * scale.to(F64).repeat_interleave(32, 1)


def _rope(rows):
    freq = 1.0 / 10_000_000.0 ** (torch.arange(32, device=DEV, dtype=F64) / 32)
    angle = (torch.arange(rows, device=DEV, dtype=torch.float32).unsqueeze(1) * freq.float()).double()
    return angle.cos().float(), angle.sin().float()


def _dn_params(g):
    return {"a_log": g.uniform((32,), 0.01, 0.1).log(), "dt_bias": torch.zeros(32, device=DEV),
            "attn_norm": g.normal((128,), 0.1, 1.0).half(), "conv_w": g.normal((8192, 4), 0.5)}


def _attn_params(g):
    return {"q_norm": g.normal((256,), 0.1).half(), "k_norm": g.normal((256,), 0.1).half()}


def _layer(g, layer):
    """A layer's parameters as a model file holds them."""
    p = {name: g.q4(k, n) for name, (k, n) in {**(DN_PROJ if layer == "dn" else ATTN_PROJ), **MLP_PROJ}.items()}
    p.update(_dn_params(g) if layer == "dn" else _attn_params(g))
    p["in_norm"], p["post_norm"] = g.normal((HIDDEN,), 0.1).half(), g.normal((HIDDEN,), 0.1).half()
    return p


def _resident(ctx, p):
    """The layer's parameters as they stay on the device: Q4 weights repacked once."""
    kept = {}
    for name, w in p.items():
        if isinstance(w, tuple):
            packed, scale = w
            k, n = packed.shape[0], packed.shape[1] * 2
            codes, gscales = torch.empty_like(packed), torch.empty_like(scale)
            ctx.q4_repack(k, n, packed.data_ptr(), scale.data_ptr(), codes.data_ptr(), gscales.data_ptr())
            kept[name] = (codes, gscales)
        else:
            kept[name] = w
    return kept


def _kinds():
    return ["attn" if i % ATTN_EVERY == ATTN_EVERY - 1 else "dn" for i in range(LAYERS)]


def _dn_cache(g, count, warm):
    shape = (count, 32, 128, 128)
    return ((g.normal(shape, 0.02), g.normal((count, 8192, 3))) if warm else
            (torch.zeros(shape, device=DEV), torch.zeros((count, 8192, 3), device=DEV)))


def _kv_cache(g, count, cap, warm):
    shape = (count, 4, cap, 256)
    if warm:
        return g.normal(shape, dtype=torch.float16), g.normal(shape, dtype=torch.float16)
    return tuple(torch.zeros(shape, device=DEV, dtype=torch.float16) for _ in range(2))


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, device=DEV, dtype=dtype)


def _inputs(case, seed):
    """What the case's call reads, from the seed alone, before anything is laid out for the device."""
    g, kind = _Gen(seed), case["kind"]
    if kind == "dn_step":
        b = case["batch"]
        state, conv_buf = _dn_cache(g, b, True)
        return {**_dn_params(g), "state": state, "conv_buf": conv_buf, "qkv": g.normal((b, 8192)),
                "a": g.normal((b, 32)), "b": g.normal((b, 32)), "z": g.normal((b, 4096))}
    if kind == "gqa_step":
        b, pos = case["batch"], case["pos"]
        k_cache, v_cache = _kv_cache(g, b, pos + 1, True)
        s = {**_attn_params(g), "k_cache": k_cache, "v_cache": v_cache, "q_gate": g.normal((b, 16, 512)),
             "k_new": g.normal((b, 4, 256)), "v_new": g.normal((b, 4, 256)), "positions": None}
        if case["ragged"]:
            s["positions"] = torch.randint(0, pos + 1, (b,), generator=g.g, device=DEV, dtype=torch.int32)
        return s
    if kind == "layer_step":
        s = {"layer": _layer(g, case["layer"]), "x": g.normal((1, HIDDEN))}
        s["state"], s["conv_buf"] = _dn_cache(g, 1, True) if case["layer"] == "dn" else (None, None)
        s["k_cache"], s["v_cache"] = _kv_cache(g, 1, case["pos"] + 1, True) if case["layer"] == "attn" else (None, None)
        return s
    if kind == "head":
        return {"x": g.normal((HIDDEN,)), "final_norm": g.normal((HIDDEN,), 0.1).half(),
                "embed": g.q4(case["vocab"], HIDDEN), "generated": g.ids(max(1, case["generated"]), case["vocab"]),
                "rng": torch.randint(1, 1 << 62, (1,), generator=g.g, device=DEV)}
    if kind == "layer_prefill":
        s = {"layer": _layer(g, case["layer"]), "x": g.normal((case["tokens"], HIDDEN))}
        s["state"], s["conv_buf"] = _dn_cache(g, 1, False) if case["layer"] == "dn" else (None, None)
        s["k_cache"], s["v_cache"] = (_kv_cache(g, 1, case["tokens"], False) if case["layer"] == "attn"
                                      else (None, None))
        return s
    # the whole model: its layers come one at a time, each from a seed of its own
    warm = kind == "model_step"
    tokens = 1 if warm else case["tokens"]
    s = {"ids": g.ids(tokens, VOCAB), "embed": g.q4(VOCAB, HIDDEN), "final_norm": g.normal((HIDDEN,), 0.1).half()}
    s["state"], s["conv_buf"] = _dn_cache(g, LAYERS - LAYERS // ATTN_EVERY, warm)
    s["k_cache"], s["v_cache"] = _kv_cache(g, LAYERS // ATTN_EVERY, case["pos"] + 1 if warm else tokens, warm)
    return s


def _model_layer(seed, i):
    return _layer(_Gen(int(seed) * 1000 + 7 + i), _kinds()[i])


# ---- the calls -----------------------------------------------------------------------------
def _p(t):
    return None if t is None else t.data_ptr()


def _w(weight):
    return weight[0].data_ptr(), weight[1].data_ptr()


def _step_buffers():
    return {"proj": _empty(8192), "z": _empty(4096), "a": _empty(32), "b": _empty(32), "k": _empty(1024),
            "v": _empty(1024), "mix": _empty(4096), "inter": _empty(INTER)}


def _decode_layer(ctx, L, t, x, state, conv_buf, k_cache, v_cache, pos, rope):
    """One layer of one token; the hidden row x is updated in place."""
    M = _binding()
    px = _p(x)
    if state is not None:
        ctx.q4_gemv_multi(HIDDEN, px, [(8192, *_w(L["in_proj_qkv"]), _p(t["proj"])),
                                       (4096, *_w(L["in_proj_z"]), _p(t["z"])),
                                       (32, *_w(L["in_proj_a"]), _p(t["a"])), (32, *_w(L["in_proj_b"]), _p(t["b"]))],
                          norm_w=_p(L["in_norm"]), conv_buf=_p(conv_buf), conv_w=_p(L["conv_w"]))
        ctx.deltanet_decode(1, M.QM_DN_POSTACT, _p(t["proj"]), None, None, _p(t["a"]), _p(t["b"]), _p(L["a_log"]),
                            _p(L["dt_bias"]), _p(t["z"]), _p(L["attn_norm"]), _p(state), _p(t["mix"]))
        ctx.q4_gemv_multi(4096, _p(t["mix"]), [(HIDDEN, *_w(L["out_proj"]), px, px)])
    else:
        ctx.q4_gemv_multi(HIDDEN, px, [(8192, *_w(L["q_proj"]), _p(t["proj"])), (1024, *_w(L["k_proj"]), _p(t["k"])),
                                       (1024, *_w(L["v_proj"]), _p(t["v"]))], norm_w=_p(L["in_norm"]))
        ctx.gqa_decode(1, _p(t["proj"]), _p(t["k"]), _p(t["v"]), _p(L["q_norm"]), _p(L["k_norm"]), _p(rope[0]),
                       _p(rope[1]), rope[0].shape[0], None, pos, _p(k_cache), _p(v_cache), k_cache.shape[-2],
                       _p(t["mix"]))
        ctx.q4_gemv_multi(4096, _p(t["mix"]), [(HIDDEN, *_w(L["o_proj"]), px, px)])
    ctx.q4_gate_up(HIDDEN, INTER, px, _p(L["post_norm"]), *_w(L["gate_proj"]), *_w(L["up_proj"]), _p(t["inter"]))
    ctx.q4_gemv_multi(INTER, _p(t["inter"]), [(HIDDEN, *_w(L["down_proj"]), px, px)])


def _prompt_buffers(tokens):
    bf = torch.bfloat16
    return {"xn": _empty(tokens, HIDDEN, dtype=torch.float16), "proj": _empty(tokens, 8192, dtype=bf),
            "z": _empty(tokens, 4096, dtype=bf), "a": _empty(tokens, 32), "b": _empty(tokens, 32),
            "k": _empty(tokens, 1024, dtype=bf), "v": _empty(tokens, 1024, dtype=bf),
            "mix": _empty(tokens, 4096, dtype=bf), "inter": _empty(tokens, INTER, dtype=bf)}


def _prefill_layer(ctx, L, t, src, x, state, conv_buf, k_cache, v_cache, rope):
    """One layer of a prompt: reads the hidden rows src, leaves the layer's in x (src and x may be the same)."""
    M = _binding()
    T = x.shape[0]
    ctx.rms_norm_f16(T, HIDDEN, _p(src), _p(L["in_norm"]), _p(t["xn"]))
    if state is not None:
        ctx.q4_gemm(T, HIDDEN, 8192, _p(t["xn"]), *_w(L["in_proj_qkv"]), y_bf16=_p(t["proj"]))
        ctx.q4_gemm(T, HIDDEN, 4096, _p(t["xn"]), *_w(L["in_proj_z"]), y_bf16=_p(t["z"]))
        ctx.q4_gemm(T, HIDDEN, 32, _p(t["xn"]), *_w(L["in_proj_a"]), y=_p(t["a"]))
        ctx.q4_gemm(T, HIDDEN, 32, _p(t["xn"]), *_w(L["in_proj_b"]), y=_p(t["b"]))
        ctx.deltanet_prefill(T, _p(t["proj"]), _p(conv_buf), _p(L["conv_w"]), _p(t["a"]), _p(t["b"]), _p(L["a_log"]),
                             _p(L["dt_bias"]), _p(t["z"]), _p(L["attn_norm"]), _p(state), _p(t["mix"]))
        ctx.q4_gemm(T, 4096, HIDDEN, _p(t["mix"]), *_w(L["out_proj"]), y=_p(x), residual=_p(src), x_dtype=M.QM_BF16)
    else:
        ctx.q4_gemm(T, HIDDEN, 8192, _p(t["xn"]), *_w(L["q_proj"]), y_bf16=_p(t["proj"]))
        ctx.q4_gemm(T, HIDDEN, 1024, _p(t["xn"]), *_w(L["k_proj"]), y_bf16=_p(t["k"]))
        ctx.q4_gemm(T, HIDDEN, 1024, _p(t["xn"]), *_w(L["v_proj"]), y_bf16=_p(t["v"]))
        ctx.gqa_prefill(T, _p(t["proj"]), _p(t["k"]), _p(t["v"]), _p(L["q_norm"]), _p(L["k_norm"]), _p(rope[0]),
                        _p(rope[1]), rope[0].shape[0], _p(k_cache), _p(v_cache), k_cache.shape[-2], _p(t["mix"]))
        ctx.q4_gemm(T, 4096, HIDDEN, _p(t["mix"]), *_w(L["o_proj"]), y=_p(x), residual=_p(src), x_dtype=M.QM_BF16)
    ctx.rms_norm_f16(T, HIDDEN, _p(x), _p(L["post_norm"]), _p(t["xn"]))
    ctx.q4_gemm_gate_up(T, HIDDEN, INTER, _p(t["xn"]), *_w(L["gate_proj"]), *_w(L["up_proj"]), _p(t["inter"]))
    ctx.q4_gemm(T, INTER, HIDDEN, _p(t["inter"]), *_w(L["down_proj"]), y=_p(x), residual=_p(x), x_dtype=M.QM_BF16)


def _layer_caches(s, i):
    """(state, conv_buf, k_cache, v_cache) of the model's layer i."""
    attn = i // ATTN_EVERY
    if _kinds()[i] == "attn":
        return None, None, s["k_cache"][attn], s["v_cache"][attn]
    return s["state"][i - attn], s["conv_buf"][i - attn], None, None


def prepare(case, seed):
    ctx, stream = _context()
    with torch.cuda.stream(stream):
        s = _inputs(case, seed)
        s["case"], kind = dict(case), case["kind"]
        if kind == "dn_step":
            s["out"] = _empty(case["batch"], 4096)
        elif kind == "gqa_step":
            s["out"] = _empty(case["batch"], 16, 256)
            s["rope"] = _rope(case["pos"] + 1)
        elif kind == "layer_step":
            s["layer"], s["t"], s["y"] = _resident(ctx, s["layer"]), _step_buffers(), _empty(1, HIDDEN)
            s["rope"] = _rope(case["pos"] + 1)
        elif kind == "head":
            s["logits"], s["token"] = _empty(case["vocab"]), _empty(1, dtype=torch.int32)
            s["top_ids"], s["top_probs"] = _empty(case["top_k"], dtype=torch.int32), _empty(case["top_k"])
        elif kind == "layer_prefill":
            s["layer"], s["t"] = _resident(ctx, s["layer"]), _prompt_buffers(case["tokens"])
            s["y"], s["rope"] = torch.empty_like(s["x"]), _rope(case["tokens"])
        else:
            tokens = s["ids"].numel()
            s["layers"] = [_resident(ctx, _model_layer(seed, i)) for i in range(LAYERS)]
            s["x"], s["logits"] = _empty(tokens, HIDDEN), _empty(VOCAB)
            s["t"] = _step_buffers() if kind == "model_step" else _prompt_buffers(tokens)
            s["rope"] = _rope(s["k_cache"].shape[-2])
            if kind == "model_step":
                torch.cuda.synchronize()
                ctx.graph_begin()
                _model(ctx, s)
                s["graph"] = ctx.graph_end()
        torch.cuda.synchronize()
    return s


def _model(ctx, s):
    x, tokens = s["x"], s["x"].shape[0]
    ctx.q4_embed(tokens, VOCAB, HIDDEN, _p(s["ids"]), *_w(s["embed"]), _p(x))
    for i, L in enumerate(s["layers"]):
        caches = _layer_caches(s, i)
        if s["case"]["kind"] == "model_step":
            _decode_layer(ctx, L, s["t"], x, *caches, s["case"]["pos"], s["rope"])
        else:
            _prefill_layer(ctx, L, s["t"], x, x, *caches, s["rope"])
    ctx.q4_lm_head(VOCAB, HIDDEN, _p(x) + (tokens - 1) * HIDDEN * 4, _p(s["final_norm"]), *_w(s["embed"]),
                   _p(s["logits"]))


def run(state):
    s, case = state, state["case"]
    ctx, stream = _context()
    M, kind = _binding(), case["kind"]
    if kind == "dn_step":
        ctx.deltanet_decode(case["batch"], M.QM_DN_PREACT if case["conv"] else M.QM_DN_POSTACT, _p(s["qkv"]),
                            _p(s["conv_buf"]), _p(s["conv_w"]), _p(s["a"]), _p(s["b"]), _p(s["a_log"]),
                            _p(s["dt_bias"]), _p(s["z"]), _p(s["attn_norm"]), _p(s["state"]), _p(s["out"]))
        return {"out": s["out"], "state": s["state"], "conv_buf": s["conv_buf"]}
    if kind == "gqa_step":
        ctx.gqa_decode(case["batch"], _p(s["q_gate"]), _p(s["k_new"]), _p(s["v_new"]), _p(s["q_norm"]),
                       _p(s["k_norm"]), _p(s["rope"][0]), _p(s["rope"][1]), case["pos"] + 1, _p(s["positions"]),
                       case["pos"], _p(s["k_cache"]), _p(s["v_cache"]), case["pos"] + 1, _p(s["out"]))
        return {"out": s["out"], "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    if kind == "layer_step":
        with torch.cuda.stream(stream):
            s["y"].copy_(s["x"])
        _decode_layer(ctx, s["layer"], s["t"], s["y"], s["state"], s["conv_buf"], s["k_cache"], s["v_cache"],
                      case["pos"], s["rope"])
        return {"y": s["y"], "state": s["state"], "conv_buf": s["conv_buf"], "k_cache": s["k_cache"],
                "v_cache": s["v_cache"]}
    if kind == "head":
        ctx.q4_lm_head(case["vocab"], HIDDEN, _p(s["x"]), _p(s["final_norm"]), *_w(s["embed"]), _p(s["logits"]))
        ctx.sample(case["vocab"], _p(s["logits"]), _p(s["generated"]), case["generated"], _p(s["rng"]),
                   _p(s["token"]), temperature=1.0, top_p=0.95, top_k=case["top_k"], presence_penalty=1.5,
                   top_ids=_p(s["top_ids"]), top_probs=_p(s["top_probs"]))
        return {"logits": s["logits"], "token": s["token"], "top_ids": s["top_ids"], "top_probs": s["top_probs"],
                "rng": s["rng"]}
    if kind == "layer_prefill":
        _prefill_layer(ctx, s["layer"], s["t"], s["x"], s["y"], s["state"], s["conv_buf"], s["k_cache"], s["v_cache"],
                       s["rope"])
        return {"y": s["y"], "state": s["state"], "conv_buf": s["conv_buf"], "k_cache": s["k_cache"],
                "v_cache": s["v_cache"]}
    if kind == "model_step":
        s["graph"].launch()
    else:
        _model(ctx, s)
    return {"logits": s["logits"], "state": s["state"], "conv_buf": s["conv_buf"], "k_cache": s["k_cache"],
            "v_cache": s["v_cache"]}


# ---- what a pass cannot do without ---------------------------------------------------------
DN_STATE = 32 * 128 * 128 * 4


def _q4_bytes(shapes):
    return sum(k * n // 2 + k * (n // 32) * 2 for k, n in shapes)


def _q4_flops(shapes):
    return sum(2 * k * n for k, n in shapes)


def _layer_work(layer, tokens, pos):
    """One layer over `tokens` tokens after `pos` cached ones: weights, hidden rows and caches once each."""
    shapes = list({**(DN_PROJ if layer == "dn" else ATTN_PROJ), **MLP_PROJ}.values())
    nbytes = _q4_bytes(shapes) + 2 * tokens * HIDDEN * 4
    flops = tokens * _q4_flops(shapes)
    if layer == "dn":
        return nbytes + 2 * (DN_STATE + 8192 * 3 * 4), flops + tokens * 32 * 128 * 128 * 7
    seen = tokens * pos + tokens * (tokens + 1) // 2
    return nbytes + (pos + tokens) * 4 * 256 * 2 * 2, flops + seen * 16 * 256 * 4


def work(case):
    kind = case["kind"]
    if kind == "dn_step":
        b = case["batch"]
        row = 4 * (8192 + 32 + 32 + 4096 + 4096) + (2 * 4 * 8192 * 3 if case["conv"] else 0)
        return {"bytes": b * (2 * DN_STATE + row) + (8192 * 16 if case["conv"] else 0),
                "flops": b * 32 * 128 * 128 * 7}
    if kind == "gqa_step":
        b = case["batch"]
        keys = b * (case["pos"] / 2 if case["ragged"] else case["pos"] + 1)
        return {"bytes": keys * 4 * 256 * 2 * 2 + b * 4 * (8192 + 2048 + 4096), "flops": keys * 16 * 256 * 4}
    if kind == "layer_step":
        nbytes, flops = _layer_work(case["layer"], 1, case["pos"])
        return {"bytes": nbytes, "flops": flops}
    if kind == "head":
        v = case["vocab"]
        return {"bytes": _q4_bytes([(v, HIDDEN)]) + 4 * (v + HIDDEN), "flops": 2 * v * HIDDEN}
    if kind == "layer_prefill":
        nbytes, flops = _layer_work(case["layer"], case["tokens"], 0)
        return {"bytes": nbytes, "flops": flops}
    tokens, pos = (1, case["pos"]) if kind == "model_step" else (case["tokens"], 0)
    each = [_layer_work(layer, tokens, pos) for layer in _kinds()]
    return {"bytes": sum(w[0] for w in each) + _q4_bytes([(VOCAB, HIDDEN)]) + 4 * VOCAB,
            "flops": sum(w[1] for w in each) + 2 * VOCAB * HIDDEN}


def tolerance(case):
    """fp32 paths differ by the order of their sums; the prompt paths round their operands to 16 bits, and in a whole
    model such a change travels through every later layer."""
    kind = case["kind"]
    if kind in ("dn_step", "gqa_step", "layer_step"):
        # the cache rows a step appends are f16: a last-place tie there is 1e-3 of one value
        return {"rel": 2e-5, "max": 2e-3}
    if kind == "head":
        return {"rel": 2e-5, "max": 2e-4}
    if kind == "layer_prefill":
        return {"rel": 1e-2, "max": 0.15}
    if kind == "model_step":
        return {"rel": 2e-4, "max": 5e-3}
    return {"rel": 3e-2, "max": 0.6}


# ---- the same in 64 bits -------------------------------------------------------------------
def _rms64(x, gain):
    return x / (x.square().mean(-1, keepdim=True) + 1e-6).sqrt() * gain


def _silu64(x):
    return x * torch.sigmoid(x)


def _l2_64(x):
    n = x.square().sum(-1, keepdim=True).sqrt()
    return torch.where(n > 1e-12, x / n, x)


def _conv64(qkv, conv_buf, conv_w):
    """qkv [T, 8192] through the causal conv1d + SiLU; the buffer after it."""
    seq = torch.cat([conv_buf.to(F64).T, qkv])
    w = conv_w.to(F64)
    act = sum(seq[j:j + qkv.shape[0]] * w[:, j] for j in range(4))
    return _silu64(act), seq[-3:].T.contiguous()


def _delta64(act, a, b, z, p, state):
    """T tokens of the gated delta rule on activated inputs [T, 8192]; state [32, 128, 128] is replaced."""
    T = act.shape[0]
    q = _l2_64(act[:, :2048].view(T, 16, 128)).repeat_interleave(2, 1) / math.sqrt(128)
    k = _l2_64(act[:, 2048:4096].view(T, 16, 128)).repeat_interleave(2, 1)
    v = act[:, 4096:].view(T, 32, 128)
    x = a + p["dt_bias"].to(F64)
    alpha = (-p["a_log"].to(F64).exp() * torch.where(x > 20, x, x.exp().log1p())).exp()
    beta = torch.sigmoid(b)
    S, ys = state.to(F64), []
    for t in range(T):
        S = S * alpha[t].view(32, 1, 1)
        delta = beta[t].view(32, 1) * (v[t] - (S * k[t].unsqueeze(1)).sum(-1))
        S = torch.baddbmm(S, delta.unsqueeze(2), k[t].unsqueeze(1))
        ys.append((S * q[t].unsqueeze(1)).sum(-1))
    y = _rms64(torch.stack(ys), p["attn_norm"].to(F64)) * _silu64(z.view(T, 32, 128))
    return y.reshape(T, 4096), S


def _rotate64(x, cos, sin):
    """Partial RoPE of [..., heads, 256] rows; cos and sin [..., 1, 32]."""
    lo, hi = x[..., :32], x[..., 32:64]
    return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin, x[..., 64:]], -1)


def _attend64(q, k, v, causal):
    """q [rows, 16, 256] over k, v [4, keys, 256], head by head; causal: row t sees keys 0 .. t."""
    out = torch.empty_like(q)
    for h in range(16):
        for lo in range(0, q.shape[0], 2048):
            rows = q[lo:lo + 2048, h]
            s = rows @ k[h // 4].T / 16
            if causal:
                at = torch.arange(lo, lo + rows.shape[0], device=DEV).unsqueeze(1)
                s.masked_fill_(torch.arange(s.shape[1], device=DEV) > at, -math.inf)
            out[lo:lo + 2048, h] = torch.softmax(s, -1) @ v[h // 4]
    return out


def _mixer_attn64(proj, k, v, p, rope, first, k_cache, v_cache):
    """Rows at positions first, first + 1, ...: attention over the caches (f64 [4, cap, 256]) after appending."""
    T = proj.shape[0]
    qg = proj.view(T, 16, 512)
    cos, sin = (r[first:first + T].to(F64).unsqueeze(1) for r in rope)
    q = _rotate64(_rms64(qg[..., :256], 1 + p["q_norm"].to(F64)), cos, sin)
    kn = _rotate64(_rms64(k.view(T, 4, 256), 1 + p["k_norm"].to(F64)), cos, sin)
    k_cache[:, first:first + T] = kn.transpose(0, 1)
    v_cache[:, first:first + T] = v.view(T, 4, 256).transpose(0, 1)
    y = _attend64(q, k_cache[:, :first + T], v_cache[:, :first + T], T > 1)
    return (y * torch.sigmoid(qg[..., 256:])).reshape(T, 4096)


def _layer64(p, x, state, conv_buf, k_cache, v_cache, first, rope):
    """One layer over the rows x; (rows after it, new state, new conv buffer)."""
    xn = _rms64(x, 1 + p["in_norm"].to(F64))
    if state is not None:
        act, conv_buf = _conv64(xn @ _dequant(p["in_proj_qkv"]), conv_buf, p["conv_w"])
        y, state = _delta64(act, xn @ _dequant(p["in_proj_a"]), xn @ _dequant(p["in_proj_b"]),
                            xn @ _dequant(p["in_proj_z"]), p, state)
        x = x + y @ _dequant(p["out_proj"])
    else:
        y = _mixer_attn64(xn @ _dequant(p["q_proj"]), xn @ _dequant(p["k_proj"]), xn @ _dequant(p["v_proj"]), p, rope,
                          first, k_cache, v_cache)
        x = x + y @ _dequant(p["o_proj"])
    xn = _rms64(x, 1 + p["post_norm"].to(F64))
    return (x + (_silu64(xn @ _dequant(p["gate_proj"])) * (xn @ _dequant(p["up_proj"]))) @ _dequant(p["down_proj"]),
            state, conv_buf)


def _first64(cache, i):
    return None if cache is None else cache[i].to(F64)


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "dn_step":
        outs, states, convs = [], [], []
        for i in range(case["batch"]):
            act, conv = s["qkv"][i:i + 1].to(F64), s["conv_buf"][i].to(F64)
            if case["conv"]:
                act, conv = _conv64(act, conv, s["conv_w"])
            y, S = _delta64(act, s["a"][i:i + 1].to(F64), s["b"][i:i + 1].to(F64), s["z"][i:i + 1].to(F64), s,
                            s["state"][i])
            outs.append(y[0]), states.append(S), convs.append(conv)
        return {"out": torch.stack(outs), "state": torch.stack(states), "conv_buf": torch.stack(convs)}
    if kind == "gqa_step":
        rope = _rope(case["pos"] + 1)
        k64, v64 = s["k_cache"].to(F64), s["v_cache"].to(F64)
        out = _empty(case["batch"], 16, 256, dtype=F64)
        for i in range(case["batch"]):
            at = case["pos"] if s["positions"] is None else int(s["positions"][i])
            out[i] = _mixer_attn64(s["q_gate"][i:i + 1].to(F64), s["k_new"][i:i + 1].to(F64),
                                   s["v_new"][i:i + 1].to(F64), s, rope, at, k64[i], v64[i]).view(16, 256)
        return {"out": out, "k_cache": k64, "v_cache": v64}
    if kind == "head":
        xn = _rms64(s["x"].to(F64), 1 + s["final_norm"].to(F64))
        logits = torch.cat([_dequant((c, e)) @ xn for c, e in zip(s["embed"][0].split(32768),
                                                                  s["embed"][1].split(32768))])
        if case["generated"]:
            logits[s["generated"][:case["generated"]].long().unique()] -= 1.5
        top = logits.sort(descending=True, stable=True)
        probs = torch.softmax(top.values[:case["top_k"]], 0)
        return {"logits": logits, "token": None, "top_ids": None, "top_probs": probs, "rng": None}
    if kind in ("layer_step", "layer_prefill"):
        first = case["pos"] if kind == "layer_step" else 0
        rope = _rope(first + s["x"].shape[0])
        k64, v64 = _first64(s["k_cache"], 0), _first64(s["v_cache"], 0)
        y, state, conv = _layer64(s["layer"], s["x"].to(F64), _first64(s["state"], 0), _first64(s["conv_buf"], 0),
                                  k64, v64, first, rope)
        return {"y": y, **{n: None if t is None else t.unsqueeze(0) for n, t in
                           (("state", state), ("conv_buf", conv), ("k_cache", k64), ("v_cache", v64))}}
    first = case["pos"] if kind == "model_step" else 0
    rope = _rope(s["k_cache"].shape[-2])
    picked = s["ids"].long()
    x = _dequant((s["embed"][0][picked], s["embed"][1][picked]))
    kept = {n: [] for n in ("state", "conv_buf", "k_cache", "v_cache")}
    for i in range(LAYERS):
        state, conv, k, v = (None if t is None else t.to(F64) for t in _layer_caches(s, i))
        x, state, conv = _layer64(_model_layer(seed, i), x, state, conv, k, v, first, rope)
        for n, t in (("state", state), ("conv_buf", conv), ("k_cache", k), ("v_cache", v)):
            if t is not None:
                kept[n].append(t)
    xn = _rms64(x[-1], 1 + s["final_norm"].to(F64))
    logits = torch.cat([_dequant((c, e)) @ xn for c, e in zip(s["embed"][0].split(32768), s["embed"][1].split(32768))])
    return {"logits": logits, **{n: torch.stack(t) for n, t in kept.items()}}
