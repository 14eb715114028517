"""Timed cases: the calls a program serving one sequence makes, at real sizes.

A serving program ingests a prompt (cold, or a new turn on top of a cached
prefix), then decodes token by token, or two tokens at a time when it verifies
a draft. The cases are the layers of that work through the op entry points,
plus two whole calls of the model. Widths are the 9B configuration's
(hidden 4096, intermediate 12288, vocabulary 248320, 16 q / 4 kv heads x 256,
Gated DeltaNet 16 k / 32 v heads x 128); token counts and contexts are what
varies in use, odd values among them.

Inputs, weights and states are made on the GPU from the seed. `exact` restates
each path in float64 with plain torch.
"""
from __future__ import annotations

import math

import torch

from peregrine_amd import ops
from peregrine_amd._lib import call
from peregrine_amd.device import init
from peregrine_amd.model import DeviceModel, ModelConfig, ModelState

HIDDEN, INTER, VOCAB = 4096, 12288, 248320
HEADS, KV_HEADS, HEAD_DIM, ROTARY, THETA = 16, 4, 256, 64, 1.0e7
CONV_DIM, KEY_DIM, VAL_DIM, HK, HV, DK = 8192, 2048, 4096, 16, 32, 128
EPS = 1e-6
MODEL_LAYERS = 4  # one period of the layer pattern: three GDN layers, one attention layer


def listed() -> list[dict]:
    return [
        # one decode token's recurrent layers between two attention layers
        {"name": "gdn_step", "kind": "gdn_decode", "layers": 3},
        # one decode token's attention layer in an ordinary chat, and near the largest context
        {"name": "attn_step_2k", "kind": "attn_decode", "context": 2047},
        {"name": "attn_step_60k", "kind": "attn_decode", "context": 60001},
        # one decode token's MLP block (add + norm, gate/up, down + residual)
        {"name": "mlp_step", "kind": "mlp_decode", "rows": 1, "inter": INTER},
        # logits of the two verified rows of a speculative step
        {"name": "head_verify", "kind": "head", "rows": 2, "vocab": VOCAB},
        # MLP block of a short chat turn, and of an ordinary prompt
        {"name": "mlp_turn", "kind": "mlp_prefill", "tokens": 43},
        {"name": "mlp_prompt", "kind": "mlp_prefill", "tokens": 1600},
        # Gated DeltaNet mixer of an ordinary prompt (conv, q/k norms and gates, recurrence, gated norm)
        {"name": "gdn_prompt", "kind": "gdn_prefill", "tokens": 1600, "history": True},
        # attention of an ordinary prompt, and of a late chunk of a long one
        {"name": "attn_prompt", "kind": "attn_prefill", "tokens": 1600, "prefix": 0},
        {"name": "attn_late_chunk", "kind": "attn_prefill", "tokens": 1021, "prefix": 15003},
        # a chat turn on a cached prefix: restore, prefill the new tokens, a few
        # sampled steps, then the logits of a two-token verify
        {"name": "model_turn", "kind": "model", "prefix": 700, "tokens": 40, "steps": 6},
        # a cold prompt, then the logits of a two-token verify
        {"name": "model_prompt", "kind": "model", "prefix": 0, "tokens": 1600, "steps": 0},
    ]


def _log_uniform(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng) -> dict:
    kind = rng.choice(["gdn_decode", "attn_decode", "mlp_decode", "head", "mlp_prefill", "mlp_prefill", "gdn_prefill",
                       "attn_prefill", "attn_prefill", "model"])
    if kind == "gdn_decode":
        return {"kind": kind, "layers": rng.randint(1, 20)}
    if kind == "attn_decode":
        return {"kind": kind, "context": _log_uniform(rng, 1, 60000)}
    if kind == "mlp_decode":
        return {"kind": kind, "rows": rng.randint(1, 2), "inter": 512 * rng.randint(4, INTER // 512)}
    if kind == "head":
        return {"kind": kind, "rows": rng.randint(1, 2), "vocab": 16 * rng.randint(2000, VOCAB // 16)}
    if kind == "mlp_prefill":
        return {"kind": kind, "tokens": _log_uniform(rng, 3, 1600)}
    if kind == "gdn_prefill":
        return {"kind": kind, "tokens": _log_uniform(rng, 3, 1600), "history": rng.random() < 0.5}
    if kind == "attn_prefill":
        tokens = _log_uniform(rng, 3, 2048)
        return {"kind": kind, "tokens": tokens,
                "prefix": 0 if rng.random() < 0.4 else _log_uniform(rng, 16, min(30000, 16000000 // tokens - tokens))}
    if rng.random() < 0.5:
        return {"kind": kind, "prefix": 0, "tokens": _log_uniform(rng, 5, 1500), "steps": 0}
    return {"kind": kind, "prefix": _log_uniform(rng, 16, 3000), "tokens": _log_uniform(rng, 3, 600),
            "steps": rng.randint(0, 8)}


# ---------------------------------------------------------------- inputs ----
class _Gen:
    """Seeded tensors on the GPU."""

    def __init__(self, seed: int) -> None:
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, shape, std: float = 1.0, mean: float = 0.0, dtype=torch.bfloat16):
        return (torch.randn(shape, generator=self.g, device="cuda") * std + mean).to(dtype)

    def uniform(self, shape, lo: float, hi: float, dtype=torch.bfloat16):
        return (torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo).to(dtype)

    def q4(self, out_dim: int, in_dim: int) -> dict:
        """Q4 weight words, scales and biases; dequantised values centred on zero."""
        w = torch.randint(-2 ** 31, 2 ** 31, (out_dim, in_dim // 8), generator=self.g, device="cuda", dtype=torch.int64)
        s = self.uniform((out_dim, in_dim // 64), 0.002, 0.02)
        b = (-7.5 * s.float() + self.normal(s.shape, 0.01, dtype=torch.float32)).to(torch.bfloat16)
        return {"w": w.to(torch.int32), "s": s, "b": b}


class _Dev:
    """A tensor as the op layer takes device memory: shape, address, bytes."""

    def __init__(self, t: torch.Tensor) -> None:
        self.t, self.shape, self.nbytes = t, tuple(t.shape), t.numel() * t.element_size()

    def __int__(self) -> int:
        return self.t.data_ptr()


def _linear(q: dict) -> ops.Q4Linear:
    return ops.Q4Linear(_Dev(q["w"]), _Dev(q["s"]), _Dev(q["b"]))


def _p(t) -> int:
    return t.data_ptr()


def _bf(*shape):
    return torch.empty(shape, device="cuda", dtype=torch.bfloat16)


def _stride(tokens: int) -> int:
    return (tokens + 255) // 256 * 256


def prepare(case: dict, seed: int) -> dict:
    init()
    st = _PREPARE[case["kind"]](case, _Gen(seed), seed)
    st["case"] = case
    torch.cuda.synchronize()  # the library's own streams do not wait for torch's
    return st


def run(st: dict):
    return _RUN[st["case"]["kind"]](st)


def exact(case: dict, seed: int):
    return _EXACT[case["kind"]](prepare(case, seed))


# ------------------------------------------------------------- GDN decode ---
def _prep_gdn_decode(case, g, seed):
    return {"layers": [{
        "recur": g.normal((HV, DK, DK), 0.1, dtype=torch.float32), "conv": g.normal((3, CONV_DIM), dtype=torch.float32),
        "x": g.normal((CONV_DIM,)), "w": g.normal((CONV_DIM, 4), 0.5), "a": g.normal((HV,)), "b": g.normal((HV,)),
        "A_log": g.normal((HV,), 0.5, dtype=torch.float32), "dt": g.normal((HV,), 0.5),
        "norm": g.normal((DK,), 0.1, 1.0), "z": g.normal((VAL_DIM,)), "c": _bf(CONV_DIM), "out": _bf(VAL_DIM),
    } for _ in range(case["layers"])]}


def _run_gdn_decode(st):
    for l in st["layers"]:
        ops.conv1d_silu_decode(_p(l["conv"]), _p(l["x"]), _p(l["w"]), _p(l["c"]), CONV_DIM)
        ops.gated_delta_decode_norm(_p(l["recur"]), _p(l["c"]), _p(l["a"]), _p(l["b"]), _p(l["A_log"]), _p(l["dt"]),
                                    _p(l["norm"]), _p(l["z"]), _p(l["out"]), EPS)
    return [{"out": l["out"], "recur": l["recur"], "conv": l["conv"]} for l in st["layers"]]


def _exact_gdn_decode(st):
    return [_ref_gdn(l, l["x"][None], l["a"][None], l["b"][None], l["z"][None], l["conv"], l["recur"], flat=True)
            for l in st["layers"]]


# ------------------------------------------------------- attention decode ---
def _prep_attn_decode(case, g, seed):
    # `context` tokens are cached; the step adds one
    stride = _stride(case["context"] + 1)
    return {"qp": g.normal((HEADS, 2 * HEAD_DIM), 2.0), "qw": g.normal((HEAD_DIM,), 0.1, 1.0),
            "k": g.normal((KV_HEADS, HEAD_DIM), 2.0), "v": g.normal((KV_HEADS, HEAD_DIM)),
            "kw": g.normal((HEAD_DIM,), 0.1, 1.0), "kc": g.normal((KV_HEADS, stride, HEAD_DIM)),
            "vc": g.normal((KV_HEADS, HEAD_DIM, stride)), "out": _bf(HEADS, HEAD_DIM), "stride": stride,
            "ws": torch.empty(ops.attn_step_workspace_bytes(stride), device="cuda", dtype=torch.uint8)}


def _run_attn_decode(st):
    n = st["case"]["context"]
    ops.attn_decode_step(_p(st["qp"]), _p(st["qw"]), _p(st["k"]), _p(st["v"]), _p(st["kw"]), _p(st["kc"]), _p(st["vc"]),
                         _p(st["out"]), _p(st["ws"]), st["stride"], n, n)
    return {"out": st["out"], "k": st["kc"][:, n], "v": st["vc"][:, :, n]}


def _exact_attn_decode(st):
    n = st["case"]["context"]
    out, kc, vc = _ref_attn(st, st["qp"][None], st["k"][None], st["v"][None], n)
    return {"out": out.reshape(HEADS, HEAD_DIM), "k": kc[:, n], "v": vc[:, :, n]}


# -------------------------------------------------------------- MLP decode --
def _prep_mlp(case, g, seed):
    rows, inter = case.get("rows", case.get("tokens")), case.get("inter", INTER)
    q = {"gate": g.q4(inter, HIDDEN), "up": g.q4(inter, HIDDEN), "down": g.q4(HIDDEN, inter)}
    return {"q": q, "gate": _linear(q["gate"]), "up": _linear(q["up"]), "down": _linear(q["down"]),
            "norm": g.normal((HIDDEN,), 0.1, 1.0), "x": g.normal((rows, HIDDEN)), "mix": g.normal((rows, HIDDEN)),
            "h": _bf(rows, HIDDEN), "n": _bf(rows, HIDDEN), "i": _bf(rows, inter), "out": _bf(rows, HIDDEN)}


def _run_mlp_decode(st):
    rows = st["case"]["rows"]
    ops.add_rmsnorm(_p(st["x"]), _p(st["mix"]), _p(st["norm"]), _p(st["h"]), _p(st["n"]), HIDDEN, rows, EPS)
    if rows == 1:
        ops.gate_up_silu(st["gate"], st["up"], _p(st["n"]), _p(st["i"]))
        st["down"].encode_bf16_fast_residual_add(_p(st["i"]), _p(st["h"]), _p(st["out"]))
    else:
        n, i, h, o = st["n"], st["i"], st["h"], st["out"]
        ops.gate_up_silu2(st["gate"], st["up"], _p(n[0]), _p(n[1]), _p(i[0]), _p(i[1]))
        st["down"].encode_bf16_fast_residual_add2(_p(i[0]), _p(i[1]), _p(h[0]), _p(h[1]), _p(o[0]), _p(o[1]))
    return {"out": st["out"], "h": st["h"]}


def _run_mlp_prefill(st):
    rows = st["case"]["tokens"]
    ops.add_rmsnorm(_p(st["x"]), _p(st["mix"]), _p(st["norm"]), _p(st["h"]), _p(st["n"]), HIDDEN, rows, EPS)
    ops.prefill_gate_up_silu(st["gate"], st["up"], _p(st["n"]), _p(st["i"]), rows)
    st["down"].encode_prefill_qmm_residual_add(_p(st["i"]), _p(st["h"]), _p(st["out"]), rows)
    return {"out": st["out"], "h": st["h"]}


def _exact_mlp(st):
    h = st["x"].double() + st["mix"].double()
    return {"out": h + _ref_mlp(_ref_norm(h, st["norm"]), st["q"]["gate"], st["q"]["up"], st["q"]["down"]), "h": h}


# -------------------------------------------------------------------- head --
def _prep_head(case, g, seed):
    q = g.q4(case["vocab"], HIDDEN)
    return {"q": q, "lin": ops.DecodeLayoutQ4(_linear(q)), "x": g.normal((case["rows"], HIDDEN)),
            "logits": _bf(case["rows"], case["vocab"])}


def _run_head(st):
    st["lin"].encode_bf16_fast(_p(st["x"]), _p(st["logits"]), st["case"]["rows"])
    return st["logits"]


def _exact_head(st):
    return _ref_q4(st["x"].double(), st["q"])


# ------------------------------------------------------------- GDN prefill --
def _prep_gdn_prefill(case, g, seed):
    T, f4 = case["tokens"], torch.float32
    return {"recur": g.normal((HV, DK, DK), 0.1, dtype=f4), "conv": g.normal((3, CONV_DIM), dtype=f4),
            "x": g.normal((T, CONV_DIM)), "w": g.normal((CONV_DIM, 4), 0.5), "a": g.normal((T, HV)),
            "b": g.normal((T, HV)), "A_log": g.normal((HV,), 0.5, dtype=f4), "dt": g.normal((HV,), 0.5),
            "norm": g.normal((DK,), 0.1, 1.0), "z": g.normal((T, VAL_DIM)), "c": _bf(T, CONV_DIM), "y": _bf(T, VAL_DIM),
            "out": _bf(T, VAL_DIM), "qn": torch.empty((T, KEY_DIM), device="cuda"),
            "kn": torch.empty((T, KEY_DIM), device="cuda"), "g": torch.empty((T, HV), device="cuda"),
            "beta": torch.empty((T, HV), device="cuda")}


def _run_gdn_prefill(st):
    T, hist = st["case"]["tokens"], st["case"]["history"]
    ops.conv1d_silu_prefill(_p(st["conv"]), _p(st["x"]), _p(st["w"]), _p(st["c"]), T, hist)
    ops.gated_delta_prefill_prepare(_p(st["c"]), _p(st["a"]), _p(st["b"]), _p(st["A_log"]), _p(st["dt"]), _p(st["qn"]),
                                    _p(st["kn"]), _p(st["g"]), _p(st["beta"]), T)
    ops.gated_delta_prefill(_p(st["recur"]), _p(st["qn"]), _p(st["kn"]), _p(st["c"]), _p(st["g"]), _p(st["beta"]),
                            _p(st["y"]), T, hist)
    ops.rmsnorm_gated(_p(st["y"]), _p(st["norm"]), _p(st["z"]), _p(st["out"]), DK, T * HV, EPS)
    return {"out": st["out"], "recur": st["recur"], "conv": st["conv"]}


def _exact_gdn_prefill(st):
    hist = 1.0 if st["case"]["history"] else 0.0
    return _ref_gdn(st, st["x"], st["a"], st["b"], st["z"], st["conv"] * hist, st["recur"] * hist)


# ------------------------------------------------------- attention prefill --
def _prep_attn_prefill(case, g, seed):
    T, P = case["tokens"], case["prefix"]
    stride = _stride(P + T)
    return {"qp": g.normal((T, HEADS, 2 * HEAD_DIM), 2.0), "qw": g.normal((HEAD_DIM,), 0.1, 1.0),
            "k": g.normal((T, KV_HEADS, HEAD_DIM), 2.0), "v": g.normal((T, KV_HEADS, HEAD_DIM)),
            "kw": g.normal((HEAD_DIM,), 0.1, 1.0), "kc": g.normal((KV_HEADS, stride, HEAD_DIM)),
            "vc": g.normal((KV_HEADS, HEAD_DIM, stride)), "q": _bf(T, HEADS, HEAD_DIM), "gate": _bf(T, HEADS, HEAD_DIM),
            "out": _bf(T, HEADS, HEAD_DIM), "stride": stride,
            "scores": torch.empty(ops.attn_prefill_scores_bytes(T, P), device="cuda", dtype=torch.uint8)}


def _run_attn_prefill(st):
    T, P, S = st["case"]["tokens"], st["case"]["prefix"], st["stride"]
    ops.attn_prefill_prepare(_p(st["qp"]), _p(st["qw"]), _p(st["k"]), _p(st["kw"]), _p(st["v"]), _p(st["q"]),
                             _p(st["gate"]), _p(st["kc"]), _p(st["vc"]), T, P, P, S)
    ops.attn_prefill(_p(st["q"]), _p(st["kc"]), _p(st["vc"]), _p(st["gate"]), _p(st["out"]), _p(st["scores"]), T, P, S)
    return {"out": st["out"], "k": st["kc"][:, P:P + T], "v": st["vc"][:, :, P:P + T]}


def _exact_attn_prefill(st):
    T, P = st["case"]["tokens"], st["case"]["prefix"]
    out, kc, vc = _ref_attn(st, st["qp"], st["k"], st["v"], P)
    return {"out": out, "k": kc[:, P:P + T], "v": vc[:, :, P:P + T]}


# ------------------------------------------------------------ whole model ---
class _Mem:
    """Library-owned device memory, for torch.as_tensor. The tensor holds this
    object, and so the handle that owns the memory, for as long as it lives."""

    def __init__(self, owner, ptr: int, shape, typestr: str) -> None:
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (ptr, False), "version": 2}


def _view(owner, ptr: int, shape, dtype) -> torch.Tensor:
    typestr = {torch.float32: "<f4", torch.int32: "<i4", torch.bfloat16: "<i2"}[dtype]
    t = torch.as_tensor(_Mem(owner, ptr, shape, typestr), device="cuda")
    return t.view(torch.bfloat16) if dtype == torch.bfloat16 else t


_DTYPES = {"U32": torch.int32, "BF16": torch.bfloat16, "F32": torch.float32}


def _tensor(model: DeviceModel, name: str) -> torch.Tensor:
    dtype, shape = model.tensor_info(name)
    return _view(model, model.tensor_ptr(name)[0], shape, _DTYPES[dtype])


def _q4_of(model: DeviceModel, base: str) -> dict:
    return {"w": _tensor(model, base + ".weight"), "s": _tensor(model, base + ".scales"),
            "b": _tensor(model, base + ".biases")}


def _state_tensor(state: ModelState, name: str, shape, dtype) -> torch.Tensor:
    import ctypes as C

    p, n = C.c_void_p(0), C.c_size_t(0)
    call("prg_model_state_tensor", state.handle, name.encode(), C.byref(p), C.byref(n))
    return _view(state, p.value, shape, dtype)


def _prep_model(case, g, seed):
    total = case["prefix"] + case["tokens"] + case["steps"] + 2
    cfg = ModelConfig(num_layers=MODEL_LAYERS)
    model = DeviceModel(cfg, seed=seed)
    model.prepare_dense()
    tokens = torch.randint(0, VOCAB, (total,), generator=g.g, device="cuda").cpu().numpy()
    work = ModelState(model, total)
    st = {"model": model, "work": work, "tokens": tokens, "saved": None,
          "lin": ops.DecodeLayoutQ4(_linear(_q4_of(model, "language_model.lm_head"))),
          "hidden": _bf(2, HIDDEN), "logits": _bf(2, VOCAB)}
    if case["prefix"]:
        st["saved"] = ModelState(model, case["prefix"])
        st["saved"].prefill(tokens[:case["prefix"]])
    else:  # the decode-layout copies are rewritten by the first call after a weight was looked up
        call("prg_model_prepare_decode", model.handle)
    outs = {}
    for i in range(MODEL_LAYERS):
        if cfg.is_linear(i):
            outs[f"recur{i}"] = _state_tensor(work, f"layers.{i}.recur", (HV, DK, DK), torch.float32)
            outs[f"conv{i}"] = _state_tensor(work, f"layers.{i}.conv", (3, CONV_DIM), torch.float32)
        else:
            kc = _state_tensor(work, f"layers.{i}.cache_k", (KV_HEADS, work.stride, HEAD_DIM), torch.bfloat16)
            vc = _state_tensor(work, f"layers.{i}.cache_v", (KV_HEADS, HEAD_DIM, work.stride), torch.bfloat16)
            outs[f"k{i}"], outs[f"v{i}"] = kc[:, :total], vc[:, :, :total]
    st["outs"] = outs
    return st


def _run_model(st):
    case, work, toks = st["case"], st["work"], st["tokens"]
    P, end = case["prefix"], case["prefix"] + case["tokens"]
    if P:
        work.copy_prefix_from(st["saved"], P)
        work.prefill_from(toks[:end], P)
    else:
        work.prefill(toks[:end])
    for pos in range(end, end + case["steps"]):
        work.forward_next_token(int(toks[pos]), pos)
    pos = end + case["steps"]
    work.forward_two_tokens(int(toks[pos]), int(toks[pos + 1]), pos, hidden_out=_p(st["hidden"]))
    st["lin"].encode_bf16_fast(_p(st["hidden"]), _p(st["logits"]), 2)
    return {"logits": st["logits"], **st["outs"]}


def _exact_model(st):
    model, L = st["model"], "language_model.model.layers."
    ids = torch.as_tensor(st["tokens"].astype("int64"), device="cuda")
    emb = _q4_of(model, "language_model.model.embed_tokens")
    x = _dequant({k: v[ids] for k, v in emb.items()})
    out = {}
    for i in range(MODEL_LAYERS):
        t = lambda n: _tensor(model, f"{L}{i}.{n}")  # noqa: E731
        q = lambda n: _q4_of(model, f"{L}{i}.{n}")  # noqa: E731
        n = _ref_norm(x, t("input_layernorm.weight"))
        if model.cfg.is_linear(i):
            a = "linear_attn."
            w = {"w": t(a + "conv1d.weight").reshape(CONV_DIM, 4), "A_log": t(a + "A_log"), "dt": t(a + "dt_bias"),
                 "norm": t(a + "norm.weight")}
            zero = torch.zeros((HV, DK, DK), device="cuda", dtype=torch.float64)
            r = _ref_gdn(w, _ref_q4(n, q(a + "in_proj_qkv")), _ref_q4(n, q(a + "in_proj_a")),
                         _ref_q4(n, q(a + "in_proj_b")), _ref_q4(n, q(a + "in_proj_z")), zero[0, :3, 0:1].expand(3, CONV_DIM), zero)
            out[f"recur{i}"], out[f"conv{i}"] = r["recur"], r["conv"]
            mix = _ref_q4(r["out"], q(a + "out_proj"))
        else:
            a, T = "self_attn.", len(ids)
            w = {"qw": t(a + "q_norm.weight"), "kw": t(a + "k_norm.weight"),
                 "kc": torch.zeros((KV_HEADS, T, HEAD_DIM), device="cuda"), "vc": torch.zeros((KV_HEADS, HEAD_DIM, T), device="cuda")}
            o, out[f"k{i}"], out[f"v{i}"] = _ref_attn(
                w, _ref_q4(n, q(a + "q_proj")).reshape(T, HEADS, 2 * HEAD_DIM),
                _ref_q4(n, q(a + "k_proj")).reshape(T, KV_HEADS, HEAD_DIM),
                _ref_q4(n, q(a + "v_proj")).reshape(T, KV_HEADS, HEAD_DIM), 0)
            mix = _ref_q4(o.reshape(T, -1), q(a + "o_proj"))
        x = x + mix
        n = _ref_norm(x, t("post_attention_layernorm.weight"))
        x = x + _ref_mlp(n, q("mlp.gate_proj"), q("mlp.up_proj"), q("mlp.down_proj"))
    n = _ref_norm(x[-2:], _tensor(model, "language_model.model.norm.weight"))
    return {"logits": _ref_q4(n, _q4_of(model, "language_model.lm_head")), **out}


# --------------------------------------------------- float64 restatements ---
def _dequant(q: dict) -> torch.Tensor:
    """s * q + b of packed rows, nibble j of word c = column 8 c + j."""
    sh = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    v = ((q["w"][:, :, None] >> sh) & 15).reshape(q["w"].shape[0], -1, 64).double()
    return (v * q["s"].double()[:, :, None] + q["b"].double()[:, :, None]).reshape(v.shape[0], -1)


def _ref_q4(x: torch.Tensor, q: dict) -> torch.Tensor:
    parts = [x @ _dequant({k: v[r:r + 16384] for k, v in q.items()}).T for r in range(0, q["w"].shape[0], 16384)]
    return torch.cat(parts, 1)


def _ref_norm(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _ref_mlp(n, gate, up, down):
    return _ref_q4(torch.nn.functional.silu(_ref_q4(n, gate)) * _ref_q4(n, up), down)


def _ref_gdn(w, x, a, b, z, conv, recur, flat=False):
    T = x.shape[0]
    seq = torch.cat([conv.double(), x.double()], 0)
    taps = w["w"].double()
    c = torch.nn.functional.silu(sum(seq[j:j + T] * taps[:, j] for j in range(4)))
    unit = lambda v: v * torch.rsqrt(v.square().sum(-1, keepdim=True) + EPS)  # noqa: E731
    rep = HV // HK
    q = (unit(c[:, :KEY_DIM].reshape(T, HK, DK)) / math.sqrt(DK)).repeat_interleave(rep, 1)
    k = unit(c[:, KEY_DIM:2 * KEY_DIM].reshape(T, HK, DK)).repeat_interleave(rep, 1)
    v = c[:, 2 * KEY_DIM:].reshape(T, HV, DK)
    decay = torch.exp(-torch.exp(w["A_log"].double()) * torch.nn.functional.softplus(a.double() + w["dt"].double()))
    beta = torch.sigmoid(b.double())
    S, y = recur.double().clone(), torch.empty_like(v)
    for t in range(T):
        S *= decay[t, :, None, None]
        delta = (v[t] - torch.bmm(S, k[t, :, :, None])[:, :, 0]) * beta[t, :, None]
        S += delta[:, :, None] * k[t, :, None, :]
        y[t] = torch.bmm(S, q[t, :, :, None])[:, :, 0]
    out = _ref_norm(y, w["norm"]).reshape(T, VAL_DIM) * torch.nn.functional.silu(z.double())
    return {"out": out[0] if flat else out, "recur": S, "conv": seq[T:T + 3]}


def _ref_rope(x: torch.Tensor, start: int) -> torch.Tensor:
    """Rotate dims [0, 64) of x [T, heads, 256], pairs (d, d + 32)."""
    half = ROTARY // 2
    d = torch.arange(half, device="cuda", dtype=torch.float64)
    pos = torch.arange(start, start + x.shape[0], device="cuda", dtype=torch.float64)
    th = (pos[:, None] * THETA ** (-2.0 * d / ROTARY))[:, None, :]
    lo, hi = x[..., :half], x[..., half:ROTARY]
    return torch.cat([lo * th.cos() - hi * th.sin(), hi * th.cos() + lo * th.sin(), x[..., ROTARY:]], -1)


def _ref_attn(w, qp, k, v, start):
    """T tokens at positions start.. over the caches' first `start` slots: context and the caches."""
    T, L, group = qp.shape[0], start + qp.shape[0], HEADS // KV_HEADS
    q = _ref_rope(_ref_norm(qp[..., :HEAD_DIM], w["qw"]), start) / math.sqrt(HEAD_DIM)
    kc, vc = w["kc"][:, :L].double(), w["vc"][:, :, :L].double()
    kc[:, start:] = _ref_rope(_ref_norm(k, w["kw"]), start).transpose(0, 1)
    vc[:, :, start:] = v.double().permute(1, 2, 0)
    out = torch.empty((T, HEADS, HEAD_DIM), device="cuda", dtype=torch.float64)
    cols = torch.arange(L, device="cuda")
    for h in range(HEADS):
        for r in range(0, T, 512):
            s = q[r:r + 512, h] @ kc[h // group].T
            hidden = cols[None, :] > start + r + torch.arange(s.shape[0], device="cuda")[:, None]
            p = torch.softmax(s.masked_fill(hidden, -math.inf), -1)
            out[r:r + 512, h] = p @ vc[h // group].T
    return out * torch.sigmoid(qp[..., HEAD_DIM:].double()), kc, vc


# ------------------------------------------------------ work and tolerance --
def _q4_bytes(n: int, k: int) -> int:
    return n * k // 2 + n * k // 16


def _attn_flops(T: int, P: int) -> float:
    return 4.0 * HEADS * HEAD_DIM * (T * P + T * (T + 1) / 2)


def work(case: dict) -> dict:
    kind = case["kind"]
    mlp = lambda rows, inter: {  # noqa: E731
        "bytes": 2 * _q4_bytes(inter, HIDDEN) + _q4_bytes(HIDDEN, inter) + 2 * 4 * rows * HIDDEN,
        "flops": 2.0 * rows * 3 * inter * HIDDEN}
    if kind == "gdn_decode":
        per = 2 * 4 * HV * DK * DK + 2 * 4 * 3 * CONV_DIM + 2 * 5 * CONV_DIM + 2 * 2 * VAL_DIM
        return {"bytes": per * case["layers"], "flops": 7.0 * HV * DK * DK * case["layers"]}
    if kind == "attn_decode":
        n = case["context"]
        return {"bytes": 2 * 2 * KV_HEADS * HEAD_DIM * (n + 2) + 2 * 3 * HEADS * HEAD_DIM, "flops": _attn_flops(1, n)}
    if kind == "mlp_decode":
        return mlp(case["rows"], case["inter"])
    if kind == "head":
        return {"bytes": _q4_bytes(case["vocab"], HIDDEN) + 2 * case["rows"] * (HIDDEN + case["vocab"]),
                "flops": 2.0 * case["rows"] * case["vocab"] * HIDDEN}
    if kind == "mlp_prefill":
        return mlp(case["tokens"], INTER)
    if kind == "gdn_prefill":
        T = case["tokens"]
        return {"bytes": 2 * T * (CONV_DIM + 2 * VAL_DIM + 2 * HV) + 2 * 4 * HV * DK * DK, "flops": 7.0 * T * HV * DK * DK}
    if kind == "attn_prefill":
        T, P = case["tokens"], case["prefix"]
        return {"bytes": 2 * T * HEADS * HEAD_DIM * 3 + 2 * 2 * KV_HEADS * HEAD_DIM * (P + 2 * T),
                "flops": _attn_flops(T, P)}
    # model: every layer's Q4 weights once for the prompt and once for each decode call, the head for each
    T, P, calls = case["tokens"], case["prefix"], case["steps"] + 1
    gdn = _q4_bytes(CONV_DIM + VAL_DIM + 2 * HV, HIDDEN) + _q4_bytes(HIDDEN, VAL_DIM)
    attn = _q4_bytes(2 * HEADS * HEAD_DIM + 2 * KV_HEADS * HEAD_DIM, HIDDEN) + _q4_bytes(HIDDEN, HEADS * HEAD_DIM)
    weights = MODEL_LAYERS * (2 * _q4_bytes(INTER, HIDDEN) + _q4_bytes(HIDDEN, INTER)) + (MODEL_LAYERS - 1) * gdn + attn
    head, state = _q4_bytes(VOCAB, HIDDEN), (MODEL_LAYERS - 1) * 4 * HV * DK * DK
    return {"bytes": weights * (1 + calls) + head * (1 + calls) + 2 * state * (1 + calls)
            + 2 * 2 * KV_HEADS * HEAD_DIM * (P + T) * (1 + calls),
            "flops": 2.0 * (T + calls + 1) * weights / 0.5625 + _attn_flops(T, P)}


def tolerance(case: dict):
    # About four times the distance from float64: bf16 stores a result to
    # 2^-9, and the values a path rounds on its way add to that. A whole model
    # compounds the rounding of its layers.
    return {"rel": {"gdn_decode": 0.012, "attn_decode": 0.015, "mlp_decode": 0.012, "head": 0.01, "mlp_prefill": 0.015,
                    "gdn_prefill": 0.015, "attn_prefill": 0.015, "model": 0.03}[case["kind"]]}


_PREPARE = {"gdn_decode": _prep_gdn_decode, "attn_decode": _prep_attn_decode, "mlp_decode": _prep_mlp,
            "head": _prep_head, "mlp_prefill": _prep_mlp, "gdn_prefill": _prep_gdn_prefill,
            "attn_prefill": _prep_attn_prefill, "model": _prep_model}
_RUN = {"gdn_decode": _run_gdn_decode, "attn_decode": _run_attn_decode, "mlp_decode": _run_mlp_decode,
        "head": _run_head, "mlp_prefill": _run_mlp_prefill, "gdn_prefill": _run_gdn_prefill,
        "attn_prefill": _run_attn_prefill, "model": _run_model}
_EXACT = {"gdn_decode": _exact_gdn_decode, "attn_decode": _exact_attn_decode, "mlp_decode": _exact_mlp,
          "head": _exact_head, "mlp_prefill": _exact_mlp, "gdn_prefill": _exact_gdn_prefill,
          "attn_prefill": _exact_attn_prefill, "model": _exact_model}
