"""The work that a program built on ``tilert_amd`` has it do, as timed cases: a decode step's
norms, projections, indexer, sparse attention and expert layers at one GPU's share, a prefill
chunk's norm and index keys, and the preparation of weights at load time.  Every ``run``
goes through the package's public operators on tensors that ``prepare`` laid out, with the weights
in the form a serving program keeps them (packed once at load), or as stored where the
operator takes that form.

Inputs are drawn on the GPU from the seed alone.  Weights have the distribution of a
block-quantised N(0, 0.02) matrix: e4m3fn codes of N(0, 112) (a 128 x 128 block's largest
magnitude is about four standard deviations, which the block scale maps to 448) and scales
around 0.02 * 4 / 448.  Activations are N(0, 1), norm weights U(0.9, 1.1), routing uniform.
"""
from __future__ import annotations

import math

import torch

from tilert_amd.common import linear
from tilert_amd.down_allreduce import down_allreduce
from tilert_amd.expert_down_allreduce import DownExperts, expert_down_allreduce
from tilert_amd.expert_sel_up_gate_silu import ROUTING, UpGateExperts, expert_select_up_gate_silu
from tilert_amd.flash_sparse_mla import flash_sparse_mla, softmax_scale
from tilert_amd.kernel import pack_weight, weight_dequant, weight_quant
from tilert_amd.layernorm_rope_rotate import layernorm_rope_rotate_ki
from tilert_amd.moe import LocalExperts, moe_forward
from tilert_amd.projo_wkvb import convert_projo_wkvb, projo_wkvb
from tilert_amd.projq_wqb import convert_projq_wqb, projq_wqb
from tilert_amd.projx import pack_wqkva, rmsnorm_projx_wqkva
from tilert_amd.rmsnorm import rmsnorm_quant
from tilert_amd.rmsnorm_projq_wqb import rmsnorm_projq_wqb_op
from tilert_amd.rmsnorm_up_gate_silu import rmsnorm_up_gate_silu
from tilert_amd.sparse_index import KI_PAGE_BYTES, KI_PAGE_KEYS, score_scale, sparse_index_topk, sparse_index_topk_fp8
from tilert_amd.sparse_index_v3 import sparse_index_topk_v3
from tilert_amd.unproj_o_allreduce import convert_unproj_o, unproj_o_allreduce

DEV = "cuda"
BF16, F32, F64, FP8 = torch.bfloat16, torch.float32, torch.float64, torch.float8_e4m3fn
EPS = 1e-6

# (K, N) of the dense layers: the MLP's up and down, wq_a, wq_b, wkv_a, wkv_b and wo at one
# GPU's share, the stacked wq_a + wkv_a, and GLM-5's wq_a
DENSE = [(7168, 18432), (18432, 7168), (7168, 1536), (1536, 3072), (7168, 576), (512, 4096), (2048, 7168),
         (7168, 2112), (6144, 2048)]
EXPERTS_TOTAL, EXPERTS_TOPK = 256, 8


def listed() -> list[dict]:
    return [
        # one token's hidden state before a layer: the smallest call of a decode step
        {"name": "norm_1", "kind": "norm", "rows": 1, "dim": 7168, "scale": "ref"},
        # a prefill chunk: the hidden rows normalised and quantised, its index keys written to the KI pages
        {"name": "prefill_4096", "kind": "prefill", "rows": 4096, "dim": 7168, "pos": 1000, "scale": "ref"},
        # the dense MLP's up projection for 4 tokens (one decode step with 3 draft tokens): the headline layer
        {"name": "up_4", "kind": "linear", "M": 4, "K": 7168, "N": 18432, "packed": True, "scale": "ref"},
        # its down projection at the largest batch the layer takes
        {"name": "down_256", "kind": "linear", "M": 256, "K": 18432, "N": 7168, "packed": True, "scale": "ref"},
        # the same layer on the checkpoint's own weight layout, with an odd batch
        {"name": "stored_up_100", "kind": "linear", "M": 100, "K": 7168, "N": 18432, "packed": False, "scale": "ref"},
        # an attention layer's projections at the 16-head share, 4 tokens
        {"name": "mla_proj_4", "kind": "mla_proj", "tokens": 4, "heads": 16},
        # an expert-parallel MoE layer (32 of 256 experts on the GPU), an ordinary step and the largest batch
        {"name": "moe_ep_4", "kind": "moe_ep", "M": 4, "D": 7168, "I": 2048, "n_local": 32},
        {"name": "moe_ep_16", "kind": "moe_ep", "M": 16, "D": 7168, "I": 2048, "n_local": 32},
        # the tensor-parallel layout: a routed layer with its shared expert, then a dense layer's share
        {"name": "mlp_tp_4", "kind": "mlp_tp", "tokens": 4, "arch": "deepseek_v3_2", "n_routed": 256, "chunks": 9},
        # the indexer over a 128K context with the fp8 key cache, 2048 positions selected
        {"name": "index_128k", "kind": "index", "dtype": "fp8", "M": 4, "H": 64, "L": 131072, "topk": 2048},
        # attention over that selection
        {"name": "sparse_mla_4", "kind": "sparse_mla", "tokens": 4, "heads": 16, "topk": 2048, "rows": 131072},
        # load time: a bf16 weight quantised, packed for the GEMM, and dequantised again
        {"name": "load_7168_18432", "kind": "load", "N": 18432, "K": 7168, "dtype": "bf16"},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(("norm", "prefill", "linear", "linear", "mla_proj", "moe_ep", "moe_ep", "mlp_tp", "index",
                       "sparse_mla", "load"))
    scale = rng.choice(("ref", "ref", "ue8m0", "div"))
    if kind == "norm":  # from one token to a batch
        return {"kind": kind, "rows": _log_int(rng, 1, 512), "dim": rng.choice((7168, 6144, 2048, 1536)), "scale": scale}
    if kind == "prefill":
        return {"kind": kind, "rows": _log_int(rng, 200, 4096), "dim": rng.choice((7168, 6144)),
                "pos": rng.randrange(0, 4096), "scale": scale}
    if kind == "linear":
        K, N = rng.choice(DENSE)
        return {"kind": kind, "M": _log_int(rng, 1, 256), "K": K, "N": N, "packed": rng.random() < 0.6, "scale": scale}
    if kind == "mla_proj":
        return {"kind": kind, "tokens": rng.choice((1, 2, 4)), "heads": rng.choice((8, 16))}
    if kind == "moe_ep":
        return {"kind": kind, "M": rng.randint(1, 16), "D": rng.choice((7168, 6144, 4096)),
                "I": 128 * rng.randint(4, 16), "n_local": rng.choice((16, 32))}
    if kind == "mlp_tp":
        return {"kind": kind, "tokens": rng.randint(1, 4), "arch": rng.choice(("deepseek_v3_2", "glm_5")),
                "n_routed": rng.choice((64, 128, 256)), "chunks": rng.randint(2, 9)}
    if kind == "index":
        dtype, H = rng.choice((("fp8", 64), ("bf16", 64), ("bf16", 32)))
        return {"kind": kind, "dtype": dtype, "M": rng.randint(1, 4), "H": H, "L": _log_int(rng, 2100, 163840), "topk": 2048}
    if kind == "sparse_mla":
        rows = _log_int(rng, 1000, 131072)
        return {"kind": kind, "tokens": rng.randint(1, 4), "heads": rng.choice((8, 10, 16, 20)),
                "topk": min(rows, rng.choice((512, 1000, 2048))), "rows": rows}
    return {"kind": kind, "N": 16 * _log_int(rng, 4, 1152), "K": 512 * rng.randint(1, 14),
            "dtype": rng.choice(("bf16", "f32"))}


# ------------------------------------------------------------------------------- inputs
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, dtype=BF16):
    return torch.randn(*shape, generator=g, device=DEV, dtype=dtype)


def _uniform(g, *shape, lo=0.9, hi=1.1):
    return torch.rand(*shape, generator=g, device=DEV, dtype=F32) * (hi - lo) + lo


def _weight(g, *shape):
    """An e4m3fn weight [..., N, K] and its fp32 scales [..., ceil(N/128), K/128]."""
    q = (_randn(g, *shape) * 112.0).clamp_(-448.0, 448.0).to(FP8)
    *lead, N, K = shape
    return q, _uniform(g, *lead, -(-N // 128), K // 128) * (0.02 * 4 / 448)


def _scale_fmt(case):
    return {"ref": None, "ue8m0": "ue8m0", "div": "div"}[case["scale"]]


def _norm_inputs(case, seed):
    g = _gen(seed)
    return {"x": _randn(g, case["rows"], case["dim"]), "gamma": _uniform(g, case["dim"])}


def _key_inputs(case, seed):
    g = _gen(seed + 7919)
    rows, pos = case["rows"], case["pos"]
    x = _randn(g, 1, rows, 128)
    ang = torch.arange(pos, pos + rows, device=DEV, dtype=F64)[:, None] * \
        (10000.0 ** (-torch.arange(32, device=DEV, dtype=F64) / 32))[None]
    freqs = torch.stack([ang.cos(), ang.sin()], -1).to(F32).reshape(rows, 1, 64).contiguous()
    return {"kx": x, "weight": _uniform(g, 128), "bias": _randn(g, 128, dtype=F32) * 0.1, "freqs": freqs}


def _linear_inputs(case, seed):
    g = _gen(seed)
    w, s = _weight(g, case["N"], case["K"])
    return {"x": _randn(g, case["M"], case["K"]), "w": w, "s": s}


def _mla_inputs(case, seed):
    g = _gen(seed)
    t, H = case["tokens"], case["heads"]
    d = {"x": _randn(g, 1, t, 7168), "gamma": _uniform(g, 7168), "gamma_q": _uniform(g, 1536),
         "o_lat": _randn(g, 1, t, H, 512)}
    for name, shape in (("wq_a", (1536, 7168)), ("wkv_a", (576, 7168)), ("wq_b", (H * 192, 1536)),
                        ("wkv_b", (H * 256, 512)), ("wo", (7168, H * 128))):
        d[name], d[name + "_s"] = _weight(g, *shape)
    return d


def _experts(g, E, I, D):
    d = {}
    for name, shape in (("gate", (E, I, D)), ("up", (E, I, D)), ("down", (E, D, I))):
        d[name], d[name + "_s"] = _weight(g, *shape)
    return d


def _moe_inputs(case, seed):
    g = _gen(seed)
    M = case["M"]
    d = _experts(g, case["n_local"], case["I"], case["D"])
    d["x"] = _randn(g, M, case["D"])
    d["idx"] = torch.rand(M, EXPERTS_TOTAL, generator=g, device=DEV).topk(EXPERTS_TOPK, dim=-1).indices.to(torch.int32).contiguous()
    d["w"] = torch.softmax(_randn(g, M, EXPERTS_TOPK, dtype=F32), -1)
    return d


def _tp_dims(case):
    return (7168, 256) if case["arch"] == "deepseek_v3_2" else (6144, 256)


def _tp_inputs(case, seed):
    g = _gen(seed)
    D, I = _tp_dims(case)
    d = _experts(g, 1 + case["n_routed"], I, D)
    d.update({"dense_" + k: v for k, v in _experts(g, case["chunks"], I, D).items()})
    t = case["tokens"]
    d.update(x=_randn(g, 1, t, D), x2=_randn(g, 1, t, D), gamma=_uniform(g, D),
             logits=_randn(g, 1, t, case["n_routed"], dtype=F32), bias=_randn(g, case["n_routed"], dtype=F32) * 0.05)
    return d


def _per_row_fp8(x, dims):
    s = (x.abs().amax(dim=dims, keepdim=True).clamp_min(1e-4) / 448.0)
    return (x / s).clamp_(-448.0, 448.0).to(FP8), s.reshape(x.shape[0]).contiguous()


def _index_inputs(case, seed):
    g = _gen(seed)
    M, H, L = case["M"], case["H"], case["L"]
    q, k = _randn(g, M, H, 128, dtype=F32), _randn(g, L, 128, dtype=F32)
    d = {"w": _randn(g, M, H) * 0.125}
    if case["dtype"] == "fp8":
        d["q"], d["q_s"] = _per_row_fp8(q, (1, 2))
        d["k"], d["k_s"] = _per_row_fp8(k, (1,))
    else:
        d["q"], d["k"] = q.to(BF16), k.to(BF16)
    return d


def _attn_inputs(case, seed):
    g = _gen(seed)
    t, H, T, k = case["tokens"], case["heads"], case["rows"], case["topk"]
    idx = torch.stack([torch.rand(T, generator=g, device=DEV).topk(k).indices.sort().values for _ in range(t)])
    return {"q": _randn(g, 1, t, H, 512), "q_pe": _randn(g, 1, t, H, 64), "kv": _randn(g, 1, T, 512),
            "pe": _randn(g, 1, T, 64), "idx": idx.to(torch.int32).reshape(1, t, k).contiguous()}


def _load_inputs(case, seed):
    w = _randn(_gen(seed), case["N"], case["K"], dtype=F32) * 0.02
    return {"w": w.to(BF16) if case["dtype"] == "bf16" else w}


# ------------------------------------------------------------------------------ prepare
def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    st = {"case": case}
    if kind in ("norm", "prefill"):
        st.update(_norm_inputs(case, seed))
        rows, dim = case["rows"], case["dim"]
        st.update(y=torch.empty(rows, dim, dtype=BF16, device=DEV), y8=torch.empty(rows, dim, dtype=FP8, device=DEV),
                  ys=torch.empty(rows, dim // 128, dtype=F32, device=DEV), logs=torch.zeros(1, device=DEV))
        if kind == "prefill":
            st.update(_key_inputs(case, seed))
            st["pages"] = torch.zeros(-(-(case["pos"] + rows) // KI_PAGE_KEYS), KI_PAGE_BYTES, dtype=torch.uint8, device=DEV)
            st["pos"] = torch.tensor([case["pos"]], dtype=torch.int32, device=DEV)
    elif kind == "linear":
        d = _linear_inputs(case, seed)
        st["x"] = d["x"]
        st["w"], st["s"] = (pack_weight(d["w"], d["s"]), None) if case["packed"] else (d["w"], d["s"])
    elif kind == "mla_proj":
        d = _mla_inputs(case, seed)
        t, H = case["tokens"], case["heads"]
        st.update({k: d[k] for k in ("x", "gamma", "gamma_q", "o_lat")})
        st.update(wqkva=pack_wqkva(d["wq_a"], d["wq_a_s"], d["wkv_a"], d["wkv_a_s"], 512),
                  wq_b=pack_weight(d["wq_b"], d["wq_b_s"]), k_up=convert_projq_wqb(d["wkv_b"], d["wkv_b_s"], H),
                  v_up=convert_projo_wkvb(d["wkv_b"], d["wkv_b_s"], H), wo=convert_unproj_o(d["wo"], d["wo_s"]))
        for name, shape in (("q", (1, t, 1536)), ("kv", (1, t, 512)), ("q_nope", (1, t, H, 128)),
                            ("q_pe", (1, t, H, 64)), ("q_lat", (1, t, H, 512)), ("o", (1, t, H, 128)), ("out", (1, t, 7168))):
            st[name] = torch.empty(*shape, dtype=BF16, device=DEV)
        st["pe"] = torch.zeros(1, 64, 64, dtype=BF16, device=DEV)
        st["pos"] = torch.tensor([17], dtype=torch.int32, device=DEV)
    elif kind == "moe_ep":
        d = _moe_inputs(case, seed)
        st.update({k: d[k] for k in ("x", "idx", "w")})
        st["experts"] = LocalExperts(*(d[k] for k in ("gate", "gate_s", "up", "up_s", "down", "down_s")))
    elif kind == "mlp_tp":
        d = _tp_inputs(case, seed)
        st.update({k: d[k] for k in ("x", "x2", "gamma", "logits", "bias")})
        for pre in ("", "dense_"):
            st[pre + "up_gate"] = UpGateExperts(*(d[pre + k] for k in ("gate", "gate_s", "up", "up_s")))
            st[pre + "down"] = DownExperts(d[pre + "down"], d[pre + "down_s"])
        t, (D, I) = case["tokens"], _tp_dims(case)
        topk = ROUTING[case["arch"]][2]
        st.update(h=torch.empty(1, t, 1 + topk, I, dtype=BF16, device=DEV), probs=torch.empty(1, t, topk, dtype=F32, device=DEV),
                  idx=torch.empty(1, t, topk, dtype=torch.int32, device=DEV), y=torch.empty(1, t, D, dtype=BF16, device=DEV),
                  h2=torch.empty(1, t, case["chunks"], I, dtype=BF16, device=DEV), y2=torch.empty(1, t, D, dtype=BF16, device=DEV))
    elif kind == "index":
        st.update(_index_inputs(case, seed))
        M, L = case["M"], case["L"]
        st.update(logits=torch.empty(M, -(-L // 4) * 4, dtype=F32, device=DEV).fill_(-math.inf),
                  indices=torch.empty(M, case["topk"], dtype=torch.int32, device=DEV))
    elif kind == "sparse_mla":
        st.update(_attn_inputs(case, seed))
        st.update(out=torch.empty(1, case["tokens"], case["heads"], 512, dtype=BF16, device=DEV),
                  pos=torch.tensor([case["rows"] - case["tokens"]], dtype=torch.int32, device=DEV))
    else:
        st.update(_load_inputs(case, seed))
    return st


# ---------------------------------------------------------------------------------- run
def run(st: dict):
    case = st["case"]
    kind = case["kind"]
    if kind in ("norm", "prefill"):
        rmsnorm_quant(st["x"], st["gamma"], st["y"], st["y8"], st["ys"], st["logs"], model_arch="deepseek_v3_2",
                      scale_fmt=_scale_fmt(case))
        if kind == "norm":
            return st["y"], st["y8"], st["ys"]
        layernorm_rope_rotate_ki(st["kx"], st["pos"], st["pages"], st["weight"], st["bias"], st["freqs"])
        return st["y"], st["y8"], st["ys"], st["pages"]
    if kind == "linear":
        return linear(st["x"], st["w"], st["s"], scale_fmt=_scale_fmt(case))
    if kind == "mla_proj":
        arch = "deepseek_v3_2"
        rmsnorm_projx_wqkva(st["x"], st["gamma"], st["wqkva"], st["pos"], st["q"], st["kv"], st["pe"], model_arch=arch)
        rmsnorm_projq_wqb_op(st["q"], st["wq_b"], None, st["gamma_q"], st["q_nope"], st["q_pe"], None, "bf16mma", arch)
        projq_wqb(st["q_nope"], st["k_up"], None, st["q_lat"], model_arch=arch)
        projo_wkvb(st["o_lat"], st["v_up"], None, st["o"])
        unproj_o_allreduce(st["o"], st["wo"], None, st["x"], 0, st["out"])
        return {k: st[k] for k in ("q", "kv", "pe", "q_nope", "q_pe", "q_lat", "o", "out")}
    if kind == "moe_ep":
        return moe_forward(st["x"], st["experts"], st["idx"], st["w"])
    if kind == "mlp_tp":
        arch = case["arch"]
        expert_select_up_gate_silu(st["x"], st["logits"], st["bias"], st["up_gate"], st["h"], st["probs"], st["idx"],
                                   model_arch=arch)
        expert_down_allreduce(st["h"], st["down"], None, st["idx"], st["probs"], st["x"], 0, st["y"], model_arch=arch)
        rmsnorm_up_gate_silu(st["x2"], st["gamma"], st["dense_up_gate"], st["h2"], model_arch=arch)
        down_allreduce(st["h2"], st["dense_down"], None, st["x2"], 0, st["y2"], model_arch=arch)
        return {k: st[k] for k in ("h", "probs", "idx", "y", "h2", "y2")}
    if kind == "index":
        args = (st["w"], st["logits"], st["indices"], case["L"] - case["M"])
        if case["dtype"] == "fp8":
            sparse_index_topk_fp8(st["q"], st["q_s"], st["k"], st["k_s"], *args)
        else:
            (sparse_index_topk if case["H"] == 64 else sparse_index_topk_v3)(st["q"], st["k"], *args)
        return st["logits"], st["indices"]
    if kind == "sparse_mla":
        lse, lse_acc, out_acc = flash_sparse_mla(st["q"], st["q_pe"], st["kv"], st["pe"], st["idx"], st["pos"], st["out"],
                                                 None, model_arch="deepseek_v3_2")
        n = -(-case["topk"] // 64)  # the splits that a selection of this length fills
        return st["out"], lse, lse_acc[..., :n], out_acc[..., :n, :]
    q, s = weight_quant(st["w"])
    packed = pack_weight(q, s)
    return q, s, packed.data, weight_dequant(q, s)


# --------------------------------------------------------------------------------- work
def _hits(M, n_local):
    return n_local * (1.0 - (1.0 - EXPERTS_TOPK / EXPERTS_TOTAL) ** M)


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("norm", "prefill"):
        rows, dim = case["rows"], case["dim"]
        b = rows * dim * 5 + rows * dim // 32 + dim * 4
        f = 8.0 * rows * dim
        if kind == "prefill":
            b += rows * (256 + 256 + 132)
            f += rows * 128 * 24.0
        return {"bytes": b, "flops": f}
    if kind == "linear":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": N * K * (1 + 4 / 16384) + M * K * 2 + M * N * 2, "flops": 2.0 * M * N * K}
    if kind == "mla_proj":
        t, H = case["tokens"], case["heads"]
        w = 2112 * 7168 + H * 192 * 1536 + H * 256 * 512 + 7168 * H * 128
        return {"bytes": w * (1 + 4 / 16384) + t * 2 * (2 * 7168 + 2 * 2112 + 2 * H * 192 + 2 * H * 512 + H * 128 + 2 * 7168),
                "flops": 2.0 * t * w}
    if kind == "moe_ep":
        M, D, I, n = case["M"], case["D"], case["I"], case["n_local"]
        return {"bytes": _hits(M, n) * 3 * D * I * (1 + 4 / 16384) + M * D * 4 + M * EXPERTS_TOPK * 8,
                "flops": 2.0 * M * EXPERTS_TOPK * n / EXPERTS_TOTAL * 3 * D * I}
    if kind == "mlp_tp":
        t, (D, I), E = case["tokens"], _tp_dims(case), case["n_routed"]
        hit = 1 + E * (1.0 - (1.0 - 8 / E) ** t) + case["chunks"]
        return {"bytes": hit * 3 * D * I * (1 + 4 / 16384) + t * (D * 8 + 4 * E + 2 * (9 + case["chunks"]) * I),
                "flops": 2.0 * t * (9 + case["chunks"]) * 3 * D * I}
    if kind == "index":
        M, H, L = case["M"], case["H"], case["L"]
        e = 1 if case["dtype"] == "fp8" else 2
        return {"bytes": L * (128 * e + (4 if e == 1 else 0)) + M * H * (128 * e + 2) + M * L * 4 + M * case["topk"] * 4,
                "flops": 2.0 * M * H * L * 129}
    if kind == "sparse_mla":
        t, H, k, T = case["tokens"], case["heads"], case["topk"], case["rows"]
        n = -(-k // 64)
        seen = T * (1.0 - (1.0 - k / T) ** t)
        return {"bytes": seen * 1152 + t * (k * 4 + H * (1152 + 1024 + n * 2052 + 4)), "flops": 2.0 * t * k * H * 1088}
    N, K = case["N"], case["K"]
    e = 2 if case["dtype"] == "bf16" else 4
    # quantised: w in, q and s out; packed: q in and out; dequantised: q in, fp32 out
    return {"bytes": N * K * (e + 1 + 2 + 5) + 2 * 4 * N * K / 16384, "flops": 3.0 * N * K}


def tolerance(case: dict):
    kind = case["kind"]
    if kind == "load":  # one IEEE division and one rounding per value, one fp32 product: every step is defined
        return "exact"
    if kind in ("norm", "prefill"):
        # another order of the fp32 sum moves a few bf16 roundings, and through them e4m3 codes (1/8 apart); the same
        # for the index keys' bytes
        return {"rel": 4e-3, "max": 0.13, "differ": 0.01}
    if kind == "index":  # fp32 scores over the matrix cores' products (1.5e-5 off exact in fp8); equal scores may change places
        return {"rel": 6e-5, "max": 1e-3, "differ": 0.01}
    if kind == "sparse_mla":  # bf16 probabilities: 2e-3 off exact
        return {"rel": 8e-3, "max": 0.05}
    return {"rel": 7e-3, "max": 0.04}  # bf16 results: 1.7e-3 off exact


# -------------------------------------------------------------------------------- exact
def _bf16(x):
    return x.to(BF16).to(F64)


def _deq(q, s, bf16=False):
    """fp8 weights [..., N, K] times their block scales, in fp64 (rounded to bf16 first where the operator
    defines its weights so)."""
    N, K = q.shape[-2:]
    if bf16:
        sc = s.repeat_interleave(128, -2)[..., :N, :].repeat_interleave(128, -1)
        return (q.to(F32) * sc).to(BF16).to(F64)
    return q.to(F64) * s.to(F64).repeat_interleave(128, -2)[..., :N, :].repeat_interleave(128, -1)


def _quant(x, fmt):
    """act_quant by its definition (fp32 scale and quotient): codes and scales, as fp64."""
    g = x.to(F32).reshape(*x.shape[:-1], -1, 128)
    amax = g.abs().amax(-1, keepdim=True).clamp_min(1e-4)
    if fmt == "ref":
        s = amax * torch.tensor(1.0 / 448.0, dtype=F32, device=x.device)
    elif fmt == "div":
        s = amax / torch.full_like(amax, 448.0)  # (a division by a Python number multiplies by its reciprocal)
    else:
        m, e = torch.frexp(amax * torch.tensor(1.0 / 448.0, dtype=F32, device=x.device))
        s = torch.ldexp(torch.ones_like(m), torch.where(m == 0.5, e - 1, e))
    q = (g / s).clamp(-448.0, 448.0).to(FP8)
    return q.to(F64).reshape(x.shape), s.squeeze(-1).to(F64)


def _rms(x, gamma):
    x = x.to(F64)
    return _bf16(x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gamma.to(F64))


def _qlinear(x, w, s, fmt):
    q, xs = _quant(x, fmt)
    return (q * xs.repeat_interleave(128, -1)) @ _deq(w, s).T


def _swiglu(x, gate, up):
    g = x @ gate.T
    return g / (1.0 + torch.exp(-g)) * (x @ up.T)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("norm", "prefill"):
        d = _norm_inputs(case, seed)
        y = _rms(d["x"], d["gamma"])
        q, s = _quant(y, case["scale"])
        return (y, q, s) if kind == "norm" else (y, q, s, None)
    if kind == "linear":
        d = _linear_inputs(case, seed)
        return _qlinear(d["x"], d["w"], d["s"], case["scale"])
    if kind == "mla_proj":
        d = _mla_inputs(case, seed)
        H = case["heads"]
        xn = _rms(d["x"], d["gamma"])
        q = _qlinear(xn, d["wq_a"], d["wq_a_s"], "ref")
        lat = _qlinear(xn, d["wkv_a"], d["wkv_a_s"], "ref")
        pe = torch.zeros(1, 64, 64, dtype=F64, device=DEV)
        pe[:, 17:17 + case["tokens"]] = lat[..., 512:]
        qb = (_rms(_bf16(q), d["gamma_q"]) @ _deq(d["wq_b"], d["wq_b_s"], True).T).reshape(1, -1, H, 192)
        kv_b = _deq(d["wkv_b"], d["wkv_b_s"], True).reshape(H, 256, 512)
        q_lat = torch.stack([_bf16(qb[0, :, h, :128]) @ kv_b[h, :128] for h in range(H)], 1)[None]
        o = torch.stack([d["o_lat"][0, :, h].to(F64) @ kv_b[h, 128:].T for h in range(H)], 1)[None]
        out = _bf16(o).reshape(1, -1, H * 128) @ _deq(d["wo"], d["wo_s"], True).T + d["x"].to(F64)
        return {"q": q, "kv": lat[..., :512], "pe": pe, "q_nope": qb[..., :128], "q_pe": qb[..., 128:], "q_lat": q_lat,
                "o": o, "out": out}
    if kind == "moe_ep":
        d = _moe_inputs(case, seed)
        y = torch.zeros(case["M"], case["D"], dtype=F64, device=DEV)
        x = d["x"].to(F64)
        for e in range(case["n_local"]):
            t, k = (d["idx"] == e).nonzero(as_tuple=True)
            if t.numel():
                gate, up, down = (_deq(d[n][e], d[n + "_s"][e], True) for n in ("gate", "up", "down"))
                y[t] += d["w"][t, k].to(F64)[:, None] * (_bf16(_swiglu(x[t], gate, up)) @ down.T)
        return y
    if kind == "mlp_tp":
        d = _tp_inputs(case, seed)
        n_groups, topk_groups, topk, route_scale = ROUTING[case["arch"]]
        t, (D, I), E = case["tokens"], _tp_dims(case), case["n_routed"]
        s = torch.sigmoid(d["logits"][0].to(F64))
        biased = s + d["bias"].to(F64)
        if n_groups > 1:
            best = biased.reshape(t, n_groups, -1).topk(2, -1).values.sum(-1).topk(topk_groups, -1).indices
            keep = torch.zeros(t, n_groups, dtype=torch.bool, device=DEV).scatter_(1, best, True)
            biased = biased.masked_fill(~keep.repeat_interleave(E // n_groups, 1), -math.inf)
        idx = biased.topk(topk, -1).indices
        probs = s.gather(1, idx)
        probs = probs / probs.sum(-1, keepdim=True) * route_scale
        x, x2 = d["x"][0].to(F64), d["x2"][0].to(F64)
        h, y = torch.empty(t, 1 + topk, I, dtype=F64, device=DEV), x.clone()
        for i in range(t):
            for p in range(1 + topk):
                e = 0 if p == 0 else 1 + int(idx[i, p - 1])
                gate, up, down = (_deq(d[n][e], d[n + "_s"][e], True) for n in ("gate", "up", "down"))
                h[i, p] = _swiglu(x[i], gate, up)
                y[i] += (1.0 if p == 0 else probs[i, p - 1]) * (_bf16(h[i, p]) @ down.T)
        xn, h2, y2 = _rms(x2, d["gamma"]), torch.empty(t, case["chunks"], I, dtype=F64, device=DEV), x2.clone()
        for c in range(case["chunks"]):
            gate, up, down = (_deq(d["dense_" + n][c], d["dense_" + n + "_s"][c], True) for n in ("gate", "up", "down"))
            h2[:, c] = _swiglu(xn, gate, up)
            y2 += _bf16(h2[:, c]) @ down.T
        return {"h": h[None], "probs": probs[None], "idx": None, "y": y[None], "h2": h2[None], "y2": y2[None]}
    if kind == "index":
        d = _index_inputs(case, seed)
        M, H, L = case["M"], case["H"], case["L"]
        q, k = d["q"].to(F64), d["k"].to(F64)
        if case["dtype"] == "fp8":
            q, k = q * d["q_s"].to(F64)[:, None, None], k * d["k_s"].to(F64)[:, None]
        out = torch.full((M, -(-L // 4) * 4), -math.inf, dtype=F64, device=DEV)
        for t in range(M):
            n = L - M + t + 1
            out[t, :n] = d["w"][t].to(F64) @ (q[t] @ k[:n].T).relu()
        return (out if case["dtype"] == "fp8" else out * score_scale(H)), None
    if kind == "sparse_mla":
        d = _attn_inputs(case, seed)
        t, H, T, k = case["tokens"], case["heads"], case["rows"], case["topk"]
        n = -(-k // 64)
        out, lse = torch.empty(1, t, H, 512, dtype=F64, device=DEV), torch.empty(1, t, H, dtype=F64, device=DEV)
        lse_acc, acc = torch.full((1, t, H, n), -math.inf, dtype=F64, device=DEV), torch.zeros(1, t, H, n, 512, dtype=F64, device=DEV)
        for i in range(t):
            sel = d["idx"][0, i].long()
            kv, pe = d["kv"][0, sel].to(F64), d["pe"][0, sel].to(F64)
            s = (d["q"][0, i].to(F64) @ kv.T + d["q_pe"][0, i].to(F64) @ pe.T) * softmax_scale("deepseek_v3_2")
            if t > 1:
                s = s.masked_fill((sel > T - t + i)[None], -math.inf)
            for j in range(n):
                sj = s[:, 64 * j:64 * j + 64]
                lse_acc[0, i, :, j] = torch.logsumexp(sj, -1)
                acc[0, i, :, j] = torch.nan_to_num(torch.softmax(sj, -1)) @ kv[64 * j:64 * j + 64]
            lse[0, i] = torch.logsumexp(s, -1)
            out[0, i] = torch.softmax(s, -1) @ kv
        return out, lse, lse_acc, acc
    w = _load_inputs(case, seed)["w"].to(F32)
    N, K = w.shape
    p = torch.zeros(-(-N // 128) * 128, K, device=DEV)
    p[:N] = w
    amax = p.reshape(-1, 128, K // 128, 128).abs().amax((1, 3))
    s = torch.where(amax > 0, amax / torch.full_like(amax, 448.0), torch.ones_like(amax))
    full = s.repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)
    q = (w / full).clamp(-448.0, 448.0).to(FP8)
    return q.to(F64), s.to(F64), None, (q.to(F32) * full).to(F64)
