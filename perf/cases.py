"""Performance cases: the work a user has this library do, through its public
entry points, from the smallest call to a whole prefill.

A case names a kind of call and its sizes:

  linear      one quantized projection (``ops.quantized_matmul``), called eagerly
  mlp         a layer's MLP half through the region API: the gate/up + SwiGLU
              region, then the down projection + residual + RMSNorm region
  attention   causal GQA attention over a KV cache
              (``ops.scaled_dot_product_attention``): a prompt, a chunk of one
              behind a cached prefix, or one decode token
  qwen_layer  one Qwen3-4B-shaped decoder layer with its regions installed,
              captured by ``GraphWrapper`` as a serving program delivers it
  lfm2_layer  one LFM2-1.2B-shaped layer (short-conv or attention), likewise
  qwen_model  a Qwen3-4B-shaped model of four layers with its embedding and
              full-width lm_head, likewise: prefill or a decode step. Four, not
              36: a last-place difference in one layer is rounded again by every
              layer after it, and past about six layers two correct orders of
              summation differ by more than a stated 3e-2 (measured: 1.9e-2 at
              four layers, 2.5e-2 at six, 4.2e-2 at 36)
  head        what follows the last layer for each new token: final RMSNorm and
              the tied quantized lm_head
  tiny_mlp    the fp32 Linear -> GELU -> Linear region

The layers and the model replay one captured graph per pass (their input is
copied into it), so their launches cost what they cost a serving program; the
single ops pay their own dispatch.
"""

from __future__ import annotations

import dataclasses
import functools
import math
import sys
from pathlib import Path

import torch

PKG = str(Path(__file__).resolve().parent.parent / "metal-autotune_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

from autotuner_runtime import kernels, ops, regions  # noqa: E402
from autotuner_runtime.graph import GraphWrapper  # noqa: E402
from workloads import lfm2, qwen3  # noqa: E402
from workloads.quantize import random_quantized  # noqa: E402

DEV = "cuda"
DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}
EPS = 1e-6


def listed():
    return [
        # The smallest call: one projection for one decode token (gate_proj of
        # the Qwen3-4B shape), where dispatch and launch count.
        {"name": "linear decode", "kind": "linear", "M": 1, "N": 9728, "K": 2560, "bits": 4,
         "gs": 64, "dtype": "bfloat16"},
        # The reference's fp32 example network, at its own sizes.
        {"name": "tiny mlp fp32", "kind": "tiny_mlp", "M": 32, "K": 256, "H": 1024, "N": 256},
        # Six draft tokens verified, or six requests decoded, together: an
        # 8-bit MLP (LFM2 widths) on the memory-bound side.
        {"name": "mlp 8bit 6 tokens", "kind": "mlp", "M": 6, "hidden": 2048, "inter": 8192,
         "bits": 8, "gs": 64, "dtype": "bfloat16"},
        # A larger, odd batch of decode tokens: fp16, group 128, Qwen3 widths.
        {"name": "mlp fp16 21 tokens", "kind": "mlp", "M": 21, "hidden": 2560, "inter": 9728,
         "bits": 4, "gs": 128, "dtype": "float16"},
        # The end of every step: one token's logits.
        {"name": "lm head", "kind": "head", "M": 1, "V": 151936, "K": 2560, "bits": 4},
        # One token against a long conversation (odd length), 32/8 heads of 128.
        {"name": "attention decode 8191", "kind": "attention", "H": 32, "HK": 8, "D": 128, "Lq": 1,
         "Lk": 8191, "cap": 8192, "dtype": "bfloat16"},
        # A long prompt's attention, Qwen3 heads.
        {"name": "attention prefill 2048", "kind": "attention", "H": 32, "HK": 8, "D": 128,
         "Lq": 2048, "Lk": 2048, "cap": 2048, "dtype": "bfloat16"},
        # A ragged chunk of a chunked prefill behind a cached prefix.
        {"name": "qwen3 layer chunk 501", "kind": "qwen_layer", "L": 501, "offset": 777,
         "bits": 4},
        # The two layer kinds of the 2048-token LFM2 prefill, at both widths.
        {"name": "lfm2 conv layer 2048", "kind": "lfm2_layer", "layer": "conv", "L": 2048,
         "offset": 0, "bits": 8},
        {"name": "lfm2 attn layer 2048", "kind": "lfm2_layer", "layer": "attn", "L": 2048,
         "offset": 0, "bits": 4},
        # A decode step in the middle of a conversation, and the 128-token
        # prefill, through a whole model.
        {"name": "qwen3 decode step", "kind": "qwen_model", "layers": 4, "L": 1, "offset": 1000},
        {"name": "qwen3 prefill 128", "kind": "qwen_model", "layers": 4, "L": 128, "offset": 0},
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm; odd ones among them."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "mlp", "mlp", "attention", "attention", "attention",
                       "qwen_layer", "lfm2_layer", "lfm2_layer", "head", "tiny_mlp"])
    dt = rng.choice(["bfloat16", "bfloat16", "float16"])
    if kind == "linear":
        return {"kind": kind, "M": _log(rng, 1, 2048), "N": 4 * _log(rng, 128, 3000),
                "K": 256 * rng.randint(2, 40), "bits": rng.choice([4, 4, 8]),
                "gs": rng.choice([32, 64, 64, 128]), "dtype": dt}
    if kind == "mlp":
        return {"kind": kind, "M": _log(rng, 1, 1024), "hidden": 256 * rng.randint(4, 16),
                "inter": 256 * rng.randint(8, 40), "bits": rng.choice([4, 4, 8]),
                "gs": rng.choice([64, 64, 128]), "dtype": dt}
    if kind == "attention":
        D, HK = rng.choice([64, 128]), rng.choice([2, 4, 8])
        H = HK * rng.choice([1, 2, 4, 5, 8])
        form = rng.choice(["decode", "prompt", "chunk"])
        if form == "decode":
            Lq, Lk = rng.choice([1, 1, 1, 4]), _log(rng, 64, 16384)
        elif form == "prompt":
            Lq = Lk = _log(rng, 16, 2048)
        else:
            Lq = _log(rng, 16, 512)
            Lk = Lq + _log(rng, 16, 4096)
        return {"kind": kind, "H": H, "HK": HK, "D": D, "Lq": Lq, "Lk": Lk,
                "cap": Lk + rng.choice([0, 1, 37, 500]), "dtype": dt}
    if kind == "qwen_layer":
        return {"kind": kind, "L": _log(rng, 1, 1024), "offset": rng.choice([0, rng.randint(1, 3000)]),
                "bits": 4}
    if kind == "lfm2_layer":
        return {"kind": kind, "layer": rng.choice(["conv", "attn"]), "L": _log(rng, 1, 2048),
                "offset": rng.choice([0, rng.randint(2, 3000)]), "bits": rng.choice([4, 8])}
    if kind == "head":
        return {"kind": kind, "M": rng.randint(1, 8), "V": rng.choice([32000, 65536, 128257, 151936]),
                "K": rng.choice([1024, 2048, 2560]), "bits": rng.choice([4, 4, 8])}
    return {"kind": kind, "M": _log(rng, 1, 512), "K": 4 * rng.randint(16, 256),
            "H": 4 * rng.randint(32, 512), "N": rng.randint(16, 512)}


# ---------------------------------------------------------------------------
# inputs

# a program keeps one spec per region
TINY_MLP = regions.tiny_mlp("perf_tiny_mlp")


@functools.lru_cache(maxsize=None)
def _mlp_specs(dtype, gs, bits):
    tag = f"{dtype}_{gs}_{bits}"
    return (regions.dual_swiglu(f"perf_dual_{tag}", dtype, gs, bits),
            regions.residual_rmsnorm(f"perf_down_{tag}", dtype, gs, bits, EPS))


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(gen, *shape, dtype, std=1.0, mean=0.0):
    return (mean + std * torch.randn(shape, generator=gen, device=DEV)).to(dtype)


def _layer_model(case, seed):
    """A one-layer model of the case's family with its regions installed."""
    if case["kind"] == "qwen_layer":
        cfg = dataclasses.replace(qwen3.Qwen3Config(), vocab_size=1024, bits=case["bits"])
        model = qwen3.build(cfg, seed=seed, num_layers=1)
        qwen3.install_regions(model)
    else:
        cfg = dataclasses.replace(lfm2.Lfm2Config(), vocab_size=1024, bits=case["bits"])
        model = lfm2.build(cfg, seed=seed, num_layers=1, layer_types=(case["layer"],))
        lfm2.install_regions(model)
    return cfg, model


def _fill_cache(cache, offset, gen):
    """A cached prefix of `offset` rows: keys as q/k-norm leaves them (unit
    scale), values of a projection's size."""
    for t, std in ((cache.keys, 1.0), (cache.values, 0.9)):
        t[:, :, :offset] = _randn(gen, *t[:, :, :offset].shape, dtype=t.dtype, std=std)


def prepare(case, seed):
    gen, kind = _gen(seed), case["kind"]
    if kind == "linear":
        dt = DTYPES[case["dtype"]]
        x = _randn(gen, case["M"], case["K"], dtype=dt)
        w = random_quantized(case["N"], case["K"], gen, DEV, case["gs"], case["bits"], dt)
        return {"case": case, "x": x, "w": w}
    if kind == "mlp":
        dt, M, Hd, I = DTYPES[case["dtype"]], case["M"], case["hidden"], case["inter"]
        q = (case["gs"], case["bits"])
        st = {"case": case, "x": _randn(gen, 1, M, Hd, dtype=dt),
              "gate": random_quantized(I, Hd, gen, DEV, *q, dt),
              "up": random_quantized(I, Hd, gen, DEV, *q, dt),
              "down": random_quantized(Hd, I, gen, DEV, *q, dt),
              "resid": _randn(gen, 1, M, Hd, dtype=dt),
              "norm": _randn(gen, Hd, dtype=dt, std=0.1, mean=1.0)}
        st["specs"] = _mlp_specs(case["dtype"], *q)
        return st
    if kind == "attention":
        dt, HK, D = DTYPES[case["dtype"]], case["HK"], case["D"]
        return {"case": case, "q": _randn(gen, 1, case["H"], case["Lq"], D, dtype=dt),
                "k": _randn(gen, 1, HK, case["cap"], D, dtype=dt),
                "v": _randn(gen, 1, HK, case["cap"], D, dtype=dt)}
    if kind in ("qwen_layer", "lfm2_layer"):
        cfg, model = _layer_model(case, seed)
        L, offset = case["L"], case["offset"]
        cache = model.make_cache(offset + L)[0]
        if isinstance(cache, lfm2.ConvCache):
            state = _randn(gen, 1, 2, cfg.hidden_size, dtype=torch.bfloat16) if offset else None
        else:
            state = None
            _fill_cache(cache, offset, gen)
        st = {"case": case, "cfg": cfg, "model": model, "layer": GraphWrapper(model.model.layers[0]),
              "cache": cache, "state": state, "offset": offset,
              "x": _randn(gen, 1, L, cfg.hidden_size, dtype=torch.bfloat16)}
        for _ in range(2):  # captures (a carried conv state is captured in its own form)
            run(st)
        return st
    if kind == "qwen_model":
        cfg = qwen3.Qwen3Config()
        model = qwen3.build(cfg, seed=seed, num_layers=case["layers"])
        qwen3.install_regions(model)
        caches = model.make_cache(case["offset"] + case["L"])
        for c in caches:
            _fill_cache(c, case["offset"], gen)
        ids = torch.randint(0, cfg.vocab_size, (1, case["L"]), generator=gen, device=DEV)
        st = {"case": case, "cfg": cfg, "model": model, "wrapped": GraphWrapper(model),
              "caches": caches, "ids": ids, "offset": case["offset"]}
        run(st)  # captures
        return st
    if kind == "head":
        K = case["K"]
        return {"case": case, "h": _randn(gen, 1, case["M"], K, dtype=torch.bfloat16),
                "norm": _randn(gen, K, dtype=torch.bfloat16, std=0.1, mean=1.0),
                "w": random_quantized(case["V"], K, gen, DEV, 64, case["bits"])}
    M, K, H, N = case["M"], case["K"], case["H"], case["N"]
    f = torch.float32
    ins = [_randn(gen, M, K, dtype=f), _randn(gen, H, K, dtype=f, std=K ** -0.5),
           _randn(gen, H, dtype=f, std=0.1), _randn(gen, N, H, dtype=f, std=H ** -0.5),
           _randn(gen, N, dtype=f, std=0.1)]
    return {"case": case, "ins": ins, "spec": TINY_MLP}


# ---------------------------------------------------------------------------
# one pass


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "linear":
        return ops.quantized_matmul(st["x"], *st["w"], group_size=case["gs"], bits=case["bits"])
    if kind == "mlp":
        dual, down = st["specs"]
        act, = kernels.try_sized(dual, [st["x"], *st["gate"], *st["up"]])
        return kernels.try_sized(down, [act, *st["down"], st["resid"], st["norm"]])
    if kind == "attention":
        D = case["D"]
        return ops.scaled_dot_product_attention(
            st["q"], st["k"], st["v"], D ** -0.5, "causal" if case["Lq"] > 1 else None,
            kv_len=case["Lk"], out_layout=1)
    if kind in ("qwen_layer", "lfm2_layer"):
        c = st["cache"]
        c.offset = st["offset"]
        if isinstance(c, lfm2.ConvCache):
            c.state = st["state"]
            return [st["layer"](st["x"], c), c.state]
        return [st["layer"](st["x"], c), c.keys, c.values]
    if kind == "qwen_model":
        for c in st["caches"]:
            c.offset = st["offset"]
        return st["wrapped"](st["ids"], st["caches"])
    if kind == "head":
        return ops.quantized_matmul(ops.rms_norm(st["h"], st["norm"], EPS), *st["w"],
                                    bits=case["bits"])
    return kernels.try_sized(st["spec"], st["ins"])


# ---------------------------------------------------------------------------
# what a pass cannot do without


def _qbytes(N, K, bits, gs=64):
    return N * K * bits // 8 + 2 * (N * K // gs) * 2


def _attn_pairs(Lq, Lk):
    """(query, key) pairs a causal pass looks at."""
    return Lq * (Lk - Lq) + Lq * (Lq + 1) // 2


def _layer_work(cfg, case, kind):
    L, off, H = case["L"], case["offset"], cfg.hidden_size
    I = cfg.intermediate_size
    if kind == "conv":
        shapes = [(3 * H, H), (H, H), (2 * I, H), (H, I)]
        extra_b, extra_f = 4 * 2 * H * 2, 0
    else:
        D, HQ, HK = cfg.head_dim, cfg.num_attention_heads, cfg.num_key_value_heads
        shapes = [((HQ + 2 * HK) * D, H), (H, HQ * D), (2 * I, H), (H, I)]
        extra_b = 2 * HK * D * 2 * (off + L) + 2 * HK * D * 2 * L
        extra_f = 4 * HQ * D * _attn_pairs(L, off + L)
    return (sum(_qbytes(n, k, cfg.bits) for n, k in shapes) + 2 * 2 * L * H + extra_b,
            2 * L * sum(n * k for n, k in shapes) + extra_f)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": _qbytes(N, K, case["bits"], case["gs"]) + 2 * M * (N + K),
                "flops": 2 * M * N * K}
    if kind == "mlp":
        M, Hd, I = case["M"], case["hidden"], case["inter"]
        return {"bytes": 3 * _qbytes(I, Hd, case["bits"], case["gs"]) + 2 * M * 4 * Hd,
                "flops": 6 * M * Hd * I}
    if kind == "attention":
        H, HK, D, Lq, Lk = case["H"], case["HK"], case["D"], case["Lq"], case["Lk"]
        return {"bytes": 2 * (2 * H * Lq + 2 * HK * Lk) * D, "flops": 4 * H * D * _attn_pairs(Lq, Lk)}
    if kind == "qwen_layer":
        b, f = _layer_work(dataclasses.replace(qwen3.Qwen3Config(), bits=case["bits"]), case, "attn")
        return {"bytes": b, "flops": f}
    if kind == "lfm2_layer":
        cfg = dataclasses.replace(lfm2.Lfm2Config(), bits=case["bits"])
        b, f = _layer_work(cfg, case, case["layer"])
        return {"bytes": b, "flops": f}
    if kind == "qwen_model":
        cfg = qwen3.Qwen3Config()
        b, f = _layer_work(cfg, case, "attn")
        n, V, H = case["layers"], cfg.vocab_size, cfg.hidden_size
        acts = 2 * 2 * case["L"] * H  # between the layers nothing has to be written
        return {"bytes": n * (b - acts) + _qbytes(V, H, cfg.bits) + case["L"] * _qbytes(1, H, cfg.bits)
                + 2 * V, "flops": n * f + 2 * V * H}
    if kind == "head":
        M, V, K = case["M"], case["V"], case["K"]
        return {"bytes": _qbytes(V, K, case["bits"]) + 2 * M * (K + V), "flops": 2 * M * V * K}
    M, K, H, N = case["M"], case["K"], case["H"], case["N"]
    return {"bytes": 4 * (M * K + H * K + N * H + H + N + M * N), "flops": 2 * M * H * (K + N)}


def tolerance(case):
    """About four times what the results differ by from the same in 64 bits
    (measured; in brackets), which is what rounding the results, and what one
    op hands to the next, to the case's data type gives. fp16 keeps three more
    bits than bf16."""
    kind = case["kind"]
    if kind == "tiny_mlp":  # fp32 sums (4e-7)
        return {"rel": 4e-6, "max": 4e-5}
    if kind == "qwen_model":  # two orders of summation against each other: 1.9e-2
        return {"rel": 3e-2, "max": 0.4}
    rel = {"linear": 7e-3,      # (1.6e-3)
           "attention": 9e-3,   # (2.3e-3)
           "head": 1.2e-2,      # (3.1e-3)
           "mlp": 1.6e-2,       # (4.0e-3)
           "qwen_layer": 2.2e-2, "lfm2_layer": 2.2e-2}[kind]  # (5.6e-3)
    if case.get("dtype") == "float16":
        rel /= 8
    return {"rel": rel, "max": 10 * rel}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch

F64 = torch.float64


def _deq(w, s, b, bits):
    words = w.view(torch.int32)
    per = 32 // bits
    shifts = torch.arange(per, device=w.device, dtype=torch.int32) * bits
    q = (words.unsqueeze(-1) >> shifts) & ((1 << bits) - 1)
    N = w.shape[0]
    q = q.reshape(N, s.shape[1], -1).to(F64)
    return (q * s.to(F64).unsqueeze(-1) + b.to(F64).unsqueeze(-1)).reshape(N, -1)


def _mm(x, wsb, bits):
    return x @ _deq(*wsb, bits).t()


def _lin(x, m):
    return _mm(x, (m.weight, m.scales, m.biases), m.bits)


def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.to(F64)


def _silu_mul(g, u):
    return g * torch.sigmoid(g) * u


def _rope(x, base, offset):
    L, D = x.shape[-2], x.shape[-1]
    freq = torch.exp2(-torch.arange(0, D, 2, device=x.device, dtype=F64) / D * math.log2(base))
    ang = (torch.arange(L, device=x.device, dtype=F64) + offset)[:, None] * freq
    a, c = x[..., : D // 2], x[..., D // 2:]
    return torch.cat([a * ang.cos() - c * ang.sin(), a * ang.sin() + c * ang.cos()], -1)


def _sdpa(q, k, v, scale, causal):
    """q [H, Lq, D], k and v [HK, Lk, D] -> [Lq, H, D]."""
    H, Lq, D = q.shape
    HK, Lk, _ = k.shape
    out = torch.empty((Lq, H, D), device=q.device, dtype=F64)
    hide = None
    if causal:
        hide = torch.arange(Lk, device=q.device)[None] > torch.arange(Lq, device=q.device)[:, None] + Lk - Lq
    for h in range(H):
        s = (q[h] @ k[h // (H // HK)].t().contiguous()) * scale
        if causal:
            s = s.masked_fill(hide, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[h // (H // HK)]
    return out


def _attention_exact(x, a, names, cfg, eps, cache, offset):
    L = x.shape[0]
    q_n, k_n, out = (getattr(a, n) for n in names)
    HQ, HK, D = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    heads = lambda t, n: t.reshape(L, n, D).transpose(0, 1)  # noqa: E731
    q = _rope(_rms(heads(_lin(x, a.q_proj), HQ), q_n.weight, eps), cfg.rope_theta, offset)
    k = _rope(_rms(heads(_lin(x, a.k_proj), HK), k_n.weight, eps), cfg.rope_theta, offset)
    v = heads(_lin(x, a.v_proj), HK)
    keys = torch.cat([cache.keys[0, :, :offset].to(F64), k], 1)
    values = torch.cat([cache.values[0, :, :offset].to(F64), v], 1)
    o = _sdpa(q, keys, values, a.scale, True).reshape(L, HQ * D)
    return _lin(o, out), keys, values


def _qwen_layer_exact(layer, cfg, x, cache, offset):
    a, m, eps = layer.self_attn, layer.mlp, cfg.rms_norm_eps
    o, keys, values = _attention_exact(_rms(x, layer.input_layernorm.weight, eps), a,
                                       ("q_norm", "k_norm", "o_proj"), cfg, eps, cache, offset)
    h = x + o
    hn = _rms(h, layer.post_attention_layernorm.weight, eps)
    return (h + _lin(_silu_mul(_lin(hn, m.gate_proj), _lin(hn, m.up_proj)), m.down_proj),
            keys, values)


def _base(layer):
    return layer.wrapped if hasattr(layer, "wrapped") else layer


def exact(case, seed):
    kind = case["kind"]
    st = prepare(case, seed)
    if kind == "linear":
        return _mm(st["x"].to(F64), st["w"], case["bits"])
    if kind == "mlp":
        x, bits = st["x"][0].to(F64), case["bits"]
        h = st["resid"][0].to(F64) + _mm(_silu_mul(_mm(x, st["gate"], bits), _mm(x, st["up"], bits)),
                                         st["down"], bits)
        return [h[None], _rms(h, st["norm"], EPS)[None]]
    if kind == "attention":
        Lk = case["Lk"]
        return _sdpa(st["q"][0].to(F64), st["k"][0, :, :Lk].to(F64), st["v"][0, :, :Lk].to(F64),
                     case["D"] ** -0.5, True)[None]
    if kind == "qwen_layer":
        h, keys, values = _qwen_layer_exact(_base(st["model"].model.layers[0]), st["cfg"],
                                            st["x"][0].to(F64), st["cache"], st["offset"])
        return [h[None], keys[None], values[None]]
    if kind == "lfm2_layer":
        layer, cfg, x = _base(st["model"].model.layers[0]), st["cfg"], st["x"][0].to(F64)
        eps = cfg.norm_eps
        xn = _rms(x, layer.operator_norm.weight, eps)
        if case["layer"] == "conv":
            c = layer.conv
            B, C, xs = _lin(xn, c.in_proj).chunk(3, -1)
            bx = B * xs
            first = (torch.zeros_like(bx[:2]) if bx.shape[0] >= 2 else
                     torch.zeros((2, bx.shape[1]), device=bx.device, dtype=F64)) \
                if st["state"] is None else st["state"][0].to(F64)
            pad = torch.cat([first, bx])
            w = c.conv.weight.reshape(-1, 3).to(F64)
            L = bx.shape[0]
            conv = pad[:L] * w[:, 0] + pad[1:L + 1] * w[:, 1] + pad[2:] * w[:, 2]
            h, carried = x + _lin(C * conv, c.out_proj), [pad[-2:][None]]
        else:
            o, keys, values = _attention_exact(xn, layer.self_attn,
                                               ("q_layernorm", "k_layernorm", "out_proj"), cfg, eps,
                                               st["cache"], st["offset"])
            h, carried = x + o, [keys[None], values[None]]
        m, hn = layer.feed_forward, _rms(h, layer.ffn_norm.weight, eps)
        return [(h + _lin(_silu_mul(_lin(hn, m.w1), _lin(hn, m.w3)), m.w2))[None], *carried]
    if kind == "qwen_model":
        cfg, inner = st["cfg"], st["model"].model
        e = inner.embed_tokens
        ids = st["ids"][0]
        h = _deq(e.weight.view(torch.int32)[ids], e.scales[ids], e.biases[ids], e.bits)
        for layer, cache in zip(inner.layers, st["caches"]):
            h = _qwen_layer_exact(_base(layer), cfg, h, cache, st["offset"])[0]
        h = _rms(h[-1:], inner.norm.weight, cfg.rms_norm_eps)
        return _lin(h, e)[None]
    if kind == "head":
        h = _rms(st["h"][0].to(F64), st["norm"], EPS)
        return _mm(h, st["w"], case["bits"])[None]
    x, w1, b1, w2, b2 = (t.to(F64) for t in st["ins"])
    a = x @ w1.t() + b1
    return [(a * (1 + torch.erf(a / math.sqrt(2.0))) / 2) @ w2.t() + b2]
