"""mi_sdpa's kernels at the edges of their dispatch, against the float64 oracle.

Bar: max|c - r| <= 1e-2 max|r| (bf16/fp16), the library's attention bar. The
kernels round P to the data type (relative 2^-9 in bf16), sum in fp32 and round
the result once (2^-9 of its own size).
"""

from __future__ import annotations

import numpy as np
import pytest

import oracle
from conftest import rng, to_np, to_torch

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from autotuner_runtime import hip, ops  # noqa: E402


def _close(got, want, tol=1e-2):
    err = np.abs(to_np(got).astype(np.float64) - want).max() / np.abs(want).max()
    assert err <= tol, err


# (B, H, HK, Lq, Lk, D, causal, scale factor, dtype)
@pytest.mark.parametrize("B,H,HK,Lq,Lk,D,causal,factor,dtype", [
    (1, 8, 2, 1, 1, 128, True, 1, "bfloat16"),        # one key
    (1, 32, 8, 8, 1024, 64, True, 1, "bfloat16"),     # decode rows 32 columns, not split
    (1, 32, 8, 8, 1025, 64, True, 1, "float16"),      # ... split, last split one tile
    (2, 10, 2, 7, 1500, 128, True, 1, "bfloat16"),    # 35 columns: two column blocks; two sequences
    (1, 4, 4, 3, 2100, 128, False, 1, "bfloat16"),    # split, no mask
    (1, 3, 1, 1, 16500, 64, True, 1, "bfloat16"),     # one kv head: 129 splits
    (1, 8, 2, 9, 9, 64, True, 1, "bfloat16"),         # first size past decode
    (1, 8, 2, 33, 1100, 128, True, 1, "float16"),     # a second row block of one row
    (3, 15, 3, 417, 417, 64, True, 1, "bfloat16"),    # a unit a workgroup, q heads 5 a group
    (1, 32, 8, 400, 431, 128, True, 1, "bfloat16"),   # ... ragged chunk behind a prefix
    (1, 32, 8, 384, 384, 64, False, 1, "float16"),    # ... no mask
    (1, 32, 8, 400, 731, 128, True, 1, "bfloat16"),   # past 640 keys: shared tiles
    (1, 32, 8, 384, 644, 64, False, 1, "float16"),
    (2, 15, 3, 641, 641, 64, True, 1, "bfloat16"),    # ... an odd unit count, q heads 5 a group
    (1, 32, 8, 390, 741, 128, True, -1, "bfloat16"),
    (1, 8, 2, 1, 70, 128, True, -1, "bfloat16"),      # a negative scale
    (1, 32, 8, 390, 390, 128, True, -1, "bfloat16"),
    (1, 8, 2, 40, 70, 64, True, 0, "bfloat16"),       # scale 0: the mean of the visible values
])
def test_sdpa_dispatch_edges(B, H, HK, Lq, Lk, D, causal, factor, dtype):
    """Rows past kv_len in the cache hold NaN: none is read."""
    r = rng(4000 + Lq + Lk + D)
    cap = Lk + 5
    q = oracle.round_to(r.normal(0, 1, (B, H, Lq, D)), dtype)
    k = oracle.round_to(r.normal(0, 1, (B, HK, cap, D)), dtype)
    v = oracle.round_to(r.normal(0, 1, (B, HK, cap, D)), dtype)
    scale = factor * D ** -0.5
    want = oracle.sdpa(q, k[:, :, :Lk], v[:, :, :Lk], scale, causal, dtype)
    kd, vd = to_torch(k, dtype), to_torch(v, dtype)
    kd[:, :, Lk:] = float("nan")
    vd[:, :, Lk:] = float("nan")
    mask = "causal" if causal else None
    for layout in (0, 1):
        o = ops.scaled_dot_product_attention(to_torch(q, dtype), kd, vd, scale, mask, kv_len=Lk,
                                             out_layout=layout)
        _close(o if layout == 0 else o.transpose(1, 2), want)


@pytest.mark.parametrize("Lq,Lk", [(1, 1025), (5, 3000)])
def test_sdpa_without_a_workspace(Lq, Lk):
    """mi_sdpa runs a split shape's keys in one workgroup per kv head: the same
    sums in another order. A workspace one byte short takes that path too."""
    r = rng(4100 + Lk)
    H, HK, D = 8, 2, 128
    t = [to_torch(oracle.round_to(r.normal(0, 1, (1, h, n, D)), "bfloat16"), "bfloat16")
         for h, n in ((H, Lq), (HK, Lk), (HK, Lk))]
    q, k, v = t
    o, o1 = torch.empty_like(q), torch.empty_like(q)
    L = hip.lib()
    args = (1, H, HK, Lq, Lk, D, Lk, D ** -0.5, 1, 0, hip.MI_BF16)
    st = torch.cuda.current_stream().cuda_stream
    assert L.mi_sdpa(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), *args, st) == 0
    need = L.mi_sdpa_workspace_bytes(1, H, HK, Lq, Lk, D)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    assert L.mi_sdpa_ws(q.data_ptr(), k.data_ptr(), v.data_ptr(), o1.data_ptr(), *args,
                        ws.data_ptr(), need - 1, st) == 0
    assert torch.equal(o, o1)
    _close(o, oracle.sdpa(*(to_np(x) for x in t), D ** -0.5, True, "bfloat16"))
    _close(ops.scaled_dot_product_attention(q, k, v, D ** -0.5), to_np(o).astype(np.float64))


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("H,HK,Lq,Lk,D", [
    (8, 2, 1, 128, 128),      # decode
    (8, 2, 2, 2048, 64),      # ... split
    (8, 2, 32, 160, 64),      # few query rows
    (32, 8, 400, 672, 128),   # shared tiles
])
@pytest.mark.parametrize("gap", [25.0, 150.0])
def test_sdpa_one_large_score(H, HK, Lq, Lk, D, gap, dtype):
    """One key's score lies far above the others', at each position of a key
    tile in turn: its value is the result (the other weights are below 2^-36),
    and no exponent overflows, whichever lane holds that score."""
    tdt = getattr(torch, dtype)
    q = torch.zeros((1, H, Lq, D), device="cuda")
    q[..., 0] = 1
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7)
    v = torch.randn((1, HK, Lk, D), generator=gen, device="cuda").to(tdt)
    for pos in [*range(32), 32 + 4, Lk - 1]:
        k = torch.zeros((1, HK, Lk, D), device="cuda")
        k[:, :, pos, 0] = 1
        o = ops.scaled_dot_product_attention(q.to(tdt), k.to(tdt), v, gap, None)
        want = v[:, :, pos].repeat_interleave(H // HK, 1)[:, :, None].expand_as(o)
        assert bool(((o.float() - want.float()).abs() <= 2 ** -7 * want.float().abs() + 1e-6).all()), pos


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("H,HK,Lq,Lk,D", [
    (8, 2, 1, 992, 128),      # decode
    (8, 2, 2, 2048, 64),      # ... split
    (8, 2, 32, 160, 64),      # few query rows
    (32, 8, 400, 672, 128),   # shared tiles
])
def test_sdpa_row_sum_adds_unrounded_weights(H, HK, Lq, Lk, D, dtype):
    """In every tile of 32 keys one has weight 1 and value 1, the others weight p
    and value 0, with p just below the middle between two values of the type:
    the result is 1 / (1 + 31 p), correctly rounded; with the rounded p in the
    sum it is the next value up."""
    half_step = 2.0 ** (-9 if dtype == "bfloat16" else -12)
    p = 0.5 + 0.95 * half_step
    q = torch.zeros((1, H, Lq, D), device="cuda")
    q[..., 0] = 1
    k = torch.zeros((1, HK, Lk, D), device="cuda")
    k[..., 0] = 1
    v = torch.zeros_like(k)
    k[:, :, ::32] = 0
    v[:, :, ::32] = 1
    tdt = getattr(torch, dtype)
    o = ops.scaled_dot_product_attention(q.to(tdt), k.to(tdt), v.to(tdt), float(np.log(p)), None)
    want = torch.tensor(1 / (1 + 31 * p), dtype=torch.float64).to(tdt)
    assert torch.tensor(1 / (1 + 31 * 0.5), dtype=torch.float64).to(tdt) != want
    assert bool((o == want.cuda()).all()), (float(o.min()), float(o.max()), float(want))


@pytest.mark.parametrize("Lq,Lk", [(1, 40), (2, 1500), (40, 40), (400, 700)])
def test_sdpa_scale_of_nan(Lq, Lk):
    q, k = torch.ones((1, 32, Lq, 64), device="cuda").bfloat16(), torch.ones(
        (1, 8, Lk, 64), device="cuda").bfloat16()
    assert bool(ops.scaled_dot_product_attention(q, k, k, float("nan")).isnan().all())


def test_sdpa_short_last_chunk():
    """The last 4 of 2052 rows as a call of their own: the whole prefill's bits
    without a workspace (the same streams), within rounding through ops (split)."""
    r = rng(4200)
    H, HK, D, L, tail = 16, 4, 128, 2052, 4
    q, k, v = (to_torch(oracle.round_to(r.normal(0, 1, (1, h, L, D)), "bfloat16"), "bfloat16")
               for h in (H, HK, HK))
    whole = ops.scaled_dot_product_attention(q, k, v, D ** -0.5)[:, :, -tail:]
    qt = q[:, :, -tail:].contiguous()
    o = torch.empty_like(qt)
    assert hip.lib().mi_sdpa(qt.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), 1, H, HK, tail,
                             L, D, L, D ** -0.5, 1, 0, hip.MI_BF16,
                             torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(o, whole)
    split = ops.scaled_dot_product_attention(qt, k, v, D ** -0.5)
    _close(split, to_np(whole).astype(np.float64))
