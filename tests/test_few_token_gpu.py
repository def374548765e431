"""The few-token quantized matmul (2 to 8 rows) at the edges of its shapes.

Bars: the region criterion max|c - r| <= 1e-2 max|r| against the factored
float oracle (the same per-group sums), and the fused epilogues bit for bit
against their op streams (one K split and group order per (M, K)).
"""

from __future__ import annotations

import numpy as np
import pytest

import oracle
from conftest import packed_to_torch, rng, to_np, to_torch

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from autotuner_runtime import ops  # noqa: E402
from workloads.quantize import random_quantized  # noqa: E402


def _dev(seed, N, K, gs, bits, dtype):
    wq, s, b = oracle.quantize_affine(rng(seed).normal(0, 0.02, (N, K)).astype(np.float32), gs, bits,
                                      dtype)
    return (wq, s, b), (packed_to_torch(wq), to_torch(s, dtype), to_torch(b, dtype))


def _close(got, want):
    err = np.abs(to_np(got).astype(np.float64) - want).max() / np.abs(want).max()
    assert err <= 1e-2, err


@pytest.mark.parametrize("M,N,K,gs,bits,dtype", [
    (3, 16, 32, 32, 4, "bfloat16"),       # one group: seven waves without work
    (5, 40, 96, 32, 4, "float16"),        # an odd group count (single groups), a ragged last tile
    (8, 200, 320, 64, 4, "bfloat16"),     # 5 groups
    (6, 72, 640, 64, 4, "float16"),       # 10 groups in pairs, runs of one and none
    (4, 64, 1152, 128, 4, "bfloat16"),    # 9 groups of four steps
    (7, 88, 4160, 64, 4, "bfloat16"),     # 16 waves, an odd group count
    (2, 56, 160, 32, 8, "bfloat16"),      # 8 bits, odd count
    (8, 200, 512, 32, 8, "float16"),      # 8 bits in pairs
    (5, 24, 1088, 64, 8, "float16"),
    (3, 104, 896, 128, 8, "bfloat16"),
    (1, 96, 8192, 64, 8, "bfloat16"),     # one token, long rows
    (8, 48, 9728, 64, 4, "bfloat16"),     # x past the LDS: two blocks of four rows
    (5, 32, 20480, 64, 8, "float16"),     # ... of three and two
    (2, 48, 90112, 128, 8, "bfloat16"),   # not one row fits: the generic kernel
])
def test_few_token_shapes(M, N, K, gs, bits, dtype):
    r = rng(5000 + M + N + K)
    x = oracle.round_to(r.normal(0, 1, (1, M, K)), dtype)
    res = oracle.round_to(r.normal(0, 1, (1, M, N)), dtype)
    host, w = _dev(5001 + N, N, K, gs, bits, dtype)
    host2, w2 = _dev(5002 + N, N, K, gs, bits, dtype)
    xd, rd = to_torch(x, dtype), to_torch(res, dtype)
    y = ops.quantized_matmul(xd, *w, group_size=gs, bits=bits)
    _close(y, oracle.qmm_factored(x, *host, gs, bits, dtype))
    assert torch.equal(ops.qmm_residual(xd, *w, rd, gs, bits), rd + y)
    u = ops.quantized_matmul(xd, *w2, group_size=gs, bits=bits)
    y1, u1 = ops.qmm_dual(xd, *w, *w2, gs, bits)
    assert torch.equal(y1, y) and torch.equal(u1, u)
    assert torch.equal(ops.qmm_dual(xd, *w, *w2, gs, bits, swiglu=True), ops.swiglu(y, u))


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("D", [64, 104])
def test_few_token_split_and_grouped(bits, D):
    """split(3) parts that start on and off a 16-feature tile, and q/k/v in one
    launch, against the plain projection."""
    M, K = 5, 1024
    r = rng(5100 + D)
    xd = to_torch(oracle.round_to(r.normal(0, 1, (1, M, K)), "bfloat16"), "bfloat16")
    _, w = _dev(5101, 3 * D, K, 64, bits, "bfloat16")
    t = ops.quantized_matmul(xd, *w, bits=bits)
    c, bx = ops.qmm_split_gate(xd, *w, bits=bits)
    assert torch.equal(c, t[..., D:2 * D]) and torch.equal(bx, t[..., :D] * t[..., 2 * D:])
    parts = [_dev(5102 + i, n, K, 64, bits, "bfloat16")[1] for i, n in enumerate((96, 32, 64))]
    for got, p in zip(ops.qmm_grouped3(xd, parts, bits=bits), parts):
        assert torch.equal(got, ops.quantized_matmul(xd, *p, bits=bits))


# K between what one part's scales leave room for in the LDS and what two or
# three parts' do: all epilogues of a shape take one kernel. (fp16 and thousands
# of outputs: two orders of summation differ in some of them.)
@pytest.mark.parametrize("K,gs", [(28672, 32), (49152, 64), (20448, 32)])
@pytest.mark.parametrize("bits,M", [(4, 3), (8, 5)])
def test_few_token_epilogues_agree_at_long_rows(K, gs, bits, M):
    D = 512
    gen = torch.Generator(device="cuda")
    gen.manual_seed(K + bits)
    xd = torch.randn((1, M, K), generator=gen, device="cuda").half()
    w, w2 = (random_quantized(3 * D, K, gen, "cuda", gs, bits, torch.float16) for _ in range(2))
    t, u = (ops.quantized_matmul(xd, *a, group_size=gs, bits=bits) for a in (w, w2))
    y1, u1 = ops.qmm_dual(xd, *w, *w2, gs, bits)
    assert torch.equal(y1, t) and torch.equal(u1, u)
    c, bx = ops.qmm_split_gate(xd, *w, gs, bits)
    assert torch.equal(c, t[..., D:2 * D]) and torch.equal(bx, t[..., :D] * t[..., 2 * D:])
    want = xd.double()[0] @ ops.dequantize(*w, group_size=gs, bits=bits).double().t().contiguous()
    assert float((t.double() - want).abs().max()) <= 1e-2 * float(want.abs().max())


@pytest.mark.parametrize("M,K", [(1, 4096), (1, 4160), (2, 5120), (2, 9728)])
def test_decode_epilogues_agree_at_long_rows(M, K):
    """One or two tokens at 4 bits: a row a wave past K = 4096, in every epilogue."""
    D = 1024
    gen = torch.Generator(device="cuda")
    gen.manual_seed(K + M)
    xd = torch.randn((1, M, K), generator=gen, device="cuda").half()
    w, w2 = (random_quantized(3 * D, K, gen, "cuda", 64, 4, torch.float16) for _ in range(2))
    t, u = (ops.quantized_matmul(xd, *a) for a in (w, w2))
    y1, u1 = ops.qmm_dual(xd, *w, *w2)
    assert torch.equal(y1, t) and torch.equal(u1, u)
    c, bx = ops.qmm_split_gate(xd, *w)
    assert torch.equal(c, t[..., D:2 * D]) and torch.equal(bx, t[..., :D] * t[..., 2 * D:])
    for y, a in zip(ops.qmm_grouped3(xd, (w, w2, w)), (t, u, t)):
        assert torch.equal(y, a)


@pytest.mark.parametrize("N,K,bits", [(2033, 320, 4), (2048, 320, 4), (2033, 576, 8)])
def test_few_token_epilogues_agree_at_unaligned_scales(N, K, bits):
    """One weight of a pair is a view whose scales and biases lie off a 16-byte
    boundary, or whose last tile's end does (which no 16-byte DMA can take)."""
    M = 4
    gen = torch.Generator(device="cuda")
    gen.manual_seed(N + bits)
    xd = torch.randn((M, K), generator=gen, device="cuda").half()
    one, w2 = (random_quantized(n, K, gen, "cuda", 64, bits, torch.float16) for n in (N + 1, N))
    off = [t[1:] for t in one]
    t, u = (ops.quantized_matmul(xd, *a, bits=bits) for a in (off, w2))
    assert torch.equal(t, ops.quantized_matmul(xd, *(a.clone() for a in off), bits=bits))
    y1, u1 = ops.qmm_dual(xd, *off, *w2, 64, bits)
    assert torch.equal(y1, t) and torch.equal(u1, u)
    want = xd.double() @ ops.dequantize(*off, bits=bits).double().t().contiguous()
    assert float((t.double() - want).abs().max()) <= 1e-2 * float(want.abs().max())


def test_few_token_unaligned_scales():
    """Scales and biases that are views off a 16-byte boundary (a value a thread
    in place of the kernel's 16-byte DMA)."""
    M, N, K = 4, 33, 320
    x = oracle.round_to(rng(5200).normal(0, 1, (M, K)), "bfloat16")
    host, w = _dev(5201, N, K, 64, 4, "bfloat16")
    y = ops.quantized_matmul(to_torch(x, "bfloat16"), *(t[1:] for t in w))
    _close(y, oracle.qmm_factored(x, *(a[1:] for a in host), 64, 4, "bfloat16"))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits,M,gs", [(4, 3, 64), (4, 5, 32), (4, 8, 128), (8, 2, 64), (8, 6, 32),
                                       (8, 8, 128)])
def test_few_token_sums_hold_small_products(bits, M, gs, dtype):
    """Every group's one code that is not zero meets a small x: sum x q is that
    product, and every partial sum of such products is exact in fp32, whatever
    the other, large x are. (Codes with an offset sum the large x as well, and
    lose the small product in their last bits.)"""
    N, K = 64, 32 * gs
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M)
    x = (1 + torch.rand((M, K), generator=gen, device="cuda")).to(dtype)
    x[:, ::gs] = 2.0 ** -12
    w = torch.zeros((N, K * bits // 32), dtype=torch.int32, device="cuda")
    w[:, ::gs * bits // 32] = 3                       # the group's first code
    s = torch.ones((N, K // gs), dtype=dtype, device="cuda")
    b = torch.zeros_like(s)
    want = torch.full((M, N), 32 * 3 * 2.0 ** -12, device="cuda").to(dtype)
    assert torch.equal(ops.quantized_matmul(x, w, s, b, group_size=gs, bits=bits), want)
    y1, y2 = ops.qmm_dual(x, w, s, b, w, s, b, gs, bits)
    assert torch.equal(y1, want) and torch.equal(y2, want)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M", [1, 2, 3, 8])
def test_generic_kernel_epilogues_agree(M, bits):
    """The fp32 kernel's sums are its outputs: an epilogue that rounds a group's
    sum in another way shows in the last bit."""
    N, K = 96, 1024
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + bits)
    xd = torch.randn((1, M, K), generator=gen, device="cuda")
    w, w2 = (random_quantized(N, K, gen, "cuda", 64, bits, torch.float32) for _ in range(2))
    t, u = (ops.quantized_matmul(xd, *a, bits=bits) for a in (w, w2))
    y1, u1 = ops.qmm_dual(xd, *w, *w2, 64, bits)
    assert torch.equal(y1, t) and torch.equal(u1, u)
    c, bx = ops.qmm_split_gate(xd, *w, 64, bits)
    assert torch.equal(c, t[..., 32:64]) and torch.equal(bx, t[..., :32] * t[..., 64:])
    assert torch.equal(ops.qmm_residual(xd, *w, torch.zeros_like(t), 64, bits), t)
    for y, a in zip(ops.qmm_grouped3(xd, (w, w2, w), 64, bits), (t, u, t)):
        assert torch.equal(y, a)
