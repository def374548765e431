"""Past 128 tokens the quantized matmul picks one of several tile shapes by the
size of its grid. Each tile adds an output's products in the order that (M, K)
alone fixes, so a feature's values depend neither on how many features the call
has (which moves the choice) nor on the epilogue, and match the oracle's
arithmetic at every tile's edges."""

from __future__ import annotations

import pytest
import torch

from autotuner_runtime import ops
from workloads.quantize import random_quantized

pytestmark = pytest.mark.gpu

# (M, N, K): N and M at, and one step past, whole tiles of 32 / 64 features and
# 32 / 64 / 128 tokens, with grids from a few workgroups to several a CU
SHAPES = [(129, 512, 256), (129, 1024, 2560), (160, 2080, 512), (200, 6144, 512),
          (256, 2560, 4096), (257, 2052, 1024), (385, 2048, 8192), (501, 2560, 9728),
          (512, 2048, 2048), (640, 996, 1024), (1025, 6176, 512)]


@pytest.mark.parametrize("bits,dtype", [(4, torch.bfloat16), (8, torch.bfloat16), (4, torch.float16)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_tile_choice(M, N, K, bits, dtype):
    print(f"\ntile choice M={M} N={N} K={K} {bits}-bit {dtype}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M * 7 + N)
    x = torch.randn(M, K, generator=gen, device="cuda").to(dtype)
    w, s, b = random_quantized(N, K, gen, "cuda", 64, bits, dtype)
    y = ops.quantized_matmul(x, w, s, b, bits=bits)
    W = ops.dequantize(w, s, b, bits=bits).double()
    want = x.double() @ W.t().contiguous()
    # fp32 sums of K exact products, then one rounding to the output type: half
    # an ulp of the value and the sums' own error, K 2^-24 of the products' size
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    size = x.double().abs() @ W.abs().t().contiguous()
    slack = ulp * want.abs() + K * 2.0 ** -24 * size
    assert bool(((y.double() - want).abs() <= slack).all())
    # a narrower call (another tile) and the residual epilogue: the same bits
    n = 4 * max(1, N // 20)
    narrow = ops.quantized_matmul(x, w[:n].contiguous(), s[:n].contiguous(), b[:n].contiguous(),
                                  bits=bits)
    assert torch.equal(narrow, y[:, :n])
    zero = torch.zeros_like(y)
    assert torch.equal(ops.qmm_residual(x, w, s, b, zero, bits=bits), y)


@pytest.mark.parametrize("M,N,K", [(129, 256, 512), (200, 8192, 512), (320, 1028, 1024), (501, 2080, 512)])
def test_dual_tile_choice(M, N, K):
    print(f"\ndual tile choice M={M} N={N} K={K}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N)
    x = torch.randn(M, K, generator=gen, device="cuda").bfloat16()
    one, two = (random_quantized(N, K, gen, "cuda", 64, 4, torch.bfloat16) for _ in range(2))
    y1, y2 = ops.qmm_dual(x, *one, *two)
    assert torch.equal(y1, ops.quantized_matmul(x, *one))
    assert torch.equal(y2, ops.quantized_matmul(x, *two))


# (M, parts): grids whose cheapest tile is, on 256 CUs, 32 x 32, 32 x 64, 64 x 64,
# 64 x 128 and, for parts that are no multiples of 64 features, 32 x 128; a ragged
# last token tile each
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,Ns", [(131, (256, 64, 128)), (261, (512, 256, 256)),
                                  (301, (1024, 512, 512)), (1025, (4096, 1024, 1024)),
                                  (1025, (4096, 1024, 1056))])
def test_grouped_tile_choice(M, Ns, bits):
    """Each part equals its own launch, which has another grid and tile."""
    print(f"\ngrouped tile choice M={M} parts={Ns} {bits}-bit", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + sum(Ns) + bits)
    K = 512
    x = torch.randn(M, K, generator=gen, device="cuda").bfloat16()
    parts = [random_quantized(n, K, gen, "cuda", 64, bits, torch.bfloat16) for n in Ns]
    for y, p in zip(ops.qmm_grouped3(x, parts, 64, bits), parts):
        assert torch.equal(y, ops.quantized_matmul(x, *p, bits=bits))
        W = ops.dequantize(*p, bits=bits).double()
        want = x.double() @ W.t().contiguous()
        # half an ulp of the value and the fp32 sums' error, as above
        size = x.double().abs() @ W.abs().t().contiguous()
        assert bool(((y.double() - want).abs()
                     <= 2.0 ** -8 * want.abs() + K * 2.0 ** -24 * size).all())
