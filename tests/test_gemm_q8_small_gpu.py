"""The small-tile W8A8 / FP8 GEMMs (csrc/gemm_q8_small.hip) at the edges of every tile shape: one row,
one row past a tile, widths that end inside a tile, one K block, K blocks that do not fill an
iteration, rows strided and packed, every output type, bias type and activation.

int8 is bit-exact: the 256 x 256 tiles' int32 accumulators (psq_gemm_i8_i32) through the oracle's
epilogue.  fp8 sums are fp32 in the kernel's order; against the exact sum of the same codes (float64)
they keep the 1e-2 rms bar of the other fp32-accumulating paths.
"""
import pytest
import torch

import oracle
from conftest import seeded
from test_fused_mlp_gpu import assert_gelu_of
from test_gated_mlp_gpu import assert_gate_of

pytestmark = pytest.mark.gpu

# M, N, K: the tile shape that a 256-CU device takes them to
SHAPES = [(1, 33, 128), (16, 40, 1152), (17, 100, 384), (3, 15360, 640),   # 16 x 32
          (32, 13000, 256), (33, 5501, 384),                              # 32 x 64
          (100, 4999, 384), (64, 13832, 128),                             # 64 x 64
          (75, 13990, 640),                                               # 80 x 64
          (2000, 1500, 256),                                              # 96 x 128
          (1025, 3544, 384),                                              # 128 x 128
          (1020, 5001, 128),                                              # 128 x 192
          (1024, 8000, 256)]                                              # 256 x 128


def codes(rows, K, seed, dtype, dev, pad):
    """[rows, K] codes of the full range, as a view with `pad` more bytes per row."""
    x = torch.randn(rows, K + pad, generator=seeded(seed))
    x = (x * 40).round().clamp(-127, 127).to(torch.int8) if dtype == torch.int8 else (x * 20).to(dtype)
    return x.to(dev)[:, :K]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("variant", range(4))
def test_int8_bitexact(gpu, M, N, K, variant):
    from powershard_amd import ops
    out = [torch.bfloat16, torch.float16, torch.float32, torch.bfloat16][variant]
    pad = 0 if variant % 2 else 48
    a, w = codes(M, K, 1, torch.int8, gpu, pad), codes(N, K, 2, torch.int8, gpu, pad)
    g = seeded(3)
    sa, sw = torch.rand(M, generator=g) * 1e-2, torch.rand(N, generator=g) * 1e-2
    bias = [None, torch.float16, torch.float32, torch.bfloat16][variant]
    b = None if bias is None else torch.randn(N, generator=g).to(bias)
    y = ops.gemm_i8(a, sa.to(gpu), w, sw.to(gpu), None if b is None else b.to(gpu), out_dtype=out)
    ref = oracle.epilogue_i32(ops.gemm_i8_i32(a, w).cpu(), sa, sw, b, out_dtype=out)
    assert torch.equal(y.cpu(), ref)


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("wdt", [torch.float8_e4m3fn, torch.float8_e5m2])
def test_fp8_within_bar(gpu, M, N, K, wdt):
    from powershard_amd import ops
    a, w = codes(M, K, 4, torch.float8_e4m3fn, gpu, 16), codes(N, K, 5, wdt, gpu, 16)
    g = seeded(6)
    sa, sw = torch.rand(M, generator=g).to(gpu), torch.rand(N if M % 2 else 1, generator=g).to(gpu)
    b = torch.randn(N, generator=g).to(gpu)
    exact = (a.float().double() @ w.float().double().T) * sa.double()[:, None] * sw.double()[None] + b.double()
    rms = exact.pow(2).mean().sqrt().item()
    y32 = ops.gemm_fp8(a, sa, w, sw, b, out_dtype=torch.float32)
    assert (y32.double() - exact).abs().max().item() <= 1e-2 * rms
    # the 16-bit outputs are the rounding of the kernel's own fp32 value
    for dt in (torch.bfloat16, torch.float16):
        assert torch.equal(ops.gemm_fp8(a, sa, w, sw, b, out_dtype=dt), y32.to(dt))


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_gelu_of_the_rounded_output(gpu, M, N, K):
    from powershard_amd import ops
    a, w = codes(M, K, 7, torch.int8, gpu, 0), codes(N, K, 8, torch.int8, gpu, 0)
    sa, sw = torch.full((M,), 2e-2, device=gpu), torch.full((N,), 1e-3, device=gpu)
    lin = ops.gemm_i8(a, sa, w, sw)
    assert_gelu_of(ops.gemm_i8(a, sa, w, sw, activation="gelu_tanh"), lin, f"{M}x{N}x{K}")


# gate + up rows; the gate pairs W tiles inside a wave, so its tiles are their own instances
@pytest.mark.parametrize("M,N,K", [(5, 256, 128), (17, 384, 1152), (20, 16640, 256), (50, 16640, 384),
                                   (2000, 1536, 256), (1025, 3584, 128), (1024, 8064, 256)])
@pytest.mark.parametrize("kind,dt", [("i8", torch.bfloat16), ("fp8", torch.float16), ("i8", torch.float32)])
def test_gate(gpu, M, N, K, kind, dt):
    from powershard_amd import ops
    cdt = torch.int8 if kind == "i8" else torch.float8_e4m3fn
    a, w = codes(M, K, 9, cdt, gpu, 0), codes(N, K, 10, cdt, gpu, 0)
    g = seeded(11)
    sa, sw = (torch.rand(M, generator=g) * 4e-3).to(gpu), (torch.rand(N, generator=g) * 1e-2).to(gpu)
    b = torch.randn(N, generator=g).to(torch.bfloat16).to(gpu)
    fn = ops.gemm_i8 if kind == "i8" else ops.gemm_fp8
    lin = fn(a, sa, w, sw, b, out_dtype=dt)
    y = fn(a, sa, w, sw, b, out_dtype=dt, activation="silu_gate")
    assert_gate_of(y, lin, f"{kind} {M}x{N}x{K} {dt}")
