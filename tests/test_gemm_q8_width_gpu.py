"""The 256 x 224 / 192 / 160 tiles of the W8A8 / FP8 GEMM (csrc/gemm_q8_kernel.hpp), at sizes that a
256-CU device takes to each of them: rows and columns that end inside a tile, in whole 8-column chunks
and not, one K stage, odd and even numbers of stages, more tiles than workgroups.

The accumulation order is the 256 x 256 tiles', so int8 and fp8 outputs are their bits: compared with
the fp32 output of the same call (always 256 x 256 tiles) rounded once, and for int8 with the int32
accumulators through the oracle's epilogue.
"""
import pytest
import torch

import oracle
from conftest import seeded
from test_fused_mlp_gpu import assert_gelu_of
from test_gemm_q8_small_gpu import codes

pytestmark = pytest.mark.gpu

SHAPES = [(1290, 5400, 384), (1561, 5121, 128), (2050, 3600, 1024),     # 160
          (2050, 4504, 128), (2047, 5000, 640), (1561, 6001, 512),      # 192
          (1561, 7004, 128), (2050, 5400, 512), (2560, 5121, 384)]      # 224


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("kind", ["i8", "e4m3", "e5m2"])
def test_width_matches_square_tiles(gpu, M, N, K, kind):
    from powershard_amd import ops
    cdt = {"i8": torch.int8, "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e4m3fn}[kind]
    wdt = torch.float8_e5m2 if kind == "e5m2" else cdt
    a, w = codes(M, K, 1, cdt, gpu, 16), codes(N, K, 2, wdt, gpu, 32)
    g = seeded(3)
    sa, sw = torch.rand(M, generator=g) * 1e-2, torch.rand(N, generator=g) * 1e-2
    b = torch.randn(N, generator=g).to(torch.bfloat16) if N % 2 == 0 else None
    fn = ops.gemm_i8 if kind == "i8" else ops.gemm_fp8
    call = lambda **kw: fn(a, sa.to(gpu), w, sw.to(gpu), None if b is None else b.to(gpu), **kw)
    y32 = call(out_dtype=torch.float32)
    for dt in (torch.bfloat16, torch.float16):
        y = call(out_dtype=dt)
        assert torch.equal(y, y32.to(dt))
        if kind == "i8":
            assert torch.equal(y.cpu(), oracle.epilogue_i32(ops.gemm_i8_i32(a, w).cpu(), sa, sw, b, out_dtype=dt))
        if kind != "e5m2":
            assert_gelu_of(call(out_dtype=dt, activation="gelu_tanh"), y, f"{kind} {M}x{N}x{K} {dt}")


# and: the 256 x 256 tiles, small tiles, outputs whose rows are not 16-byte aligned
@pytest.mark.parametrize("M,N,K", SHAPES + [(2047, 7004, 128), (3000, 5000, 256), (3, 1000, 384), (100, 4999, 128),
                                            (2000, 1500, 256), (1024, 8000, 128)])
@pytest.mark.parametrize("kind", [0, 1])
def test_fp32_rows_of_the_rounded_output(gpu, M, N, K, kind):
    """psq_linear_q8's fp32 output holds the 16-bit output's values, bit for bit."""
    from powershard_amd import ops
    g = torch.Generator(device=gpu).manual_seed(M + N)
    w = codes(N, K, 5, torch.int8 if kind == 0 else torch.float8_e4m3fn, gpu, 0)
    sw = torch.rand(N, generator=g, device=gpu) * 1e-2
    for dt in (torch.bfloat16, torch.float16):
        x = torch.randn(M, K, generator=g, device=gpu).to(dt)
        b = torch.randn(N, generator=g, device=gpu).to(dt) if dt == torch.bfloat16 else None
        call = lambda into: ops.linear_q8_direct(x, M, K, kind, w.data_ptr(), sw.data_ptr(), 1, 0, N, b, 0, into)
        y = call(None)
        wide, same = (torch.full((M, N), 7.0, dtype=t, device=gpu) for t in (torch.float32, dt))
        assert call(wide) is wide and torch.equal(wide, y.float())
        assert call(same) is same and torch.equal(same, y)
