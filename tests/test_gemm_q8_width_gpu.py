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
