"""The tiled weight-only kernel's row-tile heights (csrc/gemm_wonly.hip, plan_tiled): sizes that a
256-CU device takes to tiles of 128, 160, 192, 224 and 256 rows, with rows and columns that end inside a
tile, against the exact product (float64) of the dequantized weights."""
import pytest
import torch


pytestmark = pytest.mark.gpu

# M, N, K: 128, 160, 160 (odd N), 192, 224, 256 rows
SHAPES = [(250, 25600, 256), (300, 25600, 256), (319, 19001, 320), (380, 25590, 192), (440, 25600, 128),
          (512, 25000, 192)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", ["u4", "i8"])
def test_row_tiles(gpu, M, N, K, dt, kind):
    from powershard_amd import ops
    g = torch.Generator(device=gpu).manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device=gpu).to(dt)
    bias = torch.randn(N, generator=g, device=gpu).to(dt)
    if kind == "u4":
        wq = torch.randint(0, 256, (N, K // 2), generator=g, device=gpu, dtype=torch.uint8)
        s = (torch.rand(N, K // 64, generator=g, device=gpu) * 0.1 + 0.01).half()
        z = (torch.rand(N, K // 64, generator=g, device=gpu) * 15).half()
        y = ops.gemm_w4a16(x, wq, s, z, 64, bias, out_dtype=torch.float32)
        w = ops.dequant_uint4(wq, s, z, 64, out_dtype=dt).double()
    else:
        wq = torch.randint(-128, 128, (N, K), generator=g, device=gpu, dtype=torch.int8)
        s = torch.rand(N, generator=g, device=gpu) * 0.1
        y = ops.gemm_w8a16(x, wq, s, bias, out_dtype=torch.float32)
        w = wq.double() * s.double()[:, None]
    exact = x.double() @ w.T + bias.double()
    rms = exact.pow(2).mean().sqrt().item()
    # fp32 accumulation of K 16-bit products; a uint4 weight may round to the other 16-bit neighbour
    # (2^-9 of it at most, on about 2^-16 of the weights)
    assert (y.double() - exact).abs().max().item() <= 1e-2 * rms
    fn = (lambda o: ops.gemm_w4a16(x, wq, s, z, 64, bias, out_dtype=o)) if kind == "u4" else \
        (lambda o: ops.gemm_w8a16(x, wq, s, bias, out_dtype=o))
    assert torch.equal(fn(dt), y.to(dt))
