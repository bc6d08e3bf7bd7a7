"""One or two rows quantized and multiplied in one kernel (csrc/gemm_q8_vec.hip) against the quantizer
and the small-tile GEMM: the same bits for every rotation group, weight kind, type, stride and output
form, K blocks that do not fill an iteration, the raw rows inside and past the ring, widths that end
inside a tile; rows of zeros, infinities and NaN; and the sizes past its range on both sides."""
import pytest
import torch

from conftest import seeded
from test_gemm_q8_small_gpu import codes

pytestmark = pytest.mark.gpu


def run_both(gpu, x, w, sw, b, kind, rot, act):
    from powershard_amd import _native, ops
    (M, K), N = x.shape, w.shape[0]
    lib, dt = _native.lib(), ops._DT[x.dtype]
    y = torch.full((M, N), 7.0, dtype=x.dtype, device=gpu)
    wide = torch.full((M, N), 7.0, dtype=torch.float32, device=gpu)
    scratch = torch.empty(lib.psq_linear_q8_scratch_bytes(M, K), dtype=torch.uint8, device=gpu)
    for out in (y, wide):
        if out is wide and (act or kind == 2):
            continue
        st = lib.psq_linear_q8(kind, x.data_ptr(), dt, x.stride(0), rot, w.data_ptr(), K, sw.data_ptr(), int(sw.numel() > 1),
                               None if b is None else b.data_ptr(), 0 if b is None else ops._DT[b.dtype], act,
                               out.data_ptr(), int(out is wide), N, M, N, K, scratch.data_ptr(), ops._raw_stream(0))
        assert st == 0, _native.last_error()
    q, s = ops.quantize_rows(x, fp8=kind != 0, rot_group=rot)
    fn = ops.gemm_i8 if kind == 0 else ops.gemm_fp8
    ref = fn(q, s, w, sw, b, out_dtype=x.dtype, activation="gelu_tanh" if act else None)
    nan = torch.isnan(ref)
    assert torch.equal(torch.isnan(y), nan) and torch.equal(y[~nan], ref[~nan])
    if not act and kind != 2:
        assert torch.equal(torch.isnan(wide), nan) and torch.equal(wide[~nan], ref.float()[~nan])


@pytest.mark.parametrize("M", [1, 2, 3])
@pytest.mark.parametrize("K,N", [(128, 33), (384, 1000), (1024, 31), (4224, 512), (5120, 15363), (8192, 97), (8320, 64)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_same_bits(gpu, M, K, N, dt):
    g = seeded(M + K + N)
    x = (torch.randn(M, K + 8, generator=g) * 3).to(dt).to(gpu)[:, :K]
    for kind, wdt in ((0, torch.int8), (1, torch.float8_e4m3fn), (2, torch.float8_e5m2)):
        w = codes(N, K, 2, wdt, gpu, 0)
        sw = (torch.rand(N if kind == 0 or N % 2 else 1, generator=g) * 1e-2).to(gpu)
        bias = [None, torch.randn(N, generator=g).to(dt).to(gpu), torch.randn(N, generator=g).to(gpu)]
        groups = [r for r in (0, 4, 16, 64, 256, 1024) if not r or K % r == 0] if kind == 0 else [0]
        for i, rot in enumerate(groups):
            run_both(gpu, x, w, sw, bias[i % 3], kind, rot, 1 if kind != 2 and i % 2 else 0)


@pytest.mark.parametrize("kind", [0, 1])
def test_special_rows(gpu, kind):
    K, N = 1024, 64
    w = codes(N, K, 3, torch.int8 if kind == 0 else torch.float8_e4m3fn, gpu, 0)
    sw = torch.full((N,), 1e-2, device=gpu)
    base = torch.randn(2, K, generator=seeded(4)).to(torch.bfloat16)
    for row, col, v in ((0, 0, float("nan")), (1, K - 1, float("inf")), (0, 500, float("-inf")), (1, 7, 3.3e38)):
        x = base.clone()
        x[row, col] = v
        run_both(gpu, x.to(gpu), w, sw, None, kind, 256 if kind == 0 else 0, 0)
    x = base.clone()
    x[0] = 0
    run_both(gpu, x.to(gpu), w, sw, None, kind, 256 if kind == 0 else 0, 0)
    run_both(gpu, torch.zeros(2, K, dtype=torch.bfloat16, device=gpu), w, sw, None, kind, 0, 0)
