"""Int8Linear's one-call forward (psq_linear_w8a16) against its separate calls: the same bits, and the
same answer of the output check, which runs in the GEMM's epilogue (skinny, tiled and stream-K kernels,
whole tiles and element stores, 16-bit and edge columns)."""
import pytest
import torch

from conftest import seeded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1, 16, 256), (5, 333, 512), (40, 1000, 256), (70, 512, 512), (100, 2048, 2048),
                                   (300, 515, 256), (1024, 5120, 512), (700, 13824, 256)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rot", [0, 256])
def test_one_call(gpu, M, N, K, dt, rot):
    from powershard_amd import ops
    g = seeded(M + N)
    x = torch.randn(M, K, generator=g).to(dt).to(gpu)
    wq = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).to(gpu)
    s = (torch.rand(N, generator=g) * 1e-3).to(gpu)
    b = torch.randn(N, generator=g).to(dt).to(gpu)

    def both(s, b):
        y, finite = ops.linear_w8a16_direct(x, M, K, wq, s, rot, N, b)
        ref = ops.gemm_w8a16(ops.rotate_rows(x, rot) if rot else x, wq, s, b, out_dtype=dt)
        assert torch.equal(y.view(torch.int16), ref.view(torch.int16))
        assert finite is (not ops.any_nonfinite(ref)) and finite == bool(torch.isfinite(ref).all())
        return finite

    assert both(s, b) and both(s, None)
    big = torch.finfo(dt).max
    for at in (0, N // 2, N - 1):
        for v in (float("inf"), float("-inf"), float("nan")):
            bad = b.clone()
            bad[at] = v
            assert not both(s, bad)
        edge = b.clone()
        edge[at] = big                       # the largest finite value is finite ...
        zero = s.clone()
        zero[at] = 0.0
        assert both(zero, edge)
    if dt == torch.float16:
        assert not both(s * 1e6, b)          # ... and a sum past it rounds to infinity
    assert both(s, b)                        # a later finite call is finite again
