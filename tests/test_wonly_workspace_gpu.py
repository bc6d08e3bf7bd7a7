"""int8 weight-only calls on a workspace of exactly the queried size: shapes that split K (f16 as
bf16, or whole tiles where bf16 splits: wonly_plan.hpp) run in both types, and Int8Linear keeps its kernels."""
import pytest
import torch

from conftest import seeded
from test_int8linear_gpu import make

pytestmark = pytest.mark.gpu

SHAPES = [(576, 5120, 5120), (700, 4096, 4096), (1000, 3072, 3072), (1024, 5120, 5120)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_queried_workspace_is_enough(gpu, M, N, K, dt):
    from powershard_amd import _native
    lib = _native.lib()
    g = torch.Generator(device=gpu).manual_seed(M)
    x = torch.randn(M, K, generator=g, device=gpu).to(dt)
    wq = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8, device=gpu)
    s = torch.rand(N, generator=g, device=gpu) * 1e-3
    y = torch.empty(M, N, dtype=dt, device=gpu)
    nb = lib.psq_gemm_wonly_workspace_bytes(_native.W_INT8, K, M, N, K, 0)
    ws = torch.zeros(nb, dtype=torch.uint8, device=gpu)
    code = _native.BF16 if dt == torch.bfloat16 else _native.F16
    _native.check(lib.psq_gemm_w8a16_ws(x.data_ptr(), code, K, wq.data_ptr(), s.data_ptr(), None, 0, y.data_ptr(), code,
                                        N, M, N, K, ws.data_ptr() if nb else None, nb,
                                        torch.cuda.current_stream().cuda_stream), "gemm_w8a16_ws")
    exact = (x.double() @ wq.double().T) * s.double()
    # one rounding of the result to its type, and fp32 sums of K exact products
    ulp = 2.0 ** (-8 if dt == torch.bfloat16 else -11)
    assert ((y.double() - exact).abs() <= ulp * exact.abs() + 1e-5 * exact.pow(2).mean().sqrt()).all()


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_int8linear_stays_native(gpu, monkeypatch, M, N, K):
    from powershard_amd import ops
    monkeypatch.setattr(ops, "_workspaces", {})      # a stream's first call: nothing has grown the workspace
    layer = make(K, N, True, 256, gpu, seed=M)
    layer((torch.randn(M, K, generator=seeded(M)) * 0.5).half().to(gpu))
    assert getattr(layer, "_ps_native", True), "the kernel path fell back to tiles"
