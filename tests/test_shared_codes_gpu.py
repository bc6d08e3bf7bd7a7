"""reuse_quantized_inputs with the one-call forward: q, k and v on one input quantize it once at every
size (narrow layers on many rows too), with the bits of the calls outside the block; the general path
shares the same codes; one or two rows are quantized inside the GEMM."""
import pytest
import torch

from conftest import heavy_rows
from test_quant_linear_gpu import make_layer

pytestmark = pytest.mark.gpu

FORMATS = [("int8", {"convrot": True, "convrot_groupsize": 256}), ("int8", {"convrot": False}), ("fp8", {})]


@pytest.fixture
def quantizations(monkeypatch):
    """Names of the calls that quantize rows, in order."""
    from powershard_amd import ops
    seen = []
    for name in ("quantize_rows", "quantize_direct", "linear_q8_direct"):
        def wrap(*args, _name=name, _fn=getattr(ops, name), **kw):
            seen.append(_name)
            return _fn(*args, **kw)
        monkeypatch.setattr(ops, name, wrap)
    return seen


@pytest.mark.parametrize("fmt,opts", FORMATS)
@pytest.mark.parametrize("M,K,N", [(3, 512, 320), (300, 1024, 512), (8200, 1024, 128), (3000, 5120, 64)])
def test_quantized_once(gpu, quantizations, fmt, opts, M, K, N):
    from powershard_amd.quant_linear import reuse_quantized_inputs
    layers = [make_layer(K, N, fmt, opts, torch.bfloat16, True, gpu, seed=60 + i, bias=i != 1)[0] for i in range(3)]
    x = heavy_rows(M, K, seed=64).to(gpu).reshape(1, M, K)
    calls = [lambda l: l(x), lambda l: l(x), lambda l: l.forward_act(x, "gelu_tanh")]
    ref = [c(l) for c, l in zip(calls, layers)]
    del quantizations[:]
    with reuse_quantized_inputs():
        got = [c(l) for c, l in zip(calls, layers)]
        assert quantizations == ["quantize_direct"]
        layers[0].bias = torch.nn.Parameter(layers[0].bias.float(), requires_grad=False)   # the general path
        assert layers[0]._direct(x, None) is None
        again = layers[0](x)
        assert quantizations == ["quantize_direct"]
        x.neg_()                                  # changed in place: quantized again
        layers[1](x)
        assert quantizations == ["quantize_direct"] * 2
    for a, b in zip(got + [again], ref + [ref[0]]):
        assert a.shape == b.shape and torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_hidden_and_single_rows_are_not_shared(gpu, quantizations):
    """The rows between an MLP's layers go to one module: they are neither shared nor kept."""
    from powershard_amd import quant_linear as ql
    from powershard_amd.mlp import chunked_mlp
    up, down = (make_layer(k, n, *FORMATS[0], torch.bfloat16, True, gpu, seed=70 + k)[0] for k, n in ((256, 512), (512, 256)))
    x = heavy_rows(40, 256, seed=71).to(gpu)
    ref = chunked_mlp(up, down, x)
    del quantizations[:]
    with ql.reuse_quantized_inputs():
        y = chunked_mlp(up, down, x)
        assert quantizations == ["quantize_direct", "linear_q8_direct"] and len(ql._shared.cache) == 1
        assert torch.equal(up(x[:2]).view(torch.int16), up(x)[:2].view(torch.int16))
        assert quantizations[2:] == ["linear_q8_direct"]
    assert torch.equal(y, ref)
