"""QuantLinear's one-call forward (QuantLinear._direct) against the general path on the same module:
the same bits for every stored format, type, activation and shape that it takes, and None -- the
general path -- for what has to be converted, copied, tracked or refused."""
import warnings

import pytest
import torch
from torch import nn

from conftest import heavy_rows
from test_quant_linear_gpu import make_layer

pytestmark = pytest.mark.gpu


def both(layer, x, act=None):
    """(direct, general) outputs of one forward."""
    y = layer._direct(x, act)
    keep, type(layer)._direct = type(layer)._direct, lambda self, x, act, into=None: None
    try:
        return y, layer._forward(x, act)
    finally:
        type(layer)._direct = keep


@pytest.mark.parametrize("fmt,opts", [("int8", {"convrot": True, "convrot_groupsize": 256}), ("int8", {"convrot": False}),
                                      ("fp8", {}), ("int4", {"group_size": 128})])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lead", [(1,), (), (2, 9), (1, 300), (3, 1, 7)])
def test_same_bits(gpu, fmt, opts, dt, lead):
    K, N = 1024, 384
    layer, _, _ = make_layer(K, N, fmt, opts, dt, True, gpu, seed=3, bias=len(lead) != 1)
    M = max(1, int(torch.tensor(lead).prod())) if lead else 1
    x = heavy_rows(M, K, seed=4, dtype=dt).reshape(*lead, K).to(gpu)
    for act in (None, "gelu_tanh", "silu_gate"):
        y, ref = both(layer, x, act)
        if fmt == "int4" and act:
            assert y is None
            continue
        assert y.shape == ref.shape and y.dtype == ref.dtype
        assert torch.equal(y.view(torch.int16), ref.view(torch.int16))


def test_left_to_the_general_path(gpu):
    K, N = 512, 192
    layer, _, _ = make_layer(K, N, "int8", {"convrot": True, "convrot_groupsize": 256}, torch.bfloat16, True, gpu, seed=5)
    x = heavy_rows(8, K, seed=6, dtype=torch.bfloat16).to(gpu)
    wide = torch.zeros(8, K + 8, dtype=x.dtype, device=gpu)
    wide[:, :K] = x
    odd = torch.zeros(8 * K + 1, dtype=x.dtype, device=gpu)[1:].view(8, K).copy_(x)
    ref = layer(x)
    for other in (wide[:, :K], odd, x.t().contiguous().t(), x.float()):   # strides, alignment, type
        assert layer._direct(other, None) is None
        assert torch.equal(layer(other), ref)
    assert layer._direct(x[:0], None) is None and layer(x[:0]).shape == (0, N)
    assert layer._direct(x, "silu_gate") is None            # 192 rows: the gate is a separate pass
    layer.bias = nn.Parameter(layer.bias.float(), requires_grad=False)
    assert layer._direct(x, None) is None and torch.equal(layer(x), ref)
    other = make_layer(K, N, "int8", {"convrot": True, "convrot_groupsize": 256}, torch.bfloat16, True, gpu, seed=5)[0]
    biases = torch.stack([other.bias.data, other.bias.data + 1])
    with warnings.catch_warnings(), torch.no_grad():        # a batched parameter
        warnings.simplefilter("ignore")
        y = torch.vmap(lambda b: torch.func.functional_call(other, {"bias": b}, (x,)))(biases)
    assert y.shape == (2, 8, N) and not other._ps_native
    with warnings.catch_warnings(), torch.no_grad():        # no storage under vmap: dequantize, as before
        warnings.simplefilter("ignore")
        y = torch.vmap(layer)(x.reshape(4, 2, K))
    assert y.shape == (4, 2, N) and not layer._ps_native
    assert layer._direct(x, None) is None


@pytest.fixture
def direct_calls(monkeypatch):
    """[(op, whether it wrote into the caller's rows)] of the one-call forwards."""
    from powershard_amd import ops
    seen = []
    for name in ("linear_q8_direct", "linear_w4a16_direct"):
        def wrap(*args, _name=name, _fn=getattr(ops, name)):
            seen.append((_name, args[-1] is not None))
            return _fn(*args)
        monkeypatch.setattr(ops, name, wrap)
    return seen


@pytest.mark.parametrize("fmt,opts,op", [("int8", {"convrot": True, "convrot_groupsize": 256}, "linear_q8_direct"),
                                         ("fp8", {}, "linear_q8_direct"), ("int4", {"group_size": 128}, "linear_w4a16_direct")])
@pytest.mark.parametrize("chunk", [None, 30])
def test_modules_take_it(gpu, direct_calls, fmt, opts, op, chunk):
    """A module call runs it, and an MLP's down projection writes the result rows from it: the bits of
    the same MLP whose down projection (with a forward hook) is copied."""
    from powershard_amd.mlp import chunked_mlp, gated_mlp
    K, H = 256, 512
    x = heavy_rows(70, K, seed=8, dtype=torch.bfloat16).to(gpu)
    up, down, gate = (make_layer(k, n, fmt, opts, torch.bfloat16, True, gpu, seed=9 + n)[0]
                      for k, n in ((K, H), (H, K), (K, 2 * H)))
    up(x)
    assert direct_calls == [(op, False)]
    for mlp, first in ((chunked_mlp, up), (gated_mlp, gate)):
        del direct_calls[:]
        y = mlp(first, down, x, chunk_tokens=chunk)
        calls = 3 if chunk else 1
        # int4 outputs are 16-bit: chunked_mlp's fp32 rows are copied
        into = fmt != "int4" or mlp is gated_mlp
        assert direct_calls.count((op, True)) == (calls if into else 0)
        hook = down.register_forward_hook(lambda m, args, out: None)
        ref = mlp(first, down, x, chunk_tokens=chunk)
        hook.remove()
        assert y.dtype == ref.dtype and torch.equal(y, ref)


def test_its_errors_are_not_swallowed(gpu, monkeypatch):
    from powershard_amd import ops
    layer, _, _ = make_layer(256, 64, "int8", {"convrot": False}, torch.bfloat16, True, gpu, seed=13)

    def broken(*args):
        raise TypeError("a mistake in the one-call forward")

    monkeypatch.setattr(ops, "linear_q8_direct", broken)
    with pytest.raises(TypeError, match="a mistake"):
        layer(heavy_rows(4, 256, seed=14, dtype=torch.bfloat16).to(gpu))
