"""The measured workloads of the quantized linear path: what is timed, how its inputs are made and
what its outputs must be.

Each case is one call (or one layer group) that a diffusion or text-encoder program makes through
the package's public entry points: a QuantLinear forward, the q / k / v projections of one attention
input, a chunked or gated MLP, an Int8Linear forward, a weight decode.  Weights are drawn as codes
and scales directly, so that the 64-bit reference below needs nothing of the package.
"""
import math
import os
import sys

import torch
from torch import nn

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "comfyui-powershard_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
GROUP = 128           # uint4 scale / zero group
ROT = 256             # ConvRot group
DEVICE = "cuda:0"


def _linear(name, fmt, M, K, N, rot=0, dtype="bf16", bias=True, compute="native"):
    return dict(name=name, kind="linear", fmt=fmt, M=M, K=K, N=N, rot=rot, dtype=dtype, bias=bias, compute=compute)


def listed():
    return [
        # one conditioning vector through an int8 ConvRot projection: latency and the weight stream
        _linear("int8_vector_m1", "int8", 1, 5120, 15360, rot=ROT),
        # the 512 text tokens of a prompt through a cross-attention projection
        _linear("int8_context_m512", "int8", 512, 5120, 5120, rot=ROT),
        # q, k and v of one attention input, the ragged share of an 8-way token split of a video
        dict(name="int8_qkv_m4095", kind="qkv", fmt="int8", M=4095, K=5120, N=5120, rot=ROT, dtype="bf16", bias=True),
        # the widest projection of a video block over all its tokens
        _linear("int8_video_m32760", "int8", 32760, 5120, 13824, rot=ROT),
        # a short prompt through a fused q/k/v projection in fp8
        _linear("fp8_prompt_m77", "fp8", 77, 5120, 15360),
        # an image's tokens through the same projection
        _linear("fp8_image_m8192", "fp8", 8192, 5120, 15360),
        # int4 text encoder: one token, the next-token call
        _linear("int4_token_m1", "int4", 1, 5120, 25600, bias=False),
        # int4 text encoder: a whole prompt of ragged length
        _linear("int4_prompt_m300", "int4", 300, 5120, 25600, bias=False),
        # the int8_fp16 storage: Int8Linear with ConvRot rows, output check included
        dict(name="int8linear_m1024", kind="int8linear", fmt="int8", M=1024, K=5120, N=5120, rot=ROT, dtype="f16",
             bias=True),
        # the feed-forward of a video block over all its tokens: up, GELU, down
        dict(name="int8_gelu_mlp_m32760", kind="gelu_mlp", fmt="int8", M=32760, K=5120, N=13824, rot=ROT, dtype="bf16",
             bias=True),
        # the gated feed-forward of an image block: gate and up, SiLU product, down
        dict(name="int8_gated_mlp_m8192", kind="gated_mlp", fmt="int8", M=8192, K=5376, N=14336, rot=ROT, dtype="f16",
             bias=True),
        # a stored ConvRot weight back to bf16 (the dequantize compute mode, LoRA merges)
        dict(name="int8_decode_13824x5120", kind="decode", fmt="int8", M=0, K=5120, N=13824, rot=ROT, dtype="bf16",
             bias=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: token counts over 1..32760 on a log scale, widths of 512 to 14336 columns and
    64 to 25600 rows, aligned and odd, every format, type and option of the listed cases."""
    kind = rng.choice(["linear"] * 6 + ["qkv", "int8linear", "gelu_mlp", "gated_mlp", "decode"])
    fmt = rng.choice(["int8", "int8", "fp8", "fp8", "e5m2", "int4", "int4"]) if kind in ("linear", "decode") else \
        "int8" if kind == "int8linear" else rng.choice(["int8", "fp8"])
    M = _log(rng, 1, 4096 if fmt == "int4" else 8192 if kind == "int8linear" else 32760)
    K = 256 * _log(rng, 2, 56)
    N = _log(rng, 64, 25600)
    # most stored layers have rows in whole multiples of 16, some are odd
    if kind in ("gelu_mlp", "gated_mlp"):
        N = 256 * max(2, min(56, N // 256))
    elif rng.random() < 0.75:
        N = max(64, N // 16 * 16)
    dtype = "f16" if kind == "int8linear" else rng.choice(["bf16", "bf16", "f16"])
    rot = rng.choice([0, ROT]) if fmt == "int8" else 0
    while M * K * N > 1.0e12:
        M = max(1, M // 2)
    case = dict(kind=kind, fmt=fmt, M=0 if kind == "decode" else M, K=K, N=N, rot=rot, dtype=dtype,
                bias=kind != "decode" and rng.random() < 0.6)
    if kind == "linear":
        case["compute"] = "dequantize" if rng.random() < 0.1 else "native"
    return case


# ------------------------------------------------------------------------------- inputs
def _gen(seed, salt):
    return torch.Generator(device=DEVICE).manual_seed((seed * 1000003 + salt * 7919 + 17) % (1 << 62))


def _weight(case, seed, salt, N, K):
    """The stored tensors of one layer: codes with their scales (and zeros), and the bias."""
    g = _gen(seed, salt)
    fmt = case["fmt"]
    normal = torch.randn(N, K, generator=g, device=DEVICE)
    # unit-gain layers: weights of about 1 / sqrt(K)
    sd = 1.0 / math.sqrt(K)
    if fmt == "int8":
        w = {"q": (normal * 32).round().clamp(-127, 127).to(torch.int8)}
        w["scale"] = (torch.rand(N, 1, generator=g, device=DEVICE) + 0.5) * (sd / 32)
    elif fmt in ("fp8", "e5m2"):
        code, top = (torch.float8_e4m3fn, 448.0) if fmt == "fp8" else (torch.float8_e5m2, 57344.0)
        w = {"q": (normal * (top / 5)).clamp(-top, top).to(code)}
        w["scale"] = torch.tensor(5 * sd / top, dtype=torch.float32, device=DEVICE)
    else:
        nib = (normal * 3 + 7.5).round().clamp(0, 15).to(torch.uint8)
        w = {"q": (nib[:, 0::2] | (nib[:, 1::2] << 4)).contiguous()}
        w["scale"] = ((torch.rand(N, K // GROUP, generator=g, device=DEVICE) + 0.5) * (sd / 3)).half()
        w["zero"] = (7.5 + torch.randn(N, K // GROUP, generator=g, device=DEVICE) * 0.5).half()
    w["bias"] = (torch.randn(N, generator=g, device=DEVICE) * 0.1).to(DTYPES[case["dtype"]]) if case["bias"] else None
    return w


def _layers(case):
    """[(salt, rows, columns)] of the case's weights."""
    N, K = case["N"], case["K"]
    return {"qkv": [(1, N, K), (2, N, K), (3, N, K)],
            "gelu_mlp": [(1, N, K), (2, K, N)],
            "gated_mlp": [(1, 2 * N, K), (2, K, N)]}.get(case["kind"], [(1, N, K)])


def _rows(case, seed):
    """Activations: normal, with a hundredth of the channels twenty times larger (outlier channels)."""
    g = _gen(seed, 99)
    M, K = case["M"], case["K"]
    x = torch.randn(1, M, K, generator=g, device=DEVICE)
    x *= torch.where(torch.rand(K, generator=g, device=DEVICE) < 0.01, 20.0, 1.0)
    return x.to(DTYPES[case["dtype"]])


def _quantized(case, w):
    from powershard_amd import quant_tensor as qtm
    dtype = DTYPES[case["dtype"]]
    if case["fmt"] == "int8":
        return qtm.QuantizedWeight(w["q"], qtm.Int8RowwiseLayout,
                                   qtm.Int8RowwiseParams(w["scale"], dtype, bool(case["rot"]), case["rot"] or 256))
    if case["fmt"] in ("fp8", "e5m2"):
        return qtm.QuantizedWeight(w["q"], qtm.Float8ScaledLayout, qtm.Float8ScaledParams(w["scale"], dtype))
    return qtm.QuantizedWeight(w["q"], qtm.UInt4GroupLayout,
                               qtm.UInt4GroupParams(w["scale"], w["zero"], dtype, GROUP))


FORMATS = {"int8": "int8_tensorwise", "fp8": "float8_e4m3fn", "e5m2": "float8_e5m2", "int4": "int4_asym_group"}


def _module(case, w, N, K):
    from powershard_amd import quant_linear as ql
    dtype = DTYPES[case["dtype"]]
    src = nn.Linear(K, N, bias=False, device="meta", dtype=dtype)
    if w["bias"] is not None:
        src.bias = nn.Parameter(w["bias"], requires_grad=False)
    qt = _quantized(case, w)
    fmt = FORMATS[case["fmt"]]
    plan = ql.plan_from_quantized(qt, fmt, dict(kind="quantize", module="layer", key="layer.weight", table=None))
    layer = ql.QuantLinear(src, plan, dtype, case.get("compute", "native") == "native")
    layer.qbytes = nn.Parameter(ql.pack(qt, plan, torch.device(DEVICE)), requires_grad=False)
    return layer


def prepare(case, seed):
    kind = case["kind"]
    weights = [_weight(case, seed, salt, n, k) for salt, n, k in _layers(case)]
    state = {"kind": kind}
    if kind == "decode":
        state["weight"] = _quantized(case, weights[0])
        return state
    state["x"] = _rows(case, seed)
    if kind == "int8linear":
        from powershard_amd.operations import Int8Linear
        src = nn.Linear(case["K"], case["N"], bias=False, device="meta", dtype=torch.float16)
        layer = Int8Linear(src, dict(convrot=bool(case["rot"]), group_size=case["rot"] or 256), rows=256)
        layer.weight = nn.Parameter(weights[0]["q"], requires_grad=False)
        layer.weight_scale = nn.Parameter(weights[0]["scale"], requires_grad=False)
        layer.bias = None if weights[0]["bias"] is None else nn.Parameter(weights[0]["bias"], requires_grad=False)
        state["layers"] = [layer]
    else:
        state["layers"] = [_module(case, w, n, k) for w, (_, n, k) in zip(weights, _layers(case))]
    return state


@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "decode":
        return state["weight"].dequantize()
    x, layers = state["x"], state["layers"]
    if kind == "qkv":
        from powershard_amd.quant_linear import reuse_quantized_inputs
        with reuse_quantized_inputs():
            return [layer(x) for layer in layers]
    if kind == "gelu_mlp":
        from powershard_amd.mlp import chunked_mlp
        return chunked_mlp(layers[0], layers[1], x)
    if kind == "gated_mlp":
        from powershard_amd.mlp import gated_mlp
        return gated_mlp(layers[0], layers[1], x)
    return layers[0](x)


# ------------------------------------------------------------------------ work and bars
def _weight_bytes(case, N, K):
    if case["fmt"] == "int4":
        return N * K // 2 + 4 * N * (K // GROUP)
    return N * K + (4 * N if case["fmt"] == "int8" else 4)


def work(case):
    M, N, K, kind = case["M"], case["N"], case["K"], case["kind"]
    nbytes = sum(_weight_bytes(case, n, k) + (2 * n if case["bias"] else 0) for _, n, k in _layers(case))
    if kind == "decode":
        return {"bytes": nbytes + 2 * N * K, "flops": 2 * N * K}
    flops = sum(2 * M * n * k for _, n, k in _layers(case))
    out = {"qkv": 3 * 2 * M * N, "gelu_mlp": 4 * M * K, "gated_mlp": 2 * M * K}.get(kind, 2 * M * N)
    return {"bytes": nbytes + 2 * M * K + out, "flops": flops}


def tolerance(case):
    """About four times the error against exact() that the path shows: the 16-bit rounding of the
    outputs (2^-9 / 2^-12 of a value, uniformly spread), of the weights where they are decoded to
    16 bits, and activation codes that fall to the other side of a rounding tie."""
    kind, bf16 = case["kind"], case["dtype"] == "bf16"
    if kind == "decode":
        return {"rel": 8e-3 if bf16 else 1e-3, "max": 1.6e-2 if bf16 else 2e-3}
    if kind in ("gelu_mlp", "gated_mlp"):
        return {"rel": 2e-2 if bf16 else 1e-2, "max": 0.5}
    return {"rel": 1e-2 if bf16 else 4e-3, "max": 8e-2}


# ---------------------------------------------------------------- the 64-bit reference
def _hadamard(size):
    h4 = torch.ones(4, 4, dtype=torch.float64, device=DEVICE)
    for a in range(4):
        h4[a, 3 - a] = -1
    h = torch.ones(1, 1, dtype=torch.float64, device=DEVICE)
    while h.shape[0] < size:
        h = torch.kron(h, h4 / 2)
    return h


def _rotated(x, rot):
    return x if not rot else (x.reshape(x.shape[0], -1, rot) @ _hadamard(rot)).reshape(x.shape)


def _real(case, w):
    """The layer's matrix in 64 bits, as stored (ConvRot weights stay rotated)."""
    q, s = w["q"], w["scale"].double()
    if case["fmt"] != "int4":
        return q.float().double() * s
    nib = torch.stack([q & 15, q >> 4], -1).reshape(q.shape[0], -1).double()
    return (nib - w["zero"].double().repeat_interleave(GROUP, 1)) * s.repeat_interleave(GROUP, 1)


def _activations(case, rows):
    """What the layer multiplies: the rotated rows, per-row quantized where the format does so."""
    rows = _rotated(rows, case["rot"])
    if case["kind"] == "int8linear" or case["fmt"] == "int4":
        return rows
    top = 127.0 if case["fmt"] == "int8" else 448.0
    s = rows.abs().amax(1, keepdim=True) / top
    s = torch.where(s == 0, torch.ones_like(s), s)
    u = (rows / s).clamp(-top, top)
    return (u.round() if case["fmt"] == "int8" else u.float().to(torch.float8_e4m3fn).double()) * s


def _apply(case, rows, w):
    if case.get("compute", "native") == "native":
        y = _activations(case, rows) @ _real(case, w).T
    else:
        y = rows @ _rotated(_real(case, w), case["rot"]).T
    return y if w["bias"] is None else y + w["bias"].double()


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    weights = [_weight(case, seed, salt, n, k) for salt, n, k in _layers(case)]
    if kind == "decode":
        return _rotated(_real(case, weights[0]), case["rot"])
    x = _rows(case, seed)
    rows = x[0].double()
    if kind == "qkv":
        return [_apply(case, rows, w).reshape(1, -1, case["N"]) for w in weights]
    if kind in ("linear", "int8linear"):
        return _apply(case, rows, weights[0]).reshape(1, -1, case["N"])
    out = []
    for part in rows.split(4096):   # bounds the 64-bit hidden state
        h = _apply(case, part, weights[0])
        if kind == "gelu_mlp":
            h = nn.functional.gelu(h, approximate="tanh")
        else:
            gate, up = h.chunk(2, -1)
            h = nn.functional.silu(gate) * up
        out.append(_apply(case, h, weights[1]))
    return torch.cat(out).reshape(1, -1, case["K"])
