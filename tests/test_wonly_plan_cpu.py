"""The tiled weight-only kernel's launch plan (csrc/wonly_plan.hpp, host arithmetic) against the workspace
that callers are told to pass: whatever the activation type, no launch needs more than the query's bytes.
Compiled for the CPU from the library's own header."""
import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "comfyui-powershard_amd" / "powershard_amd" / "csrc"
SHIM = """
#include "wonly_plan.hpp"
using namespace psq;
extern "C" long long need(int wk, int x_dtype, long long M, long long N, long long K, int cus)
{
    return plan_tiled(wk, x_dtype, M, N, K, cus, true).ws_bytes;
}
extern "C" long long told(int wk, long long M, long long N, long long K, int cus)
{
    return plan_workspace(wk, M, N, K, cus);
}
extern "C" long long most() { return kMaxWsBytes; }
// shapes of a grid whose query is too small, and the first of them
extern "C" long long short_of(int cus, long long *first)
{
    const long long widths[] = {64, 640, 1024, 2048, 2560, 3072, 4096, 5120, 5376, 6144, 8192, 10240, 13824, 14336, 25600};
    long long bad = 0;
    for (int wk = W_UINT4; wk <= W_INT8; wk++)
        for (long long N : widths)
            for (long long K : widths)
                for (long long M = 1; M <= 4096; M += M < 16 ? 5 : 61)
                    for (int dt : {PSQ_BF16, PSQ_F16})
                        if (need(wk, dt, M, N, K, cus) > told(wk, M, N, K, cus) && bad++ == 0) {
                            first[0] = M, first[1] = N, first[2] = K;
                        }
    return bad;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("plan")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run([gxx, "-O2", "-std=c++20", "-shared", "-fPIC", f"-I{CSRC}", "-o", str(d / "plan.so"), str(d / "shim.cpp")],
                   check=True)
    lib = ctypes.CDLL(str(d / "plan.so"))
    i64, i = ctypes.c_longlong, ctypes.c_int
    lib.need.restype = lib.told.restype = lib.most.restype = lib.short_of.restype = i64
    lib.need.argtypes, lib.told.argtypes = [i, i, i64, i64, i64, i], [i, i64, i64, i64, i]
    lib.short_of.argtypes = [i, ctypes.POINTER(i64)]
    return lib


@pytest.mark.parametrize("cus", [256, 104, 64])
def test_query_covers_every_launch(plan, cus):
    first = (ctypes.c_longlong * 3)()
    assert plan.short_of(cus, first) == 0, f"first at M, N, K = {list(first)}"


@pytest.mark.parametrize("M,N,K,split", [(576, 5120, 5120, True), (700, 4096, 4096, True), (128, 13824, 13824, True),
                                         (827, 5120, 13824, True), (202, 1137, 2048, True), (1081, 5120, 25600, True),
                                         (1024, 5120, 5120, False), (2500, 2048, 5376, False), (69, 4608, 1024, False)])
def test_f16_splits_as_bf16_or_not_at_all(plan, M, N, K, split):
    """f16 on int8 weights: bf16's split where it measured faster, else whole tiles (and then the query
    still covers bf16)."""
    bf16, f16 = (plan.need(1, dt, M, N, K, 256) for dt in (0, 1))
    assert f16 == (bf16 if split else 0) and 0 < bf16 == plan.told(1, M, N, K, 256) <= plan.most()
