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


def test_flags_of_threads_and_their_bound(gpu, monkeypatch):
    """Calls that run at once have a flag each; past the bound the separate ops answer."""
    import threading
    from powershard_amd import ops
    x = torch.randn(4, 256, device=gpu).half()
    wq = torch.randint(-127, 128, (64, 256), dtype=torch.int8, device=gpu)
    s = torch.full((64,), 1e-3, device=gpu)
    bad = torch.full((64,), float("inf"), device=gpu).half()
    seen = {}

    def work(i):
        seen[i] = [ops.linear_w8a16_direct(x, 4, 256, wq, s, 256, 64, bad if (i + j) % 2 else None)[1] for j in range(50)]

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert all(seen[i] == [(i + j) % 2 == 0 for j in range(50)] for i in range(4))
    monkeypatch.setattr(ops, "_host_flags", {})
    monkeypatch.setattr(ops, "_MAX_FLAGS", 0)
    assert ops.linear_w8a16_direct(x, 4, 256, wq, s, 256, 64, None) is None


def test_flags_are_given_back(gpu, monkeypatch):
    """More threads than flags, all alive, one call each at a time: one flag serves them all.  A refused
    call gives its flag back, one whose wait failed does not (its kernel may still write there)."""
    import threading
    from powershard_amd import ops
    monkeypatch.setattr(ops, "_host_flags", {})
    x = torch.randn(4, 256, device=gpu).half()
    wq = torch.randint(-127, 128, (64, 256), dtype=torch.int8, device=gpu)
    s = torch.full((64,), 1e-3, device=gpu)
    one, done, seen = threading.Lock(), threading.Event(), []

    def work():
        with one:
            seen.append(ops.linear_w8a16_direct(x, 4, 256, wq, s, 256, 64, None))
        done.wait(60)

    threads = [threading.Thread(target=work) for _ in range(ops._MAX_FLAGS + 6)]
    [t.start() for t in threads]
    while len(seen) < len(threads) and any(t.is_alive() for t in threads):
        threads[0].join(0.01)
    done.set()
    [t.join() for t in threads]
    assert len(seen) == len(threads) and all(r is not None and r[1] for r in seen)
    made, free = ops._host_flags[gpu.index]
    assert len(made) == len(free) == 1
    with pytest.raises(RuntimeError):            # 96 elements are not whole 64-element stages
        ops.linear_w8a16_direct(x[:, :96].contiguous(), 4, 96, wq[:, :96].contiguous(), s, 0, 64, None)
    assert len(made) == len(free) == 1

    def fail(self):
        raise RuntimeError("reported by the wait")

    with monkeypatch.context() as m:
        m.setattr(torch.cuda.Stream, "synchronize", fail)
        with pytest.raises(RuntimeError, match="by the wait"):
            ops.linear_w8a16_direct(x, 4, 256, wq, s, 256, 64, None)
    assert len(made) == 1 and not free
    assert ops.linear_w8a16_direct(x, 4, 256, wq, s, 256, 64, None)[1] and len(made) == 2
    torch.cuda.synchronize()   # (before the flags of this test go)
