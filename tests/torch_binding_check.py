"""Run by test_gpu_torch_binding.py in a process of its own (torch has to be imported before beam): every operator through the
compiled binding and through the general path gives the same bits, and what the binding leaves alone is answered as before."""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "general-nvgpu-testing_amd"))
from beam import _C  # noqa: E402

native = _C._native
assert native is not None
calls = []


class Counting:
    """The binding, noting what it answers."""

    def __getattr__(self, name):
        def call(*args):
            status = getattr(native, name)(*args)
            calls.append((name, status))
            return status
        return call


def both(what, f, outs, handled=True):
    got = []
    for binding in (Counting(), None):
        _C._native = binding
        for o in outs:
            o.fill_(float("nan"))
        calls.clear()
        f()
        torch.cuda.synchronize()
        if binding is not None:
            assert bool(calls and calls[-1][1] >= 0) == handled, (what, calls)
        got.append([o.clone() for o in outs])
    assert all((x.view(torch.int16) == y.view(torch.int16)).all() for x, y in zip(*got)), what


def ordered(what, f, a, c):
    """f's operand is written by work in front of it that is still running when f returns; launched on another stream, f would
    read what was there before."""
    late = torch.full_like(a, float("nan"))
    big = torch.zeros(1 << 28, device="cuda", dtype=torch.int32)
    torch.cuda.synchronize()
    _C._native = Counting()
    calls.clear()
    f(a)
    want = c.clone()
    torch.cuda.synchronize()
    for _ in range(8):  # 8 x 2 GiB of traffic, milliseconds
        big.add_(1)
    late.copy_(a)
    f(late)
    done = torch.cuda.Event()
    done.record()
    assert not done.query(), "the work in front is too short to tell"
    torch.cuda.synchronize()
    assert len(calls) == 2 and all(s >= 0 for _, s in calls), (what, calls)
    assert (c.view(torch.int16) == want.view(torch.int16)).all(), what


def same_error(what, f):
    said = []
    for binding in (Counting(), None):
        _C._native = binding
        try:
            f()
        except Exception as e:  # noqa: BLE001
            said.append((type(e), str(e)))
    assert len(said) == 2 and said[0] == said[1], (what, said)


for dtype in (torch.float16, torch.bfloat16):
    for M, N, K in ((65, 72, 200), (1, 1000, 71), (300, 520, 4096)):
        a, b, c = (torch.randn(s, device="cuda", dtype=dtype) for s in ((M, K), (N, K), (M, N)))
        bt = b.t().contiguous()
        g, be = torch.randn(N, device="cuda", dtype=dtype), torch.randn(N, device="cuda", dtype=dtype)
        x = torch.randn(33, 31, device="cuda", dtype=dtype)
        y = torch.empty_like(x)
        both("gemmrc", lambda: _C.gemmrc(a, b, c), [c])
        both("gemmrc, parameters", lambda: _C.gemmrc(torch.nn.Parameter(a), b, c=c), [c])
        both("matmul", lambda: _C.matmul(a, bt, c), [c])
        _C._native = None
        _C.gemmrc_splitk(a, b, c)  # the workspaces grow on the general path
        _C.gemmrc_ln(a, b, c, g, be)
        both("split-K", lambda: _C.gemmrc_splitk(a, b, c), [c])
        for check in (True, False):
            both(f"LayerNorm, check {check}", lambda: _C.gemmrc_ln(a, b, c, g, be, check=check), [c])
        both("GEMM and SiLU", lambda: _C.parallel_gemmrc_silu(a, b, c, x, y), [c, y])
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            both("another stream", lambda: _C.gemmrc(a, b, c), [c])
            ordered("gemmrc behind its stream's work", lambda x: _C.gemmrc(x, b, c), a, c)
            ordered("matmul behind its stream's work", lambda x: _C.matmul(x, bt, c), a, c)
            ordered("split-K behind its stream's work", lambda x: _C.gemmrc_splitk(x, b, c), a, c)
            ordered("LayerNorm behind its stream's work", lambda x: _C.gemmrc_ln(x, b, c, g, be, check=False), a, c)
            ordered("SiLU behind its stream's work", lambda x: _C.parallel_gemmrc_silu(x, b, c, x, torch.empty_like(x)), a, c)
        view = torch.randn(M + 1, K, device="cuda", dtype=dtype)[1:]  # contiguous, at another offset
        both("a view", lambda: _C.gemmrc(view, b, c), [c])
        both("a named tile", lambda: _C.gemmrc(a, b, c, config=_C.TileConfig(64, 64, 32, 32)), [c], handled=False)

    class Sub(torch.Tensor):
        pass

    both("a subclass", lambda: _C.gemmrc(a.as_subclass(Sub), b, c), [c], handled=False)
    wide = torch.randn(M, 2 * K, device="cuda", dtype=dtype)
    same_error("rows apart", lambda: _C.gemmrc(wide[:, :K], b, c))
    same_error("on the CPU", lambda: _C.gemmrc(a.cpu(), b, c))
    same_error("fp32", lambda: _C.gemmrc(a.float(), b, c))
    same_error("two types", lambda: _C.gemmrc(a, b.to(torch.float16 if dtype == torch.bfloat16 else torch.bfloat16), c))
    same_error("K differs", lambda: _C.gemmrc(a[:, :-1].contiguous(), b, c))
    same_error("shape of c", lambda: _C.matmul(a, bt, c[:-1]))
    same_error("one dimension", lambda: _C.gemmrc(a[0], b, c))
    same_error("gamma", lambda: _C.gemmrc_ln(a, b, c, g[:-1], be))
    same_error("eps", lambda: _C.gemmrc_ln(a, b, c, g, be, eps=-1.0))
    same_error("elements", lambda: _C.parallel_gemmrc_silu(a, b, c, x, y[:-1]))
    same_error("alignment", lambda: _C.parallel_gemmrc_silu(a, b, c, x.view(-1)[1:], y.view(-1)[1:]))
    same_error("no tensor", lambda: _C.gemmrc(a, b, None))
    same_error("batched", lambda: torch.vmap(lambda t: _C.gemmrc(t, b, c))(torch.stack([a, a])))
print("torch binding OK")
