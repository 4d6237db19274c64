"""Run by test_gpu_ln.py in a process of its own: when a checked GEMM+LayerNorm returns, its result is there for a copy on another
stream that does not wait for this one's, and in host memory for the calling thread, however long the stream's earlier work keeps
the call waiting.  The same steps without the check find the old contents, so nothing else orders the copy.  And what the call
saves is not left to whoever synchronises behind it."""
import ctypes
import os
import sys
import threading
import time

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "general-nvgpu-testing_amd"))
from beam import _C  # noqa: E402

L, BF16 = _C.lib, torch.bfloat16
ONE_TILE = _C.TileConfig(64, 64, 32, 32, 0, 0).to_c()
FRONT_K = 1 << 17


class Caller:
    """Operands and streams of one thread; torch's streams wait for no other, not even the default one."""

    def __init__(self, M, N, K, seed):
        gen = torch.Generator(device="cuda").manual_seed(seed)
        normal = lambda *shape: torch.randn(*shape, generator=gen, device="cuda", dtype=BF16)
        self.shape = M, N, K
        self.a, self.b, self.gamma, self.beta = normal(M, K), normal(N, K) * K ** -0.5, 1 + 0.1 * normal(N), 0.1 * normal(N)
        self.y, self.host = torch.empty(M, N, device="cuda", dtype=BF16), torch.empty(M, N, dtype=BF16, pin_memory=True)
        self.ws = torch.empty(L.beam_gemmrc_ln_workspace_bytes_for(M, N, K, None, _C.LN_AUTO), device="cuda", dtype=torch.uint8)
        self.front, self.front_c = torch.zeros(64, FRONT_K, device="cuda", dtype=BF16), torch.empty(64, 64, device="cuda", dtype=BF16)
        self.stream, self.other = torch.cuda.Stream(), torch.cuda.Stream()
        torch.cuda.synchronize()
        self.want = None

    def launch(self, y, fronts, checked):
        """`fronts` products of a single workgroup (the rest of the device stays free), then the call; True if it fell back."""
        M, N, K = self.shape
        st, fell_back = ctypes.c_void_p(self.stream.cuda_stream), ctypes.c_int()
        for _ in range(fronts):
            f = self.front.data_ptr()
            _C._check(L.beam_gemmrc(f, f, self.front_c.data_ptr(), 64, 64, FRONT_K, _C.BF16, ctypes.byref(ONE_TILE), st))
        args = [self.a.data_ptr(), self.b.data_ptr(), self.gamma.data_ptr(), self.beta.data_ptr(), ctypes.c_float(1e-5), y.data_ptr(), M, N, K,
                _C.BF16, None]
        if checked:
            _C._check(L.beam_gemmrc_ln_checked(*args, self.ws.data_ptr(), self.ws.numel(), st, ctypes.byref(fell_back)))
        else:
            _C._check(L.beam_gemmrc_ln_ex(*args, _C.LN_AUTO, self.ws.data_ptr(), self.ws.numel(), st))
        return bool(fell_back.value)

    def copied(self, fronts, checked):
        """What a copy on the other stream finds right after the call."""
        with torch.cuda.stream(self.other):
            self.y.fill_(float("nan"))
        self.other.synchronize()
        assert not self.launch(self.y, fronts, checked), f"{self.shape} fell back"
        with torch.cuda.stream(self.other):
            self.host.copy_(self.y, non_blocking=True)
        self.other.synchronize()
        got = self.host.clone()
        self.stream.synchronize()
        return got


def same(x, y):
    return bool((x.view(torch.int16) == y.view(torch.int16)).all())


# (one launch's workgroups leave room for the others': 13 to 65 of them)
callers = [Caller(*shape, seed) for seed, shape in enumerate([(96, 200, 72), (300, 264, 1000), (130, 520, 256), (64, 1000, 520)])]
for c in callers:
    c.copied(0, True)
    c.want = c.copied(0, True)
    assert c.want.isfinite().all()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    start.record(c.stream)
    stale = c.copied(1, False)
    end.record(c.stream)
    end.synchronize()
    print(f"{c.shape}: work in front of the call {start.elapsed_time(end):.2f} ms", flush=True)
    assert stale.isnan().all(), "the copy waits for the call by itself: this check would see nothing"
    for fronts in (0, 1, 6):  # the third beyond what the call watches for
        for rep in range(3):
            assert same(c.copied(fronts, True), c.want), (c.shape, fronts, rep)
    # Y in host memory, read by this thread
    for fronts in (0, 1):
        y = torch.full(c.y.shape, float("nan"), dtype=BF16, pin_memory=True)
        assert not c.launch(y, fronts, True) and same(y, c.want), (c.shape, fronts)

# A caller that synchronises behind the call pays what one does whose call has synchronised by itself (1.06 times it; without the
# event that the wait records 1.24)
M, N, K = 512, 1024, 1024
c = Caller(M, N, K, 9)
args = [t.data_ptr() for t in (c.a, c.b, c.gamma, c.beta)] + [ctypes.c_float(1e-5), c.y.data_ptr(), M, N, K, _C.BF16, None]
ws, fell_back = (c.ws.data_ptr(), c.ws.numel()), ctypes.c_int()
took = ([], [])
for _ in range(220):
    t0 = time.perf_counter()
    _C._check(L.beam_gemmrc_ln_checked(*args, *ws, None, ctypes.byref(fell_back)))
    _C._check(L.beam_sync(None))
    t1 = time.perf_counter()
    _C._check(L.beam_gemmrc_ln_ex(*args, _C.LN_AUTO, *ws, None))
    _C._check(L.beam_sync(None))
    _C._check(L.beam_sync(None))
    took[0].append(t1 - t0)
    took[1].append(time.perf_counter() - t1)
    assert not fell_back.value
checked, parts = (sorted(t[20:])[100] * 1e6 for t in took)
print(f"{c.shape}: checked and synchronised {checked:.1f} us, synchronised twice {parts:.1f} us", flush=True)
assert checked <= 1.15 * parts, (checked, parts)
torch.cuda.synchronize()

bad = []


def worker(c):
    for rep in range(20):
        if not same(c.copied(rep % 2, True), c.want):
            bad.append((c.shape, rep))


threads = [threading.Thread(target=worker, args=(c,)) for c in callers]
for t in threads:
    t.start()
for t in threads:
    t.join()
assert not bad, bad
print("checked calls OK")
