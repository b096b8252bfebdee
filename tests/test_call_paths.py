"""call_paths.cpp (the decode step's calls with their checks in C++) against the general way of kernels.py: over the
forms both accept the results are the same bits; forms that need a conversion or a copy, and wrong ones, are left to the
general way, which gives the results and exceptions it always gave."""
import ctypes
import signal
import sys
import threading
import time

import pytest
import torch

import quant
import workloads as wl
from native import kernels

DEV = "cuda:0"


class _General:
    """Every question answered with None: the general way."""

    def __getattr__(self, name):
        return lambda *a: None


class _Watch:
    """The C++ calls, noting each by name and whether it answered."""

    def __init__(self, mod):
        self.mod, self.answered = mod, []

    def __getattr__(self, name):
        def call(*a):
            r = getattr(self.mod, name)(*a)
            self.answered.append((name, r is not None))
            return r
        return call


def both(monkeypatch, fn):
    """(result with the C++ calls, result the general way, whether a C++ call answered)."""
    fast, slow, calls = both_calls(monkeypatch, fn)
    return fast, slow, any(answered for _, answered in calls)


def both_calls(monkeypatch, fn):
    """(result with the C++ calls, result the general way, [(C++ call, whether it answered)])."""
    watch = _Watch(kernels._calls())
    monkeypatch.setattr(kernels, "_native_calls", watch)
    fast = fn()
    monkeypatch.setattr(kernels, "_native_calls", _General())
    slow = fn()
    monkeypatch.setattr(kernels, "_native_calls", watch.mod)
    return fast, slow, watch.answered


def equal(a, b):
    a, b = (x if isinstance(x, tuple) else (x,) for x in (a, b))
    return len(a) == len(b) and all((x is None and y is None) or torch.equal(x, y) for x, y in zip(a, b))


def test_host_tensors_and_wrong_counts_are_not_answered():
    mod = kernels._calls()
    x = torch.zeros(2, 64)
    assert mod.linear(x, 1, x, None, None, 2, 64, None, None, None, None, 0.0, False, False, None, None, 0) is None
    assert mod.norm(False, x, torch.ones(64), 1e-6, 0) is None
    assert mod.paged_decode(x, x, x, x, x, 16, 0, None, None, None, 0) is None
    assert mod.norm(False, "x", torch.ones(64), 1e-6, 0) is None
    with pytest.raises(TypeError):
        mod.linear(x)


def test_a_library_of_another_interface_is_refused():
    """The addresses come from whichever library is loaded: the prototypes compiled in must be that library's."""
    mod, lib = kernels._calls(), kernels.load().lib
    real = {n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in kernels.CALLED}
    other = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: lib.rk_abi_version() - 1)
    with pytest.raises(ImportError, match="ABI version"):
        mod.init({**real, "rk_abi_version": ctypes.cast(other, ctypes.c_void_p).value}, print)
    with pytest.raises(KeyError):
        mod.init({n: a for n, a in real.items() if n != "rk_abi_version"}, print)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bf16", "int8", "int4"])
@pytest.mark.parametrize("M,N,K", [(1, 96, 256), (5, 2048, 2048), (8, 4096, 512), (16, 100, 1056), (3, 64, 6144)])
def test_linears(backend, monkeypatch, kind, M, N, K):
    g = torch.Generator(device=DEV).manual_seed(N + K)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    w = r(N, K) / K ** 0.5
    w = w.bfloat16() if kind == "bf16" else quant.quantize(w, kind)
    x, b, res, nw = r(M, K), r(N), r(M, N), r(K)
    wide = r(M, K + 64)
    ss = (x * x).view(M, K // 16, 16).sum(-1)
    backend.linear(x, w), backend.swiglu(x, w)                  # the shared workspace and counters exist
    forms = [lambda: backend.linear(x, w), lambda: backend.linear(x, w, b, res), lambda: backend.linear_ss(x, w, residual=res),
             lambda: backend.linear(wide[:, :K], w, b), lambda: backend.linear_ss(wide[:, 32:32 + K], w, b)]
    if N % 16 == 0:
        forms.append(lambda: backend.swiglu(x, w))
    for f in forms:
        fast, slow, used = both(monkeypatch, f)
        assert used and equal(fast, slow)
    # the norm inside the linear: one call, answered; elsewhere that call is declined, and the two parts follow
    inside = M <= 8 and K % 256 == 0 and K <= 2048
    for f, whole in ((lambda: backend.rms_norm_linear(x, ss, nw, 1e-6, w, b), inside),
                     (lambda: backend.rms_norm_swiglu(x, ss, nw, 1e-6, w), inside and N % 16 == 0)):
        fast, slow, calls = both_calls(monkeypatch, f)
        assert equal(fast, slow)
        if whole:
            assert calls == [("linear", True)]
        else:
            assert calls[0] == ("linear", False) and ("norm" in [n for n, _ in calls]) == (not inside)
    # left to the general way
    for f in (lambda: backend.linear(x.double(), w), lambda: backend.linear(wide[:, 1:K + 1], w),
              lambda: backend.linear(x, w, b.bfloat16()), lambda: backend.linear(x, w, None, res.double())):
        fast, slow, used = both(monkeypatch, f)
        assert not used and equal(fast, slow)
    for f in (lambda: backend.linear(x[:, :-32], w), lambda: backend.linear(x, w, residual=r(M + 1, N)),
              lambda: backend.linear(x.cpu(), w)):
        for mod in (kernels._calls(), _General()):
            monkeypatch.setattr(kernels, "_native_calls", mod)
            with pytest.raises((ValueError, RuntimeError)):
                f()
        monkeypatch.undo()


@pytest.mark.gpu
def test_row_norms(backend, monkeypatch):
    x, w = torch.randn(7, 2048, device=DEV), torch.randn(2048, device=DEV)
    for f, want in ((lambda: backend.rms_norm(x, w, 1e-6), True), (lambda: backend.layer_norm(x[:, :100], w[:100], 1e-5), True),
                    (lambda: backend.rms_norm(x[:1], w, 1e-6), True), (lambda: backend.rms_norm(x.bfloat16(), w, 1e-6), False),
                    (lambda: backend.rms_norm(x.view(7, 8, 256), w[:256], 1e-6), False),
                    (lambda: backend.rms_norm(x, w.bfloat16(), 1e-6), False), (lambda: backend.rms_norm(x.T, w[:7], 1e-6), False)):
        fast, slow, used = both(monkeypatch, f)
        assert used == want and equal(fast, slow)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_paged_decode(backend, monkeypatch, dtype):
    c = wl.paged_decode_case([1, 40, 300, 17], 64, 8, 2, 128, 16, dtype, seed=3).to(DEV)
    run = lambda q=c.q, gate=None, window=None, plan=None, lens=c.lens: backend.paged_attention(
        q, c.k_pool, c.v_pool, c.tables, lens, 16, window, gate=gate, plan=plan)
    run()
    plan = backend.decode_plan(c.tables, c.lens, 16, 8, 2, 128, c.k_pool.shape[0])
    wide = torch.cat([c.gate, c.gate], 1)
    for f, want in ((run, True), (lambda: run(gate=c.gate), True), (lambda: run(gate=wide[:, 1024:], window=33), True),
                    (lambda: run(gate=c.gate, plan=plan), True), (lambda: run(q=c.q.bfloat16()), False),
                    (lambda: run(gate=c.gate.view(4, 8, 128)), False), (lambda: run(gate=wide[:, 1:1025]), False)):
        fast, slow, used = both(monkeypatch, f)
        assert used == want and equal(fast, slow)
    for bad in (lambda: run(lens=c.lens.long()), lambda: run(window=5, plan=plan), lambda: run(lens=c.lens[:3])):
        with pytest.raises((TypeError, ValueError)):
            bad()


@pytest.mark.gpu
def test_deltanet_step_and_attention_prep(backend, monkeypatch):
    c = wl.c2_deltanet_step(batch=3, max_seqs=5, n_linear=2, slot=1).to(DEV)
    y = torch.cat([c.qkv, c.z, c.b, c.a], 1)
    C, Z, H = c.qkv.shape[1], c.z.shape[1], c.b.shape[1]
    cols = lambda t: (t[:, :C], t[:, C:C + Z], t[:, C + Z:C + Z + H], t[:, C + Z + H:])

    def step(inputs, seqs=c.seq_index):
        S, conv = c.S.clone(), c.conv.clone()
        o = kernels.deltanet_decode(*inputs, conv, S, seqs, 1, c.conv_w, c.A_log, c.dt_bias, c.norm_w, c.eps, c.dims)
        return o, S, conv
    for f, want in ((lambda: step((c.qkv, c.z, c.b, c.a)), True), (lambda: step(cols(y)), True),
                    (lambda: step(tuple(t[:1] for t in cols(y)), c.seq_index[:1]), True),
                    (lambda: step((c.qkv, c.z, c.b, y[:, -H:])), False),                 # b and a at different strides
                    (lambda: step(cols(y.double())), False), (lambda: step(cols(y), c.seq_index.long()), False)):
        fast, slow, used = both(monkeypatch, f)
        assert used == want and equal(fast, slow)
    with pytest.raises(ValueError):
        kernels.deltanet_decode(c.qkv, c.z, c.b, c.a, c.conv, c.S, c.seq_index, 2, c.conv_w, c.A_log, c.dt_bias, c.norm_w,
                                c.eps, c.dims)

    Hq, Hkv, d = 8, 2, 128
    yp = torch.randn(6, (2 * Hq + 2 * Hkv) * d + 8, device=DEV)
    qw, kw = torch.randn(d, device=DEV), torch.randn(d, device=DEV)
    pos = torch.arange(6, device=DEV, dtype=torch.int32) * 11
    slots = torch.tensor([5, 17, 40, 1, 99, 63], device=DEV)
    for dt in (torch.float32, torch.bfloat16):
        def prep(yy, rot=64, p=pos):
            k, v = torch.zeros(8, 16, Hkv, d, device=DEV, dtype=dt), torch.zeros(8, 16, Hkv, d, device=DEV, dtype=dt)
            q, gate = backend.attention_prep(yy, qw, kw, 1e-6, p, 1e6, rot, (Hq, Hkv, d), k, v, slots)
            return q, gate, k, v
        for f, want in ((lambda: prep(yp), True), (lambda: prep(yp[:, 8:], 0), True), (lambda: prep(yp.bfloat16()), False),
                        (lambda: prep(yp[:, 1:-1]), False)):
            fast, slow, used = both(monkeypatch, f)
            assert used == want and equal(fast, slow)
    with pytest.raises(ValueError):
        prep(yp, p=pos.long())


@pytest.mark.gpu
def test_out_of_memory_is_torchs_own_exception(backend):
    """An engine catches torch.OutOfMemoryError to evict and try again. Each call below is answered in C++ and its
    output (16 MiB) does not fit the limit set for the process; the workspaces it needs exist already."""
    x, nw = torch.zeros(2048, 2048, device=DEV), torch.ones(2048, device=DEV)
    w, xr = torch.zeros(1 << 18, 32, dtype=torch.bfloat16, device=DEV), torch.zeros(16, 32, device=DEV)
    q, pool = torch.zeros(1024, 16, 256, device=DEV), torch.zeros(1, 16, 4, 256, device=DEV)
    tables, lens = (f(1024, *s, dtype=torch.int32, device=DEV) for f, s in ((torch.zeros, (1,)), (torch.ones, ())))
    calls = [lambda: backend.rms_norm(x, nw, 1e-6), lambda: backend.linear(xr, w),
             lambda: backend.paged_attention(q, pool, pool, tables, lens, 16)]
    for f in calls:
        f()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / torch.cuda.mem_get_info()[1])
    held = []
    try:
        with pytest.raises(torch.OutOfMemoryError):
            while True:                                         # what is left of segments in use
                held.append(torch.empty(1 << 22, device=DEV))
        for f in calls:
            with pytest.raises(torch.OutOfMemoryError):
                f()
    finally:
        held.clear()
        torch.cuda.set_per_process_memory_fraction(1.0)
    for f in calls:
        f()


@pytest.mark.gpu
def test_other_threads_run_during_a_launch(backend, monkeypatch):
    """A launch may wait for room in the device's queue. pause() in the place of rk_rms_norm stands for that: it returns
    only when a signal comes, which another Python thread sends (a timer ends it if that thread cannot run)."""
    x, w = torch.zeros(2, 64, device=DEV), torch.ones(64, device=DEV)
    mod, lib = kernels._calls(), kernels.load().lib
    address = lambda f: ctypes.cast(f, ctypes.c_void_p).value
    real = {n: address(getattr(lib, n)) for n in kernels.CALLED}

    def failed(entry, status):
        raise RuntimeError(f"{entry}: {status}")
    order, main, sent = [], threading.get_ident(), threading.Event()

    def other():
        sent.wait()
        order.append("other thread")
        time.sleep(0.2)                                         # the main thread gets to pause()
        signal.pthread_kill(main, signal.SIGUSR1)
    interval = sys.getswitchinterval()
    old = [signal.signal(s, lambda *a: None) for s in (signal.SIGUSR1, signal.SIGALRM)]
    thread = threading.Thread(target=other)
    try:
        mod.init({**real, "rk_rms_norm": address(ctypes.CDLL(None).pause)}, failed)
        thread.start()
        signal.setitimer(signal.ITIMER_REAL, 5.0)
        sys.setswitchinterval(60.0)                             # the GIL changes hands only where it is given up
        sent.set()
        with pytest.raises(RuntimeError, match="rk_rms_norm: -1"):
            mod.norm(False, x, w, 1e-6, 0)
        order.append("call returned")
    finally:
        sys.setswitchinterval(interval)
        signal.setitimer(signal.ITIMER_REAL, 0)
        sent.set()
        thread.join()
        for s, h in zip((signal.SIGUSR1, signal.SIGALRM), old):
            signal.signal(s, h)
        monkeypatch.setattr(kernels, "_native_calls", None)
        kernels._calls()                                        # the entry points again
    assert order == ["other thread", "call returned"]
