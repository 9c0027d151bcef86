"""Device sigma calls on callers' streams: what later calls of the context may
and may not do to calls that are still queued and to captured graphs."""
from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest

from quantum_package_amd.hamiltonian import fci_space, synthetic_hamiltonian
from hip_rt import CAPTURE_THREAD_LOCAL, Arr, Hip
from test_gpu_sigma import _say, _singles_space
from test_gpu_sigma_paths import failing_allocations

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    return Hip()


@pytest.fixture()
def ctx():
    from quantum_package_amd.api import Context
    c = Context(0)
    yield c
    c.close()


def _space(kind):
    """(M, na, nb, determinants): a product space or a selected one"""
    if kind == "product":
        return 10, 4, 3, fci_space(10, 4, 3)
    return 20, 3, 2, _singles_space(20, 3, 2, 0.9, 1)


class Vectors:
    """u, v, s of a device sigma call (bilinear order, state-fastest)"""

    def __init__(self, hip, n, nst, prec, seed):
        dt = np.float64 if prec == 0 else np.float32
        a = np.random.default_rng(seed).standard_normal((n, nst)).astype(dt)
        self.nst, self.prec = nst, prec
        self.u, self.v, self.s = Arr(hip, a), Arr(hip, np.zeros_like(a)), Arr(hip, np.zeros_like(a))

    def sigma(self, ctx, stream):
        ctx._check(ctx.L.qpx_sigma_device(ctx.ptr, self.prec, self.nst, self.u.p, self.v.p, self.s.p, stream))

    def out(self):
        return self.v.get(), self.s.get()

    def clear(self):
        z = np.zeros(self.v.shape, dtype=self.v.dtype)
        self.v.put(z)
        self.s.put(z)

    def free(self):
        for a in (self.u, self.v, self.s):
            a.free()


def _same(x, y):
    return all(np.array_equal(a, b) for a, b in zip(x, y))


def _prepare(ctx, kind):
    M, na, nb, dets = _space(kind)
    ctx.set_hamiltonian(synthetic_hamiltonian(M, na, nb, seed=4))
    ctx.set_wavefunction(dets)
    return dets.shape[0]


@pytest.mark.parametrize("what", ["wavefunction", "hamiltonian"])
@pytest.mark.parametrize("path", [1, 3, 4, 5])
def test_new_inputs_wait_for_queued_calls(ctx, hip, path, what):
    """A wavefunction of the same sizes (every array is reused) or another
    Hamiltonian, set while calls are queued on a caller's stream: the queued
    calls give what they give alone, bit for bit."""
    M, na, nb, dets = _space("product" if path in (1, 4) else "selected")
    other = dets[:, :, 0].copy()
    lo, hi = np.uint64(1) << np.uint64(M - 2), np.uint64(1) << np.uint64(M - 1)
    swap = ((other & lo) != 0) ^ ((other & hi) != 0)       # the two highest orbitals trade places
    other = np.where(swap, other ^ lo ^ hi, other)[:, :, None]
    _say(f"[sigma queued] path={path} new {what} n_det={dets.shape[0]}")
    ctx.set_hamiltonian(synthetic_hamiltonian(M, na, nb, seed=4))
    ctx.set_wavefunction(dets)
    ctx._force_sigma_path(path)
    st = hip.stream()
    x = Vectors(hip, dets.shape[0], 4, 0, 1)
    x.sigma(ctx, st)
    hip.sync()
    alone = x.out()
    for _ in range(3):
        x.clear()
        ctx.set_hamiltonian(synthetic_hamiltonian(M, na, nb, seed=4))
        ctx.set_wavefunction(dets)
        for _ in range(50):
            x.sigma(ctx, st)
        if what == "wavefunction":
            ctx.set_wavefunction(other)
        else:
            ctx.set_hamiltonian(synthetic_hamiltonian(M, na, nb, seed=5))
        hip.sync()
        assert _same(x.out(), alone)
    x.free()


@pytest.mark.parametrize("kind,kernels", [("product", 1), ("selected", 3)])
def test_failed_calls_leave_the_others_alone(ctx, hip, kind, kernels):
    """Calls that find no memory for the tables of another precision, or for
    the scratch of more vectors, fail or take another path; a graph captured
    before and the eager calls give the same bits as before, from the same
    kernels, and the calls that failed work once there is memory."""
    from quantum_package_amd.api import QpxError
    n = _prepare(ctx, kind)
    _say(f"[sigma failing] {kind} n_det={n}")
    ctx._force_sigma_path(kernels)
    st = hip.stream()
    x, single, more = Vectors(hip, n, 1, 0, 1), Vectors(hip, n, 1, 1, 2), Vectors(hip, n, 4, 0, 3)
    x.sigma(ctx, st)
    hip.sync()
    want = x.out()
    g = hip.capture(st, lambda: x.sigma(ctx, st))
    for call in (single, more):
        with failing_allocations(ctx, 1000):
            try:
                call.sigma(ctx, st)
                assert ctx._sigma_kernels() != kernels
            except QpxError as e:
                assert "memory" in str(e)
        hip.sync()
        x.clear()
        hip.replay(g, st)
        hip.sync()
        assert _same(x.out(), want)
        x.clear()
        x.sigma(ctx, st)
        hip.sync()
        assert ctx._sigma_kernels() == kernels and _same(x.out(), want)
    for call in (single, more):
        call.sigma(ctx, st)
        assert ctx._sigma_kernels() == kernels
    hip.sync()
    x.clear()
    hip.replay(g, st)
    hip.sync()
    assert _same(x.out(), want)
    hip.drop(g)
    for v in (x, single, more):
        v.free()


@pytest.mark.parametrize("what", ["sums", "entries"])
def test_bucket_calls_without_memory_walk(ctx, hip, what):
    """Sums that do not fit send that call alone to the walk; entries that do
    not fit send the wavefunction's calls there.  FP64 against the walk."""
    n = _prepare(ctx, "selected")
    _say(f"[sigma walk] {what} n_det={n}")
    x, st = Vectors(hip, n, 4, 0, 2), hip.stream()

    def run(path):
        x.clear()
        ctx._force_sigma_path(path)
        x.sigma(ctx, st)
        hip.sync()
        return x.out()

    def close(out):
        return all(np.max(np.abs(a - b)) < 1e-11 * np.max(np.abs(b)) for a, b in zip(out, want))

    dets = _space("selected")[3]
    ctx._force_sigma_path(3)
    ctx.set_wavefunction(dets[:50])   # leaves the integral tables, not the room for more entries
    ctx.H_S2_u_0_nstates(np.ones(50))
    ctx.set_wavefunction(dets)
    want = run(5)
    if what == "sums":
        assert close(run(3)) and ctx._sigma_kernels() == 3
        with failing_allocations(ctx, 1000):   # a captured call's sums are memory of its own
            g = hip.capture(st, lambda: x.sigma(ctx, st))
            assert ctx._sigma_kernels() == 5
        x.clear()
        hip.replay(g, st)
        hip.sync()
        assert _same(x.out(), want)
        hip.drop(g)
    else:
        with failing_allocations(ctx, 1 << 16):
            assert close(run(3)) and ctx._sigma_kernels() == 5
        assert close(run(3)) and ctx._sigma_kernels() == 5
        ctx.set_wavefunction(dets)
    assert close(run(3)) and ctx._sigma_kernels() == 3
    x.free()


@pytest.mark.parametrize("first", ["precision", "call"])
@pytest.mark.parametrize("kind,path", [("product", 1), ("product", 4), ("selected", 3), ("selected", 5)])
def test_captured_call_builds_its_tables(ctx, hip, kind, path, first):
    """A captured call may be the first of its precision, or of the
    wavefunction: replays give the bits of an eager call, which runs the same
    kernels."""
    n = _prepare(ctx, kind)
    _say(f"[sigma captured] {kind} path={path} first {first} n_det={n}")
    ctx._force_sigma_path(path)
    st = hip.stream()
    x, y = Vectors(hip, n, 2, 1, 1), Vectors(hip, n, 1, 0, 2)
    if first == "precision":
        y.sigma(ctx, st)
        hip.sync()
        before = y.out()
    g = hip.capture(st, lambda: x.sigma(ctx, st))
    assert ctx._sigma_kernels() == path
    x.clear()
    hip.replay(g, st)
    hip.sync()
    got = x.out()
    x.sigma(ctx, st)
    hip.sync()
    assert ctx._sigma_kernels() == path and _same(x.out(), got)
    for _ in range(3):
        y.sigma(ctx, st)
        x.clear()
        hip.replay(g, st)
        hip.sync()
        assert _same(x.out(), got)
    if first == "precision":
        assert _same(y.out(), before)
    hip.drop(g)
    x.free()
    y.free()


def test_kept_memory_is_bounded(ctx, hip):
    """811,801 determinants of 100 orbitals, 10a10b: 170M entries, whose set-up
    sorts in 4.7 GB of scratch.  After the set-up the scratch is what the sums
    need (1.4 GB); after the next wavefunction entries and scratch together are
    no more than 4 GiB, as before the large one."""
    M, na, nb = 100, 10, 10
    dets = _singles_space(M, na, nb, 2.0, 1)
    n = dets.shape[0]
    assert n == (1 + na * (M - na)) ** 2
    ctx.set_hamiltonian(synthetic_hamiltonian(M, na, nb, seed=4))
    ctx._force_sigma_path(3)
    ctx.set_wavefunction(dets[:50])
    ctx.H_S2_u_0_nstates(np.ones(50))
    small = hip.free_bytes()
    _say(f"[sigma memory] n_det={n}")
    ctx.set_wavefunction(dets)
    before = hip.free_bytes()
    ctx.H_S2_u_0_nstates(np.ones(n))
    assert ctx._sigma_kernels() == 3
    slots = n * (na * nb + na * (na - 1) + 2 * na)
    # entries 12 bytes, positions 4, sums 8; host vectors' staging 6 x 8 per determinant; 10 % for whole wavefronts
    assert before - hip.free_bytes() < 1.1 * 24 * slots + 48 * n + (256 << 20)
    ctx.set_wavefunction(dets[:50])
    assert small - hip.free_bytes() < (4 << 30) + 48 * n + (256 << 20)


@pytest.mark.parametrize("kind,path", [("product", 1), ("selected", 3)])
def test_calls_on_per_thread_streams(ctx, hip, kind, path):
    """Calls of several threads, one after another, each on its thread's default
    stream: one handle, as many streams, one scratch.  Every call gives what it
    gives alone, bit for bit."""
    n = _prepare(ctx, kind)
    ctx._force_sigma_path(path)
    _say(f"[sigma threads] {kind} n_det={n}")
    per_thread = ctypes.c_void_p(2)   # hipStreamPerThread
    xs = [Vectors(hip, n, 4, 0, seed) for seed in range(4)]
    alone = []
    for x in xs:
        x.sigma(ctx, per_thread)
        hip.sync()
        alone.append(x.out())
        x.clear()

    turn = [threading.Event() for _ in range(len(xs) + 1)]

    def enqueue(k):
        turn[k].wait()
        for _ in range(20):
            xs[k].sigma(ctx, per_thread)
        turn[k + 1].set()
        turn[-1].wait()   # the thread, and with it its stream, lasts as long as its work
        hip.sync()

    threads = [threading.Thread(target=enqueue, args=(k,)) for k in range(len(xs))]
    for t in threads:
        t.start()
    turn[0].set()
    for t in threads:
        t.join()
    for x, want in zip(xs, alone):
        assert _same(x.out(), want)
        x.free()


@pytest.mark.parametrize("kind,path", [("product", 1), ("selected", 3)])
def test_released_captures_give_their_memory_back(ctx, hip, kind, path):
    """A program that captures again and again holds no more memory than one
    capture needs; later captures replay as the first."""
    n = _prepare(ctx, kind)
    ctx._force_sigma_path(path)
    st = hip.stream()
    x = Vectors(hip, n, 4, 0, 1)
    x.sigma(ctx, st)
    hip.sync()
    want = x.out()

    def round_trip():
        g = hip.capture(st, lambda: x.sigma(ctx, st))
        x.clear()
        hip.replay(g, st)
        hip.sync()
        assert _same(x.out(), want)
        hip.drop(g)
        ctx.release_captured()

    round_trip()
    free = hip.free_bytes()
    _say(f"[sigma captures] {kind} n_det={n}")
    for _ in range(100):   # 100 scratch buffers: 240 MB for the product space, tens of MB for the other
        round_trip()
    assert free - hip.free_bytes() < 8 << 20
    x.free()


def test_set_up_beside_a_capture(ctx, hip):
    """Another thread sets up a context of its own, runs it and gives captures
    back while this one captures in the thread-local mode: both work."""
    from quantum_package_amd.api import Context
    n = _prepare(ctx, "product")
    x, st = Vectors(hip, n, 1, 0, 1), hip.stream()
    x.sigma(ctx, st)
    hip.sync()
    want = x.out()
    M, na, nb, dets = _space("selected")
    u = np.random.default_rng(2).standard_normal(dets.shape[0])
    got = []

    def other():
        c = Context(0)
        for _ in range(2):
            c.set_hamiltonian(synthetic_hamiltonian(M, na, nb, seed=4))
            c.set_wavefunction(dets)
            c._force_sigma_path(3)
            got.append(c.H_S2_u_0_nstates(u))
            c.release_captured()
        c.close()

    def enqueue():
        x.sigma(ctx, st)
        t = threading.Thread(target=other)
        t.start()
        t.join()

    _say(f"[sigma beside a capture] n_det={n}")
    g = hip.capture(st, enqueue, CAPTURE_THREAD_LOCAL)
    x.clear()
    hip.replay(g, st)
    hip.sync()
    assert _same(x.out(), want) and len(got) == 2 and _same(got[0], got[1])
    hip.drop(g)
    x.free()
