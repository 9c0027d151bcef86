"""Padded host arrays, and what is left of a call that ran out of memory."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from quantum_package_amd.hamiltonian import fci_space, synthetic_hamiltonian
from test_gpu_sigma import _say
from test_gpu_sigma_paths import failing_allocations

pytestmark = pytest.mark.gpu


@pytest.fixture()
def ctx():
    from quantum_package_amd.api import Context
    c = Context(0)
    yield c
    c.close()


def _davidson(ctx, u, sze, n_st, n_diag):
    """qpx_davidson on u (dim_in, n_diag) column-major, in place: energies"""
    e, s2, ns = np.zeros(n_diag), np.zeros(n_diag), (C.c_int * 2)()
    dp = C.POINTER(C.c_double)
    ctx._check(ctx.L.qpx_davidson(ctx.ptr, n_st, n_diag, 1e-10, 8, 0, 0, 0, 1e-7, 1, u.ctypes.data_as(dp), u.shape[0],
                                  e.ctypes.data_as(dp), s2.ctypes.data_as(dp), C.cast(ns, C.POINTER(C.c_int))))
    return e


@pytest.mark.parametrize("pad", [0, 3])
def test_davidson_of_padded_columns(ctx, pad):
    """dim_in > n_det: the rows behind a column's determinants are neither read
    nor written; eigenvalues of the dense matrix to 1e-9."""
    ctx.set_hamiltonian(synthetic_hamiltonian(8, 4, 3, seed=4))
    dets = fci_space(8, 4, 3)[::7]
    n = dets.shape[0]
    _say(f"[davidson padded] n_det={n} pad={pad}")
    ctx.set_wavefunction(dets)
    Hm = np.concatenate([ctx.H_S2_u_0_nstates(np.eye(n)[:, k:k + 4])[0] for k in range(0, n, 4)], axis=1)
    u = np.full((n + pad, 4), np.nan, order="F")
    u[:n, :2] = np.random.default_rng(1).standard_normal((n, 2))
    e = _davidson(ctx, u, n, 2, 4)
    assert np.max(np.abs(e[:2] - np.linalg.eigvalsh(0.5 * (Hm + Hm.T))[:2])) < 1e-9
    assert np.isfinite(u[:n]).all() and np.isnan(u[n:]).all()


def test_hamiltonian_without_memory(ctx):
    """A Hamiltonian whose arrays did not fit leaves none, and no wavefunction:
    calls say so until both are set again."""
    from quantum_package_amd.api import QpxError
    H, dets = synthetic_hamiltonian(8, 4, 3, seed=4), fci_space(8, 4, 3)
    u = np.random.default_rng(1).standard_normal(dets.shape[0])
    ctx.set_hamiltonian(H)
    ctx.set_wavefunction(dets)
    want = ctx.H_S2_u_0_nstates(u)
    _say("[hamiltonian without memory] M=12 after M=8")
    with failing_allocations(ctx, 20000):   # 12 orbitals: the pair matrix takes 48,672 bytes
        with pytest.raises(QpxError, match="memory"):
            ctx.set_hamiltonian(synthetic_hamiltonian(12, 4, 3, seed=4))
    with pytest.raises(QpxError):
        ctx.H_S2_u_0_nstates(u)
    with pytest.raises(QpxError):
        ctx.set_wavefunction(dets)
    ctx.set_hamiltonian(H)
    ctx.set_wavefunction(dets)
    assert all(np.array_equal(a, b) for a, b in zip(ctx.H_S2_u_0_nstates(u), want))


@pytest.mark.parametrize("above", [1000, 40000, 100000, 1000000])
def test_network_batch_without_memory(above):
    """A batch whose buffers did not fit, at whichever of them it failed, leaves
    the network as it was: the next batch trains and predicts as in a network
    that never saw it."""
    from quantum_package_amd.api import BlockMLP, QpxError
    rng = np.random.default_rng(3)

    def batch(n):
        d = np.stack([rng.integers(0, 20, n), rng.integers(0, 20, n), rng.integers(0, 3, n), rng.integers(0, 5, n)],
                     axis=1).astype(np.int32)
        return d, rng.standard_normal((n, 3)).astype(np.float32), rng.standard_normal(n).astype(np.float32)

    small, large = batch(64), batch(5000)
    _say(f"[network without memory] above {above}")
    m, fresh = BlockMLP(n_orb=20, seed=1), BlockMLP(n_orb=20, seed=1)
    for net in (m, fresh):
        net.train_step(*small, 0.0)
    with failing_allocations(m, above):
        with pytest.raises(QpxError, match="memory"):
            m.train_step(*large, 0.0)
    for net in (m, fresh):
        net.train_step(*small, 0.0)
    assert np.array_equal(m.get("W2", grad=True), fresh.get("W2", grad=True))
    assert np.array_equal(m.predict(*large[:2]), fresh.predict(*large[:2]))
    m.close()
    fresh.close()
