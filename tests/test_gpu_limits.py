"""Padded host arrays, and what is left of a call that ran out of memory."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from quantum_package_amd.hamiltonian import fci_space, synthetic_hamiltonian
from test_gpu_sigma import _say

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
