"""Which kernels a sigma call runs, and what becomes of errors on the way."""
from __future__ import annotations

import contextlib

import numpy as np
import pytest

from quantum_package_amd.hamiltonian import Hamiltonian, fci_space, hf_determinant, synthetic_hamiltonian
from oracle import oracle as O
from test_gpu_sigma import BUCKETS, PRODUCT, _product_space, _random_space, _say, _singles_space

pytestmark = pytest.mark.gpu

STRINGS, SCAN, BUCKET, DENSE, WALK = 1, 2, 3, 4, 5
LAUNCH_FAILURE = 719   # a hipError_t that is not about memory


@pytest.fixture()
def ctx():
    from quantum_package_amd.api import Context
    c = Context(0)
    yield c
    c.close()


@contextlib.contextmanager
def failing_allocations(ctx, above, error=0):
    ctx.L.qpx_debug_fail_alloc(above, error)
    try:
        yield
    finally:
        ctx.L.qpx_debug_fail_alloc(-1, 0)


def _set(ctx, M, na, nb, dets):
    ctx.set_hamiltonian(synthetic_hamiltonian(M, na, nb, seed=4))
    ctx.set_wavefunction(dets)
    return np.random.default_rng(1).standard_normal((dets.shape[0], 2))


# of PRODUCT, the space with 26 orbitals is the dense map's: the integrals of
# 88 singles do not fit the string-driven kernel's LDS
@pytest.mark.parametrize("kind,M,na,nb,arg", [("product", *p) for p in PRODUCT if p[0] < 26] +
                         [("buckets", *p) for p in BUCKETS])
def test_forced_kernels_run(ctx, kind, M, na, nb, arg):
    """The spaces the kernels of sigma_fci.hip and sigma_pairs.hip are checked
    on are computed by them, in both precisions."""
    dets = _product_space(M, na, nb, arg, 7) if kind == "product" else _singles_space(M, na, nb, arg, M + 1)
    u = _set(ctx, M, na, nb, dets)
    _say(f"[sigma kernels] {kind} M={M} {na}a{nb}b n_det={dets.shape[0]}")
    for path, kernels in ((1, STRINGS),) if kind == "product" else ((3, BUCKET), (5, WALK)):
        ctx._force_sigma_path(path)
        for prec in (0, 1):
            ctx.H_S2_u_0_nstates(u, prec=prec)
            assert ctx._sigma_kernels() == kernels


def test_kernels_by_path(ctx):
    dets = fci_space(8, 4, 4)
    u = _set(ctx, 8, 4, 4, dets)
    for path, kernels in ((0, STRINGS), (1, STRINGS), (2, SCAN), (3, BUCKET), (4, DENSE), (5, WALK)):
        ctx._force_sigma_path(path)
        ctx.H_S2_u_0_nstates(u)
        assert ctx._sigma_kernels() == kernels


@pytest.mark.parametrize("path", [1, 3])
def test_errors_reach_the_caller(ctx, path):
    """Only the want of memory sends a call to another path; any other error
    of the set-up is the call's, and the next call is as if it had not been."""
    from quantum_package_amd.api import QpxError
    M, na, nb = (10, 4, 3) if path == 1 else (20, 3, 2)
    dets = fci_space(M, na, nb) if path == 1 else _singles_space(M, na, nb, 0.9, 1)
    u = _set(ctx, M, na, nb, dets)
    ctx._force_sigma_path(path)
    ctx.H_S2_u_0_nstates(u)
    _say(f"[sigma errors] path={path} n_det={dets.shape[0]}")
    with failing_allocations(ctx, 0, LAUNCH_FAILURE):
        with pytest.raises(QpxError):
            ctx.H_S2_u_0_nstates(u, prec=1)
    ctx.H_S2_u_0_nstates(u, prec=1)
    assert ctx._sigma_kernels() == path


@pytest.mark.parametrize("vector", ["noise", "HF and a tail"])
@pytest.mark.parametrize("M,na,nb,n", [(40, 5, 4, 6000), (96, 6, 6, 6000)])
def test_bucket_fp32_error(ctx, M, na, nb, n, vector):
    """An FP32 sigma by bucket is no further from the FP64 one than the walk's,
    which spreads a determinant's terms over the lanes of a wavefront."""
    dets = _random_space(M, na, nb, n, M)
    _set(ctx, M, na, nb, dets)
    rng = np.random.default_rng(2)
    u = rng.standard_normal((n, 2)) / np.sqrt(n)
    if vector != "noise":
        u *= 0.3
        u[np.nonzero((dets == hf_determinant(M, na, nb)).all((1, 2)))[0][0]] = 0.95
    u = u.astype(np.float32).astype(np.float64)
    _say(f"[sigma fp32 error] M={M} {na}a{nb}b n_det={n} {vector}")
    ctx._force_sigma_path(3)
    ref, by_bucket = ctx.H_S2_u_0_nstates(u), ctx.H_S2_u_0_nstates(u, prec=1)
    ctx._force_sigma_path(5)
    walk = ctx.H_S2_u_0_nstates(u, prec=1)
    for x, y, r in zip(by_bucket, walk, ref):
        assert np.linalg.norm(x - r) <= np.linalg.norm(y - r)


# complete spaces of few beta strings: measured 0.46, 0.92 and 0.73 of the
# string-driven kernels' time with the dense map, then 1.8, 2.0 and 1.9 of it;
# one alpha string and more beta strings than the dense map takes: 0.08 by bucket
@pytest.mark.parametrize("M,na,nb,nst,prec,kernels", [
    (20, 4, 1, 2, 1, DENSE), (14, 6, 1, 4, 0, DENSE), (14, 7, 0, 4, 0, DENSE), (16, 16, 6, 4, 0, BUCKET),
    (12, 6, 1, 4, 0, STRINGS), (14, 6, 2, 4, 0, STRINGS), (8, 4, 4, 4, 1, STRINGS)])
def test_few_beta_strings(ctx, M, na, nb, nst, prec, kernels):
    """The automatic path takes the faster kernels; its values are those of the
    forced paths (FP64: 1e-11 of the largest entry, FP32: 2e-5 of the norm)."""
    H = synthetic_hamiltonian(M, na, max(nb, 1), seed=4)
    ctx.set_hamiltonian(Hamiltonian(M=M, n_alpha=na, n_beta=nb, h=H.h, eri=H.eri, seed=H.seed))
    dets = fci_space(M, na, nb)
    ctx.set_wavefunction(dets)
    u = np.random.default_rng(1).standard_normal((dets.shape[0], nst))
    _say(f"[sigma few beta] M={M} {na}a{nb}b nst={nst} prec={prec} n_det={dets.shape[0]}")
    got = ctx.H_S2_u_0_nstates(u, prec=prec)
    assert ctx._sigma_kernels() == kernels
    ctx._force_sigma_path(DENSE if kernels == STRINGS else STRINGS)
    for x, r in zip(got, ctx.H_S2_u_0_nstates(u)):
        if prec == 0:
            assert np.max(np.abs(x - r)) < 1e-11 * max(1.0, np.max(np.abs(r)))
        else:
            assert np.linalg.norm(x - r) < 2e-5 * max(1.0, np.linalg.norm(r))


def test_product_spaces_in_turn(ctx):
    """Tables and connections of one wavefunction are laid out in the memory of
    the last: spaces of growing and shrinking string sets in one context, with
    few and with many partners per string, give the bits of a context of their
    own, in both precisions."""
    from quantum_package_amd.api import Context
    spaces = [(8, 4, 4), (4, 4, 2), (12, 4, 3), (6, 3, 1), (14, 6, 1), (8, 4, 4), (2, 1, 1), (12, 5, 3)]
    for M, na, nb in spaces:
        dets = fci_space(M, na, nb)
        _say(f"[sigma in turn] M={M} {na}a{nb}b n_det={dets.shape[0]}")
        own = Context(0)
        got = []
        for c in (ctx, own):
            u = _set(c, M, na, nb, dets)
            c._force_sigma_path(1)
            got.append([x for prec in (0, 1) for x in c.H_S2_u_0_nstates(u, prec=prec)])
            assert c._sigma_kernels() == STRINGS
        own.close()
        assert all(np.array_equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("kind,arg", [("product", (8, 4, 4, 0.0)), ("product", (12, 3, 2, 0.4)), ("product", (14, 6, 1, 0.0)),
                                      ("buckets", (20, 3, 2, 0.9)), ("buckets", (14, 3, 2, 0.7)), ("buckets", (70, 2, 1, 0.25))])
def test_infinities_stay_where_they_are(ctx, kind, arg, prec, bad):
    """An infinite or NaN entry of u reaches the determinants connected to its
    own and no others, and one state only, as with the scanning kernel; the
    other entries keep their values (FP64: 1e-11, FP32: 2e-5 of the largest)."""
    M, na, nb, x = arg
    dets = _product_space(M, na, nb, x, 7) if kind == "product" else _singles_space(M, na, nb, x, M + 1)
    u = _set(ctx, M, na, nb, dets)
    u[dets.shape[0] // 3, 0] = bad
    _say(f"[sigma not finite] {kind} M={M} {na}a{nb}b prec={prec} {bad} n_det={dets.shape[0]}")
    ctx._force_sigma_path(SCAN)
    want = ctx.H_S2_u_0_nstates(u)
    ctx._force_sigma_path(1 if kind == "product" else 3)
    got = ctx.H_S2_u_0_nstates(u, prec=prec)
    assert ctx._sigma_kernels() == (STRINGS if kind == "product" else BUCKET)
    for x, r in zip(got, want):
        ok = np.isfinite(r)
        assert np.array_equal(np.isfinite(x), ok) and not ok.all()
        assert np.max(np.abs(x[ok] - r[ok])) < (1e-11 if prec == 0 else 2e-5) * np.max(np.abs(r[ok]))


def _against_oracle(ctx, M, na, nb, dets, nst, path, kernels):
    """FP64 to 1e-11 of the largest entry, FP32 to 2e-5 of the norm"""
    H = synthetic_hamiltonian(M, na, nb, seed=77)
    ctx.set_hamiltonian(H)
    ctx.set_wavefunction(dets)
    u = np.random.default_rng(5).standard_normal((dets.shape[0], nst))
    want = O.sigma(O.Ham(H), O.Bilinear(dets), u)
    ctx._force_sigma_path(path)
    for prec in (0, 1):
        for x, r in zip(ctx.H_S2_u_0_nstates(u, prec=prec), want):
            if prec == 0:
                assert np.max(np.abs(x - r)) < 1e-11 * max(1.0, np.max(np.abs(r)))
            else:
                assert np.linalg.norm(x - r) < 2e-5 * max(1.0, np.linalg.norm(r))
        assert ctx._sigma_kernels() == kernels


# by the most alpha singles a string has: up to 48, 64 and 96, and sets that are
# no product space, which the automatic path sends to the dense map
@pytest.mark.parametrize("M,na,nb,n,nst,path", [
    (8, 4, 4, None, 4, 4), (14, 3, 3, None, 4, 4), (24, 3, 1, None, 4, 4), (30, 3, 1, None, 1, 4),
    (12, 4, 4, 3000, 3, 4), (12, 4, 4, 3000, 2, 0)])
def test_dense_map_kernels(ctx, M, na, nb, n, nst, path):
    dets = fci_space(M, na, nb) if n is None else _random_space(M, na, nb, n, 7)
    _say(f"[dense map] M={M} {na}a{nb}b nst={nst} path={path} n_det={dets.shape[0]}")
    _against_oracle(ctx, M, na, nb, dets, nst, path, DENSE)


@pytest.mark.parametrize("M,ne,nst", [(17, 8, 1), (17, 8, 4), (19, 9, 2), (19, 9, 4)])
def test_string_driven_kernels_of_many_singles(ctx, M, ne, nst):
    """72 and 90 beta singles of a string (20 and 24 steps of four): the first
    string and its single excitations, of both spins."""
    dets = _singles_space(M, ne, ne, 2.0, 1)
    _say(f"[sigma many singles] M={M} {ne}a{ne}b nst={nst} n_det={dets.shape[0]}")
    _against_oracle(ctx, M, ne, ne, dets, nst, 1, STRINGS)
