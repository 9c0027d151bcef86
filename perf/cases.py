"""What a user of this framework runs, as cases that can be timed and checked.

Families (the "path" of a case):

  sigma_fci     v = H u and s = S^2 u over a full CI space, on vectors that stay on the GPU (the call the
                Davidson driver makes, qpx_sigma_device) or on host arrays (H_S2_u_0_nstates);
  sigma_sel     the same on a selected (CIPSI-like) wavefunction;
  davidson      davidson_diag_hs2 on a full CI space, from a guess to converged states;
  cipsi_diag    what the CIPSI loop does with a grown psi: S^2 completion, set_wavefunction, Davidson;
  select        one selection with EN-PT2 (ZMQ_selection);
  mlp_train     one epoch of the block-proposal network on a sweep's blocks;
  mlp_predict   the network's ranking of the blocks of a sweep.

The Hamiltonians are the package's seeded synthetic ones; wavefunctions, vectors, guesses, weights and training
sets come from the case's seed.  exact() restates each result with plain torch / numpy in 64 bits: string-driven
full CI (Knowles-Handy), pairwise Slater-Condon rules for selected wavefunctions, Lanczos for eigenvalues, direct
enumeration for the selection and a float64 network.
"""
from __future__ import annotations

import functools
import itertools
import math

import numpy as np
import torch

from quantum_package_amd.api import FP32, FP64, PARAM_NAMES, BlockMLP, Context
from quantum_package_amd.hamiltonian import Hamiltonian, fci_space, synthetic_hamiltonian

# ---------------------------------------------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------------------------------------------


def listed():
    return [
        # the smallest full CI space of the configurations: one call is launches and latency
        dict(name="sigma_fci_m8", path="sigma_fci", M=8, na=4, nb=4, n_st=4, prec="f64", host=False),
        # the benchmark's space, 9,018,009 determinants, with a Davidson block of vectors
        dict(name="sigma_fci_m14", path="sigma_fci", M=14, na=6, nb=6, n_st=4, prec="f64", host=False),
        # the same in single precision: the correction vectors of a mixed-precision Davidson
        dict(name="sigma_fci_m14_f32", path="sigma_fci", M=14, na=6, nb=6, n_st=4, prec="f32", host=False),
        # an open-shell space, three vectors, through the host arrays a plugin holds (transfers included)
        dict(name="sigma_fci_m13_host", path="sigma_fci", M=13, na=6, nb=5, n_st=3, prec="f64", host=True),
        # a selected wavefunction of the 96-orbital system with a Davidson block of vectors
        dict(name="sigma_sel_m96", path="sigma_sel", M=96, na=10, nb=10, n_det=262144, n_st=4, prec="f64",
             host=False),
        # a mid-sized, open-shell selected wavefunction, one word per string, single precision, two vectors
        dict(name="sigma_sel_m50_f32", path="sigma_sel", M=50, na=7, nb=6, n_det=40003, n_st=2, prec="f32",
             host=False),
        # three roots of an open-shell full CI, guess to convergence
        dict(name="davidson_fci_m12", path="davidson", M=12, na=6, nb=5, n_st=3),
        # the diagonalisation half of a CIPSI iteration: S^2 completion, new wavefunction, ground state
        dict(name="cipsi_diag_m96", path="cipsi_diag", M=96, na=10, nb=10, n_det=5000, n_st=1),
        # early CIPSI iterations: every determinant of a small psi is a generator, two states
        dict(name="select_m24", path="select", M=24, na=5, nb=5, n_det=600, n_gen=600, n_st=2),
        # a late iteration of the largest system: the leading generators against a long selector list
        dict(name="select_m128", path="select", M=128, na=12, nb=12, n_det=30000, n_gen=48, n_st=1),
        # one epoch over the blocks of a sweep (the batch the proposer trains with)
        dict(name="mlp_train", path="mlp_train", M=96, n=65536, batch=4096),
        # ranking the blocks of the next sweep
        dict(name="mlp_predict", path="mlp_predict", M=96, n=200003),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a family, and sizes over its whole range."""
    path = rng.choice(["sigma_fci", "sigma_fci", "sigma_fci", "sigma_sel", "sigma_sel", "davidson", "cipsi_diag",
                       "select", "select", "mlp_train", "mlp_predict"])
    if path == "sigma_fci":
        target = _log_int(rng, 400, 9_000_000)   # determinants, log-uniform; the space nearest to it
        n_st = rng.randint(1, 4)
        spaces = [(abs(math.log(math.comb(M, na) * math.comb(M, nb) / target)) + 0.3 * rng.random(), M, na, nb)
                  for M in range(6, 15) for na in range(2, M - 1) for nb in range(max(1, na - 2), na + 1)
                  if math.comb(M, na) * math.comb(M, nb) <= 9_018_009 and math.comb(M, na) <= 3003]
        _, M, na, nb = min(spaces)
        return dict(path=path, M=M, na=na, nb=nb, n_st=n_st, prec=rng.choice(["f64", "f64", "f32"]),
                    host=rng.random() < 0.25)
    if path == "sigma_sel":
        M = rng.randint(40, 100)
        na = rng.randint(5, 10)
        return dict(path=path, M=M, na=na, nb=rng.randint(max(4, na - 1), na), n_det=_log_int(rng, 3000, 260000),
                    n_st=rng.randint(1, 4), prec=rng.choice(["f64", "f64", "f32"]), host=rng.random() < 0.25)
    if path == "davidson":
        M = rng.randint(8, 12)
        na = rng.randint(3, M // 2)
        return dict(path=path, M=M, na=na, nb=rng.randint(na - 1, na), n_st=rng.randint(1, 3))
    if path == "cipsi_diag":
        M = rng.randint(40, 96)
        na = rng.randint(5, 10)
        return dict(path=path, M=M, na=na, nb=na, n_det=_log_int(rng, 500, 5000), n_st=1)
    if path == "select":
        M = rng.randint(24, 128)
        na = rng.randint(5, 12)
        n_det = _log_int(rng, 300, 30000)
        # about as much work as the listed ones: fewer generators where a generator has more blocks and cells
        n_gen = max(4, min(n_det, int(6.0e9 / (n_det + 2000) / (na * na * M))))
        return dict(path=path, M=M, na=na, nb=rng.randint(na - 1, na), n_det=n_det, n_gen=n_gen,
                    n_st=rng.randint(1, 2))
    if path == "mlp_train":
        batch = rng.choice([1024, 2048, 4096, 4096, 16384])
        return dict(path=path, M=rng.randint(24, 128), n=batch * rng.randint(1, max(1, 65536 // batch)) + rng.randint(0, 99),
                    batch=batch)
    return dict(path=path, M=rng.randint(24, 128), n=_log_int(rng, 300, 262144))


# ---------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------


def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


@functools.lru_cache(maxsize=4)
def _hamiltonian(M, na, nb):
    """The system's integrals: a given of the run, not of the seed."""
    H = synthetic_hamiltonian(M, max(na, 1), max(nb, 1), seed=1000 + M)
    return Hamiltonian(M=M, n_alpha=na, n_beta=nb, h=H.h, eri=H.eri, seed=H.seed)


@functools.lru_cache(maxsize=None)
def _stream():
    """The one stream a program drives its contexts on."""
    return torch.cuda.Stream()


def _generator(seed, salt):
    return torch.Generator(device=_dev()).manual_seed(1_000_003 * int(seed) + salt)


def _selected_space(M, na, nb, n, seed):
    """n distinct determinants as a CIPSI run grows them: HF, then excitations of degree <= 4 that favour low
    virtual and high occupied orbitals, the lowest ones by orbital energy up to the seed's noise.  Returns the
    determinants (n, 2, n_int) uint64 and their scores, in ascending order of score, HF first."""
    dev, g = _dev(), _generator(seed, 1)
    n_int = (M + 63) // 64
    occ = torch.empty((0, 2, M), dtype=torch.bool, device=dev)
    orb = torch.arange(M, device=dev, dtype=torch.float32)
    tau = max(4.0, M / 6.0)
    # chance of each (alpha degree, beta degree)
    kinds = [(a, b) for a in range(5) for b in range(5) if 1 <= a + b <= 4]
    share = torch.tensor([{1: 0.02, 2: 0.60, 3: 0.23, 4: 0.15}[a + b] / (a + b + 1) for a, b in kinds], device=dev)

    def spin(ne, degree, m):
        # weighted sampling without replacement: the largest of log-weight + Gumbel noise
        noise = -torch.log(-torch.log(torch.rand((m, M), generator=g, device=dev).clamp_(1e-9, 1 - 1e-7)))
        key = noise + torch.where(orb < ne, (orb - ne) / 3.0, (ne - orb) / tau)
        is_occ = (orb < ne).expand(m, M)
        lim = torch.minimum(degree, torch.tensor(min(ne, M - ne), device=dev))[:, None]
        rank_h = torch.where(is_occ, key, -torch.inf).argsort(1, descending=True).argsort(1)
        rank_p = torch.where(is_occ, -torch.inf, key).argsort(1, descending=True).argsort(1)
        return torch.where(is_occ, rank_h >= lim, rank_p < lim)

    while True:
        m = 3 * n + 64
        k = torch.multinomial(share, m, replacement=True, generator=g)
        deg = torch.tensor(kinds, device=dev)[k]
        new = torch.stack([spin(na, deg[:, 0], m), spin(nb, deg[:, 1], m)], dim=1)
        occ = torch.cat([occ, new])
        mix = torch.randint(-(1 << 62), 1 << 62, (2 * M,), generator=torch.Generator().manual_seed(77)).to(dev)
        label = (occ.reshape(occ.shape[0], -1).to(torch.int64) * mix).sum(1)
        order = label.argsort(stable=True)
        first = torch.ones_like(order, dtype=torch.bool)
        first[1:] = label[order][1:] != label[order][:-1]
        occ = occ[order[first].sort().values]
        if occ.shape[0] >= 2 * n:
            break
    hf = torch.stack([orb < na, orb < nb])
    occ = occ[~(occ == hf).flatten(1).all(1)]
    score = (occ * orb).sum((1, 2)) - (hf * orb).sum()
    score = 0.5 * score + 3.0 * torch.rand(score.shape, generator=g, device=dev)
    keep = score.argsort()[: n - 1]
    occ = torch.cat([hf[None], occ[keep]])
    score = torch.cat([score.new_zeros(1), score[keep]])
    return _words(occ, n_int), score.cpu().numpy().astype(np.float64)


def _words(occ, n_int):
    """(n, 2, M) occupations -> (n, 2, n_int) uint64 words on the host."""
    n, _, M = occ.shape
    pad = torch.zeros((n, 2, 64 * n_int), dtype=torch.bool, device=occ.device)
    pad[:, :, :M] = occ
    by = pad.reshape(n, 2, n_int, 8, 8).to(torch.uint8)
    by = (by << torch.arange(8, dtype=torch.uint8, device=occ.device)).sum(-1).to(torch.uint8)
    return np.ascontiguousarray(by.cpu().numpy()).view(np.uint64).reshape(n, 2, n_int)


def _occupations(dets, M):
    """(n, 2, n_int) words -> (n, 2, M) bool on the device."""
    by = np.ascontiguousarray(dets).view(np.uint8).reshape(dets.shape[0], 2, -1)
    by = torch.from_numpy(by.copy()).to(_dev())
    bits = (by[..., None] >> torch.arange(8, dtype=torch.uint8, device=by.device)) & 1
    return bits.flatten(2)[:, :, :M].bool()


def _selected_psi(case, seed):
    """A wavefunction in psi_det_sorted order: determinants, and coefficients that fall with the score."""
    dets, score = _selected_space(case["M"], case["na"], case["nb"], case["n_det"], seed)
    rng = np.random.default_rng([int(seed), 3])
    c = np.exp(-0.25 * score)[:, None] * rng.uniform(0.3, 1.0, (len(score), case["n_st"]))
    c *= rng.choice([-1.0, 1.0], c.shape)
    c[0, :] = 1.5 * np.abs(c).max()
    c /= np.linalg.norm(c, axis=0)
    order = np.argsort(-(c ** 2).sum(1), kind="stable")
    return dets[order], np.asfortranarray(c[order])


def _reference_energy(H):
    """Energy of the HF determinant."""
    def integral(i, j, k, l):
        return float(H.integral(i, j, k, l))
    a, b = range(1, H.n_alpha + 1), range(1, H.n_beta + 1)
    e = sum(H.h[i - 1, i - 1] for i in a) + sum(H.h[i - 1, i - 1] for i in b)
    e += 0.5 * sum(integral(i, j, i, j) - integral(i, j, j, i) for s in (a, b) for i in s for j in s)
    return e + sum(integral(i, j, i, j) for i in a for j in b)


def _training_set(case, seed):
    """Block descriptors (holes, spin class, excitation degree; orbital energies and log|c|) and their labels."""
    rng = np.random.default_rng([int(seed), 5])
    n, ne = case["n"], 12
    desc = np.stack([rng.integers(0, ne, n), rng.integers(0, ne, n), rng.integers(0, 3, n), rng.integers(0, 5, n)],
                    axis=1).astype(np.int32)
    f = np.empty((n, 3), dtype=np.float32)
    f[:, :2] = -2.0 + 0.5 * desc[:, :2] + 0.05 * rng.standard_normal((n, 2))
    f[:, 2] = -np.abs(rng.standard_normal(n)) * 3.0
    y = 2.0 * f[:, 2] + 0.2 * f[:, 0] - 0.5 * desc[:, 3] + 0.3 * rng.standard_normal(n)
    return desc, f, ((y - y.mean()) / y.std()).astype(np.float32)


def _weights(case, seed):
    rng = np.random.default_rng([int(seed), 6])
    shapes = {"W1": (80, 256), "W2": (256, 256), "W3": (256, 256), "b1": (256,), "b2": (256,), "b3": (256,),
              "w4": (256,), "emb": (case["M"], 32), "b4": (1,)}
    scale = {"W1": 0.16, "W2": 0.088, "W3": 0.088, "w4": 0.0625, "emb": 0.3, "b1": 0.05, "b2": 0.05, "b3": 0.05,
             "b4": 0.05}
    return {k: (scale[k] * rng.standard_normal(s)).astype(np.float32) for k, s in shapes.items()}


def _guess(case, seed, dets):
    """Guess vectors: HF (with a little noise where no spin filter is asked for), then seeded noise."""
    g = np.random.default_rng([int(seed), 4]).standard_normal((dets.shape[0], case["n_st"]))
    g[:, 0] *= 0.05 / math.sqrt(dets.shape[0]) if case["path"] == "davidson" else 0.0
    hf = np.zeros((2, dets.shape[2]), dtype=np.uint64)
    for s, ne in enumerate((case["na"], case["nb"])):
        for p in range(ne):
            hf[s, p // 64] |= np.uint64(1) << np.uint64(p % 64)
    g[np.nonzero((dets == hf).all((1, 2)))[0][0], 0] = 1.0
    return g


def _vectors(case, seed, n):
    """(n, n_st) vectors in psi order on the device: unit-norm noise, as orthonormal correction vectors are."""
    u = torch.randn((n, case["n_st"]), generator=_generator(seed, 2), dtype=torch.float64, device=_dev())
    u = u / u.norm(dim=0)
    return u.float().double() if case["prec"] == "f32" else u


def prepare(case, seed):
    path, M, ctx = case["path"], case["M"], None
    st = dict(case=case)
    if path.startswith("mlp"):
        m = st["mlp"] = BlockMLP(n_orb=M, seed=1)
        for k, w in _weights(case, seed).items():
            m.set(k, w)
        st["desc"], st["fdesc"], st["y"] = _training_set(case, seed)
        st["seed"] = int(seed) & 0xFFFF
        return st
    ctx = st["ctx"] = Context(0)
    H = _hamiltonian(M, case["na"], case["nb"])
    ctx.set_hamiltonian(H)
    if path in ("sigma_fci", "davidson"):
        dets = fci_space(M, case["na"], case["nb"])
    elif path == "select":
        dets, st["coef"] = _selected_psi(case, seed)
        st["E0"] = _reference_energy(H) - 1.0 + 0.3 * np.arange(case["n_st"])
    else:
        dets, _ = _selected_space(M, case["na"], case["nb"], case["n_det"], seed)
    if path == "cipsi_diag":
        st["dets"] = dets
        st["guess"] = _guess(case, seed, dets)
        # the loop's psi arrays, with room for the determinants the S^2 completion adds
        st["psi"] = np.zeros((16 * dets.shape[0],) + dets.shape[1:], dtype=np.uint64)
        st["coef"] = np.zeros((16 * dets.shape[0], case["n_st"]))
        return st
    ctx.set_wavefunction(dets)
    if path == "davidson":
        st["guess"] = _guess(case, seed, dets)
    if path.startswith("sigma"):
        u = _vectors(case, seed, dets.shape[0])
        if case["host"]:
            st["u"] = np.asfortranarray(u.cpu().numpy())
        else:
            perm = torch.from_numpy(ctx.bilinear_order()).to(u.device)
            dtype = torch.float64 if case["prec"] == "f64" else torch.float32
            st["u"] = u[perm].to(dtype).contiguous()
            st["v"], st["s"] = torch.empty_like(st["u"]), torch.empty_like(st["u"])
            st["stream"] = _stream()
            torch.cuda.synchronize()
    return st


def run(st):
    case = st["case"]
    path = case["path"]
    if path.startswith("sigma"):
        ctx, prec = st["ctx"], FP64 if case["prec"] == "f64" else FP32
        if case["host"]:
            return ctx.H_S2_u_0_nstates(st["u"], prec)
        ctx._check(ctx.L.qpx_sigma_device(ctx.ptr, prec, case["n_st"], st["u"].data_ptr(), st["v"].data_ptr(),
                                          st["s"].data_ptr(), st["stream"].cuda_stream))
        return st["v"], st["s"]
    if path == "davidson":
        e, s2, u, _ = st["ctx"].davidson_diag_hs2(st["guess"], N_st=case["n_st"], N_st_diag=case["n_st"] + 1,
                                                  threshold=1e-10, s2_eig=False)
        return e[: case["n_st"]], np.sqrt(1.0 + 4.0 * s2[: case["n_st"]]), u[:, : case["n_st"]]
    if path == "cipsi_diag":
        ctx = st["ctx"]
        extra = ctx.s2_complete(st["dets"], case["na"])
        dets = np.concatenate([st["dets"], extra])
        guess = np.concatenate([st["guess"], np.zeros((extra.shape[0], case["n_st"]))])
        ctx.set_wavefunction(dets)
        e, _, u, _ = ctx.davidson_diag_hs2(guess, N_st=case["n_st"], N_st_diag=4, threshold=1e-10, s2_eig=True)
        st["psi"][: dets.shape[0]] = dets
        st["coef"][: dets.shape[0]] = u[:, : case["n_st"]]
        return e[: case["n_st"]], st["coef"], st["psi"].view(np.int64)
    if path == "select":
        n_det = st["coef"].shape[0]
        pt2, dets, vals = st["ctx"].ZMQ_selection(st["coef"], case["n_gen"], n_det, st["E0"], n_det)
        return pt2, vals, dets.view(np.int64)
    if path == "mlp_train":
        m = st["mlp"]
        loss = m.train_epochs(st["desc"], st["fdesc"], st["y"], 1e-3, 1, case["batch"], st["seed"])
        return [loss] + [m.get(k) for k in PARAM_NAMES]
    return st["mlp"].predict(st["desc"], st["fdesc"])


# ---------------------------------------------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------------------------------------------


def _fci_pairs(M, na, nb):
    """Connected pairs of one full-CI determinant."""
    def singles(n):
        return n * (M - n)

    def doubles(n):
        return math.comb(n, 2) * math.comb(M - n, 2)
    return singles(na) * singles(nb) + singles(na) + singles(nb) + doubles(na) + doubles(nb)


@functools.lru_cache(maxsize=None)
def _selected_pairs(M, na, nb, n_det):
    """Connected pairs of one determinant of a selected wavefunction, from 256 of its rows."""
    dets, _ = _selected_space(M, na, nb, n_det, 0)
    occ = _occupations(dets, M).flatten(1).float()
    rows = torch.arange(0, n_det, max(1, n_det // 256), device=occ.device)
    return float(((occ[rows] @ occ.T) >= na + nb - 2.5).sum() / len(rows)) - 1.0


def work(case):
    path, M = case["path"], case["M"]
    if path.startswith("mlp"):
        flops = 2.0 * (80 * 256 + 2 * 256 * 256 + 256)
        weights = 4.0 * (80 * 256 + 2 * 256 * 256 + 4 * 256 + 32 * M)
        if path == "mlp_train":
            n = case["n"] // case["batch"] * case["batch"]
            return {"bytes": 32.0 * n + 6 * weights, "flops": 3 * flops * n}
        return {"bytes": 32.0 * case["n"] + weights, "flops": flops * case["n"]}
    na, nb, n_st = case["na"], case["nb"], case["n_st"]
    if path == "select":
        # every determinant reached from a generator: its coupling and its perturbative term
        reach = na * nb * (M - na) * (M - nb) + math.comb(na, 2) * math.comb(M - na, 2) + math.comb(nb, 2) * math.comb(M - nb, 2)
        return {"bytes": case["n_det"] * (32.0 * ((M + 63) // 64) + 16.0 * n_st) + M ** 4, "flops": 16.0 * n_st * reach * case["n_gen"]}
    w = 4 if case.get("prec") == "f32" else 8
    if path in ("sigma_fci", "davidson"):
        n, pairs = math.comb(M, na) * math.comb(M, nb), _fci_pairs(M, na, nb)
    else:
        n, pairs = case["n_det"], _selected_pairs(M, na, nb, case["n_det"])
    calls = 1 if path.startswith("sigma") else 15
    block = n_st if path.startswith("sigma") else max(4 if path == "cipsi_diag" else 1, n_st + 1)
    # the vectors, the determinants and the distinct integrals
    return {"bytes": calls * (3.0 * n * block * w + 16.0 * n * ((M + 63) // 64) + w * M ** 4 / 8),
            "flops": calls * 2.0 * n * pairs * block}


# ---------------------------------------------------------------------------------------------------------------
# exact results, in 64 bits
# ---------------------------------------------------------------------------------------------------------------


class _FullCI:
    """sigma over a full CI space by spin strings: H = sum h'_pq E_pq + 1/2 sum (pq|rs) E_pq E_rs."""

    def __init__(self, H):
        M, self.M = H.M, H.M
        eri = torch.from_numpy(H.eri_dense_chemist()).to(_dev())
        self.eri = eri
        self.h1 = torch.from_numpy(np.asarray(H.h)).to(_dev()) - 0.5 * torch.einsum("prrq->pq", eri)
        self.ne = (H.n_alpha, H.n_beta)
        self.tab = [self._table(M, n) for n in self.ne]

    @staticmethod
    def _table(M, n):
        """E_pq |J> for every string: index and sign (0: none) of the result, as (M, M, n_strings)."""
        s = np.sort(np.array([sum(1 << p for p in c) for c in itertools.combinations(range(M), n)], dtype=np.int64))
        idx, sgn = np.zeros((M, M, len(s)), dtype=np.int64), np.zeros((M, M, len(s)))
        bits = (s[:, None] >> np.arange(M)) & 1
        below = np.cumsum(bits, 1) - bits
        for p in range(M):
            for q in range(M):
                ok = (bits[:, q] == 1) & ((bits[:, p] == 0) | (p == q))
                t = (s ^ (1 << q)) | (1 << p)
                par = below[:, q] + below[:, p] - (q < p)
                idx[p, q] = np.where(ok, np.searchsorted(s, np.where(ok, t, s)), 0)
                sgn[p, q] = np.where(ok, np.where((par & 1) & (p != q), -1.0, 1.0), 0.0)
        return torch.from_numpy(idx).to(_dev()), torch.from_numpy(sgn).to(_dev())

    def excite(self, p, q, x):
        """E_pq x (both spins); x is (n_alpha strings, n_beta strings).  <I|E_pq|J>: row I takes J = E_qp I."""
        (ia, sa), (ib, sb) = self.tab
        return x[ia[q, p]] * sa[q, p][:, None] + x[:, ib[q, p]] * sb[q, p]

    def sigma(self, x):
        M = self.M
        pairs = [(p, q) for p in range(M) for q in range(p + 1)]
        D = torch.empty((len(pairs), x.numel()), dtype=x.dtype, device=x.device)
        for k, (p, q) in enumerate(pairs):
            D[k] = (self.excite(p, q, x) + (self.excite(q, p, x) if p != q else 0.0)).flatten()
        V = torch.stack([torch.stack([self.eri[p, q, r, s] for r, s in pairs]) for p, q in pairs])
        step = max(1, D.shape[1] // 8)
        for c in range(0, D.shape[1], step):
            D[:, c:c + step] = V @ D[:, c:c + step]
        v = torch.zeros_like(x)
        for k, (p, q) in enumerate(pairs):
            t = 0.5 * D[k].view_as(x)
            v += self.excite(p, q, t + self.h1[p, q] * x)
            if p != q:
                v += self.excite(q, p, t + self.h1[q, p] * x)
        return v

    def s_plus_s_minus(self, x):
        """(S^2 - Sz (Sz - 1)) x = S_+ S_- x = n_alpha x - sum_pq E^alpha_qp E^beta_pq x."""
        (ia, sa), (ib, sb) = self.tab
        s = self.ne[0] * x
        for p in range(self.M):
            for q in range(self.M):
                s = s - (x[ia[p, q]] * sa[p, q][:, None])[:, ib[q, p]] * sb[q, p]
        return s


class _Pairs:
    """Matrix elements between determinants of two lists by the Slater-Condon rules, pair by pair."""

    def __init__(self, H):
        M = self.M = H.M
        p = np.arange(1, M + 1)
        tri = np.minimum(p[:, None], p) + np.maximum(p[:, None], p) * (np.maximum(p[:, None], p) - 1) // 2 - 1
        self.tri = torch.from_numpy(tri).to(_dev())
        self.eri = torch.from_numpy(H.eri).to(_dev())
        self.h = torch.from_numpy(np.asarray(H.h)).to(_dev())
        d = torch.arange(M, device=_dev())
        self.hpkk = self.get(d[:, None, None], d[None, :, None], d[None, None, :], d[None, None, :])
        self.hkkp = self.get(d[:, None, None], d[None, None, :], d[None, None, :], d[None, :, None])
        self.J = self.get(d[:, None], d[:, None], d[None, :], d[None, :])
        self.K = self.get(d[:, None], d[None, :], d[:, None], d[None, :])
        self.sz = 0.5 * (H.n_alpha - H.n_beta)
        self.ne = H.n_alpha + H.n_beta

    def get(self, p, q, r, s):
        """(pq|rs)"""
        a, b = self.tri[p, q], self.tri[r, s]
        lo, hi = torch.minimum(a, b), torch.maximum(a, b)
        return self.eri[hi * (hi + 1) // 2 + lo]

    def diagonal(self, occ):
        a, b = occ[:, 0].double(), occ[:, 1].double()
        JK = 0.5 * (self.J - self.K)
        return (a + b) @ self.h.diagonal() + ((a @ JK) * a).sum(1) + ((b @ JK) * b).sum(1) + ((a @ self.J) * b).sum(1)

    def s2_diagonal(self, occ):
        return occ[:, 0].sum(1).double() - (occ[:, 0] & occ[:, 1]).sum(1).double()

    def connected(self, occ_i, occ_j):
        """(i, j) with at most two excitations between them, themselves excluded."""
        ov = occ_i.flatten(1).half() @ occ_j.flatten(1).half().T
        return torch.nonzero((ov > self.ne - 2.5) & (ov < self.ne - 0.5), as_tuple=True)

    def elements(self, occ_i, occ_j, i, j):
        """H_ij and (S_+ S_-)_ij of connected pairs."""
        M = self.M
        orb = torch.arange(1, M + 1, dtype=torch.uint8, device=i.device)
        ends = []   # per spin: number of excitations, first and last hole and particle, parity of their positions
        for s in (0, 1):
            x, y = occ_i[:, s][i], occ_j[:, s][j]
            hole, part = (x & ~y), (y & ~x)
            n = hole.sum(1)
            e = [n]
            for z in (hole, part):
                last = (z * orb).amax(1).long() - 1
                first = M - (z * orb.flip(0)).amax(1).long()
                e += [first.clamp_(0, M - 1), last.clamp_(0, M - 1)]
            bi = (occ_i[:, s].long().cumsum(1) - occ_i[:, s].long())
            bj = (occ_j[:, s].long().cumsum(1) - occ_j[:, s].long())
            par = torch.where(n > 0, bi[i, e[1]] + bj[j, e[3]], 0) + torch.where(n > 1, bi[i, e[2]] + bj[j, e[4]], 0)
            ends.append(e + [par])
        a, b = ends
        sign = 1.0 - 2.0 * ((a[5] + b[5]) & 1).double()
        H = torch.zeros(len(i), dtype=torch.float64, device=i.device)
        S = torch.zeros_like(H)
        k = torch.nonzero((a[0] == 1) & (b[0] == 1)).flatten()
        H[k] = self.get(a[1][k], a[3][k], b[1][k], b[3][k])
        S[k] = -((a[1][k] == b[3][k]) & (a[3][k] == b[1][k])).double()
        for s, (t, o) in enumerate(((a, b), (b, a))):
            k = torch.nonzero((t[0] == 2) & (o[0] == 0)).flatten()
            H[k] = self.get(t[1][k], t[3][k], t[2][k], t[4][k]) - self.get(t[1][k], t[4][k], t[2][k], t[3][k])
            for k in torch.nonzero((t[0] == 1) & (o[0] == 0)).flatten().split(1 << 18):
                h, p = t[1][k], t[3][k]
                tot = occ_i[i[k]].sum(1).double()
                same = occ_i[:, s][i[k]].double()
                H[k] = self.h[h, p] + (self.hpkk[h, p] * tot).sum(1) - (self.hkkp[h, p] * same).sum(1)
        return sign * H, sign * S

    def chunks(self, occ_i, occ_j, rows, most=1 << 21):
        """(i, j, H_ij, S_ij) of all connected pairs, some rows at a time."""
        for r0 in range(0, occ_i.shape[0], rows):
            part = occ_i[r0:r0 + rows]
            i, j = self.connected(part, occ_j)
            for c in range(0, len(i), most):
                # positions are cumulated over the determinants at hand only
                ic, jc = i[c:c + most], j[c:c + most]
                uj, back = torch.unique(jc, return_inverse=True)
                H, S = self.elements(part, occ_j[uj], ic, back)
                yield ic + r0, jc, H, S

    def sigma(self, occ, u):
        v, s = self.diagonal(occ)[:, None] * u, self.s2_diagonal(occ)[:, None] * u
        for i, j, H, S in self.chunks(occ, occ, max(64, (1 << 27) // occ.shape[0])):
            v.index_add_(0, i, H[:, None] * u[j])
            k = torch.nonzero(S).flatten()
            s.index_add_(0, i[k], S[k, None] * u[j[k]])
        return v, s


def _lowest(apply, n, k, x, steps=160):
    """The k lowest eigenvalues seen from x: Lanczos with full reorthogonalisation."""
    Q = torch.zeros((steps + 1, n), dtype=torch.float64, device=x.device)
    Q[0] = x / x.norm()
    T = np.zeros((steps, steps))
    for m in range(min(steps, n)):
        w = apply(Q[m])
        T[m, m] = float(w @ Q[m])
        for _ in range(2):
            w = w - Q[: m + 1].T @ (Q[: m + 1] @ w)
        b = float(w.norm())
        e, y = np.linalg.eigh(T[: m + 1, : m + 1])
        if b < 1e-10 or m + 1 == steps or (m > 20 and m % 5 == 0 and np.all(np.abs(b * y[-1, :k]) < 1e-9)):
            return e[:k]
        T[m, m + 1] = T[m + 1, m] = b
        Q[m + 1] = w / b
    return e[:k]


def _bilinear(dets):
    """Positions of the determinants in order of (beta string, alpha string), strings by the exclusive-or of their
    words, then the words."""
    keys = []
    for s in (0, 1):   # alpha varies fastest
        keys += [dets[:, s, w] for w in range(dets.shape[2] - 1, -1, -1)] + [np.bitwise_xor.reduce(dets[:, s], axis=1)]
    return np.lexsort(keys)


def _spin_completed(dets, M):
    """Occupations of the space with every spin coupling of the given determinants' patterns."""
    occ = _occupations(dets, M).cpu().numpy()
    two, one = occ.all(1), occ.any(1) & ~occ.all(1)
    pattern = np.unique(np.packbits(np.concatenate([two, one], axis=1), axis=1), axis=0)
    pattern = np.unpackbits(pattern, axis=1)[:, : 2 * M].astype(bool).reshape(-1, 2, M)
    n_up = int(occ[0, 0].sum()) - pattern[:, 0].sum(1)
    n_open = pattern[:, 1].sum(1)
    out = []
    for no, nu in set(zip(n_open.tolist(), n_up.tolist())):
        pat = pattern[(n_open == no) & (n_up == nu)]
        at = np.nonzero(pat[:, 1])[1].reshape(len(pat), no)
        for up in itertools.combinations(range(no), nu):
            d = np.repeat(pat[:, :1], 2, axis=1)
            down = [x for x in range(no) if x not in up]
            rows = np.arange(len(pat))[:, None]
            d[rows, 0, at[:, list(up)]] = True
            d[rows, 1, at[:, down]] = True
            out.append(d)
    return torch.from_numpy(np.concatenate(out)).to(_dev())


def _exact_selection(case, seed):
    """EN-PT2 by enumeration of the space reached from the generators, and its best determinants' terms."""
    H = _hamiltonian(case["M"], case["na"], case["nb"])
    M, n_int = case["M"], (case["M"] + 63) // 64
    dets, coef = _selected_psi(case, seed)
    occ = _occupations(dets, M)
    P = _Pairs(H)
    E0 = torch.tensor(_reference_energy(H) - 1.0 + 0.3 * np.arange(case["n_st"]), device=occ.device)
    mix = torch.randint(-(1 << 62), 1 << 62, (2 * M,), generator=torch.Generator().manual_seed(78)).to(occ.device)
    label = (occ.flatten(1).long() * mix).sum(1)
    reached, seen = [], []
    for d, l in zip(occ, label):
        h = torch.nonzero(d.flatten()).flatten()
        p = torch.nonzero(~d.flatten()).flatten()
        sz_h, sz_p = (h >= M).long(), (p >= M).long()
        h1, p1 = torch.meshgrid(torch.arange(len(h), device=h.device), torch.arange(len(p), device=h.device), indexing="ij")
        k = sz_h[h1] == sz_p[p1]
        single = torch.stack([h[h1[k]], h[h1[k]], p[p1[k]], p[p1[k]]], 1)
        hh, pp = torch.combinations(h, 2), torch.combinations(p, 2)
        nh, np_ = (hh >= M).sum(1), (pp >= M).sum(1)
        many = [torch.cat([hh[nh == x].repeat_interleave(int((np_ == x).sum()), 0), pp[np_ == x].repeat(int((nh == x).sum()), 1)], 1)
                for x in (0, 1, 2)]
        ex = torch.cat([single] + many)
        two = (ex[:, 0] != ex[:, 1])
        new = l - mix[ex[:, 0]] + mix[ex[:, 2]] + torch.where(two, mix[ex[:, 3]] - mix[ex[:, 1]], 0)
        reached.append(torch.stack([torch.full_like(new, len(seen)), *ex.T], 1))
        seen.append(new)
    lab, ex = torch.cat(seen), torch.cat(reached)
    order = lab.argsort(stable=True)
    first = torch.ones_like(order, dtype=torch.bool)
    first[1:] = lab[order][1:] != lab[order][:-1]
    pick = order[first]
    pick = pick[~torch.isin(lab[pick], label)]
    pt2 = torch.zeros(case["n_st"], dtype=torch.float64, device=occ.device)
    c, terms = torch.from_numpy(np.ascontiguousarray(coef)).to(occ.device), []
    for part in pick.split(1 << 18):
        e = ex[part]
        o = occ[e[:, 0]].flatten(1).clone()
        r = torch.arange(len(e), device=o.device)
        o[r, e[:, 1]] = o[r, e[:, 2]] = False
        o[r, e[:, 3]] = o[r, e[:, 4]] = True
        o = o.view(-1, 2, M)
        V = torch.zeros((len(e), case["n_st"]), dtype=torch.float64, device=o.device)
        for i, j, Hij, _ in P.chunks(o, occ, 1 << 18):
            V.index_add_(0, i, Hij[:, None] * c[j])
        dE = E0 - P.diagonal(o)[:, None]
        val = 2.0 * V
        tmp = torch.sqrt(dE * dE + val * val)
        e2 = 0.5 * (torch.where(dE < 0, -tmp, tmp) - dE)
        pt2 += e2.sum(0)
        terms.append(e2.amin(1))
    best = torch.cat(terms)
    return pt2, best.sort().values[: case["n_det"]]


def _network(W, desc, fdesc):
    """Features and layers of the block-proposal network in float64."""
    d = torch.from_numpy(desc).long().to(_dev())
    f = torch.from_numpy(fdesc).double().to(_dev())
    one = torch.nn.functional.one_hot
    x = torch.cat([W["emb"][d[:, 0]], W["emb"][d[:, 1]], f, one(d[:, 2], 3).double(), one(d[:, 3], 5).double(),
                   f.new_zeros((len(f), 5))], 1)
    for k in "123":
        x = torch.relu(x @ W["W" + k] + W["b" + k])
    return x @ W["w4"] + W["b4"]


def _exact_training(case, seed):
    """Adam on the batches of one epoch: a SplitMix64 Fisher-Yates permutation, leftover rows dropped."""
    W = {k: torch.from_numpy(w).double().to(_dev()).requires_grad_() for k, w in _weights(case, seed).items()}
    desc, fdesc, y = _training_set(case, seed)
    n, batch, mask = case["n"], case["batch"], (1 << 64) - 1
    perm, s = list(range(n)), int(seed) & 0xFFFF
    for i in range(n - 1, 0, -1):
        s = (s + 0x9E3779B97F4A7C15) & mask
        z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        j = (z ^ (z >> 31)) % (i + 1)
        perm[i], perm[j] = perm[j], perm[i]
    opt = torch.optim.Adam(W.values(), lr=1e-3, betas=(0.9, 0.999), eps=1e-8)
    losses = []
    for k in range(n // batch):
        at = np.array(perm[k * batch:(k + 1) * batch])
        loss = ((_network(W, desc[at], fdesc[at]) - torch.from_numpy(y[at]).double().to(_dev())) ** 2).mean()
        opt.zero_grad()
        loss.backward()
        opt.step()
        losses.append(float(loss.detach()))
    return [np.array([np.mean(losses)])] + [W[k].detach() for k in PARAM_NAMES]


def exact(case, seed):
    path, M = case["path"], case["M"]
    if path == "mlp_predict":
        desc, fdesc, _ = _training_set(case, seed)
        W = {k: torch.from_numpy(w).double().to(_dev()) for k, w in _weights(case, seed).items()}
        return torch.cat([_network(W, desc[i:i + 65536], fdesc[i:i + 65536]) for i in range(0, case["n"], 65536)])
    if path == "mlp_train":
        return _exact_training(case, seed)
    na, nb = case["na"], case["nb"]
    H = _hamiltonian(M, na, nb)
    if path == "sigma_fci":
        F = _FullCI(H)
        ns, nt = math.comb(M, na), math.comb(M, nb)
        u = _vectors(case, seed, ns * nt)
        cols = [u[:, k].reshape(ns, nt).contiguous() for k in range(case["n_st"])]
        v, s = [F.sigma(x) for x in cols], [F.s_plus_s_minus(x) for x in cols]
        if case["host"]:   # psi order: alpha-major
            return torch.stack([x.flatten() for x in v], 1), torch.stack([x.flatten() for x in s], 1)
        return torch.stack([x.T.flatten() for x in v], 1), torch.stack([x.T.flatten() for x in s], 1)
    if path == "sigma_sel":
        dets, _ = _selected_space(M, na, nb, case["n_det"], seed)
        v, s = _Pairs(H).sigma(_occupations(dets, M), _vectors(case, seed, dets.shape[0]))
        if not case["host"]:
            order = torch.from_numpy(_bilinear(dets)).to(v.device)
            v, s = v[order], s[order]
        return v, s
    if path == "davidson":
        F = _FullCI(H)
        ns, nt = math.comb(M, na), math.comb(M, nb)
        x = torch.randn(ns * nt, generator=_generator(0, 9), dtype=torch.float64, device=_dev())
        e = _lowest(lambda q: F.sigma(q.view(ns, nt)).flatten(), ns * nt, case["n_st"], x)
        return e, None, None
    if path == "cipsi_diag":
        occ = _spin_completed(_selected_space(M, na, nb, case["n_det"], seed)[0], M)
        P, n = _Pairs(H), occ.shape[0]
        if n > 120_000:
            return None
        parts = list(P.chunks(occ, occ, max(64, (1 << 27) // n)))
        i, j, v = (torch.cat([p[k] for p in parts]) for k in (0, 1, 2))
        A = torch.sparse_coo_tensor(torch.stack([i, j]), v, (n, n)).to_sparse_csr()
        d = P.diagonal(occ)
        hf = torch.arange(M, device=occ.device) < na
        x = (occ == hf).all(2).all(1).double()   # the closed-shell determinant: Lanczos stays among singlets
        return _lowest(lambda q: d * q + A @ q, n, 1, x), None, None
    if path == "select" and case["n_gen"] == case["n_det"] <= 700 and M <= 32:
        pt2, vals = _exact_selection(case, seed)
        return pt2, vals, None
    return None
