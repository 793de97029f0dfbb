"""Timed cases of operator application: mul! and what surrounds it in a
simulation, through the package's public functions.

Families (the ``kind`` of a case) and their sizes:

  chain     H psi, <psi| H or a first-order time step of one spin-1/2 chain
            (LazySum of two-site and one-site Pauli terms), 6..24 sites
  batch     one time step of many chains of uneven lengths in one launch
  fock      the commutator -i [H, rho] of two coupled Fock modes and a spin, as
            a SparseOperator or as a LazySum of LazyTensors, N = 300..6400
  lt        a LazyTensor of dense factors on a density matrix, from the left
            or from both sides (rho -> U rho U^dagger), N = 200..8192
  dense     the commutator of a DenseOperator with a density matrix
  denseket  a DenseOperator on a Ket and on a Bra
  lazyket   a LazySum of sparse LazyTensors (two Fock modes and a spin) on a Ket
  lindblad  a sparse Liouvillian on vec(rho) of a driven, damped cavity with a
            spin
  measure   expect, variance and norm of a chain's state (results on the host)

States: normalised complex-Gaussian Kets, Ginibre density matrices of trace 1.
Coefficients: uniform in [-1, 1] (chains) or [0, 1] (couplings); dense factors:
Hermitian complex Gaussian.
"""
from __future__ import annotations

import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "quantumopticsbase.jl_amd"))

import qobhip as Q  # noqa: E402
from qobhip import workloads as W  # noqa: E402

DT = 0.01  # time step of the first-order steps


# ------------------------------------------------------------------- cases
def listed():
    return [
        # a 10-site chain stepped by an explicit integrator: the smallest call,
        # where the launches and the host count
        dict(name="chain10_step", kind="chain", op="step", L=10, dtype="c64"),
        # one large closed-system state, H psi inside a Krylov or ODE solver
        dict(name="chain22_ket", kind="chain", op="ket", L=22, dtype="c64"),
        # an ensemble of disorder realisations of uneven length, stepped together
        dict(name="batch256_step", kind="batch", n=256, lmin=8, lmax=20, dtype="c64"),
        # von Neumann equation, the largest truncation, H held as a sparse matrix
        dict(name="fock6400_commutator", kind="fock", form="sparse", na=39, nb=39, spin2=3, dtype="c64"),
        # the same equation in single precision on an odd dimension (1173), H kept lazy
        dict(name="fock1173_lazy_c32", kind="fock", form="lazy", na=22, nb=16, spin2=2, dtype="c32"),
        # dense local operators on the largest density matrix
        dict(name="lt8192_left", kind="lt", op="left", dims="16,32,16", dtype="c64"),
        # a product gate on three many-level systems: U rho U^dagger, ragged widths (N = 2160)
        dict(name="lt2160_sandwich", kind="lt", op="both", dims="12,20,9", dtype="c64"),
        # von Neumann equation with a dense Hamiltonian of odd size
        dict(name="dense3001_commutator", kind="dense", n=3001, dtype="c64"),
        # dense Hamiltonian on a Ket and a Bra, single precision
        dict(name="denseket6143_c32", kind="denseket", n=6143, dtype="c32"),
        # closed dynamics of two field modes and a spin, never forming H
        dict(name="lazyket1012084", kind="lazyket", na=600, nb=420, spin2=3, dtype="c64"),
        # master equation as a superoperator (vec(rho) of 90000 elements)
        dict(name="lindblad300", kind="lindblad", n=149, spin2=1, dtype="c64"),
        # observables along a trajectory
        dict(name="measure18", kind="measure", L=18, dtype="c64"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("chain", "batch", "fock", "lt", "dense", "denseket", "lazyket", "lindblad", "measure"))
    c = dict(kind=kind, dtype=rng.choice(("c64", "c32")))
    if kind == "chain":
        c.update(op=rng.choice(("ket", "bra", "step")), L=rng.randint(6, 23 if c["dtype"] == "c64" else 24))
    elif kind == "batch":
        c.update(n=_log(rng, 16, 256), lmin=rng.randint(6, 10), lmax=rng.randint(14, 20))
    elif kind == "fock":
        form = rng.choice(("sparse", "lazy"))
        na = rng.randint(11, 39)
        c.update(form=form, na=na, nb=na if form == "sparse" else rng.randint(11, 39), spin2=rng.randint(1, 3))
    elif kind == "lt":
        while True:
            dims = [_log(rng, 4, 40) for _ in range(rng.randint(2, 4))]
            if 200 <= math.prod(dims) <= 8192:
                break
        c.update(op=rng.choice(("left", "both")), dims=",".join(map(str, dims)))
    elif kind == "dense":
        c.update(n=_log(rng, 200, 3001))
    elif kind == "denseket":
        c.update(n=_log(rng, 300, 8192))
    elif kind == "lazyket":
        c.update(na=_log(rng, 19, 600), nb=_log(rng, 19, 420), spin2=rng.randint(1, 3))
    elif kind == "lindblad":
        c.update(n=_log(rng, 9, 99), spin2=rng.randint(1, 2))
    else:
        c.update(L=rng.randint(8, 20))
    return c


# ------------------------------------------------------------------ inputs
def _np_dtype(case):
    return np.complex128 if case["dtype"] == "c64" else np.complex64


def _t_dtype(case):
    return torch.complex128 if case["dtype"] == "c64" else torch.complex64


def _esize(case):
    return 16 if case["dtype"] == "c64" else 8


class _Memory:
    """Device memory of a DeviceArray as the array interface describes it."""

    def __init__(self, d):
        self.d = d
        self.__cuda_array_interface__ = dict(shape=(d.n,), typestr="<c16" if d.dtype == np.complex128 else "<c8",
                                             data=(d.ptr.value, False), version=2)


def _view(d):
    """A flat torch tensor over a DeviceArray (no copy)."""
    return torch.as_tensor(_Memory(d), device="cuda")


def _upload(x, dtype):
    """A DeviceArray holding the flat device tensor x."""
    d = Q.DeviceArray(x.numel(), dtype)
    _view(d).copy_(x)
    return d


def _gauss(seed, *shape):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, dtype=torch.complex128, device="cuda", generator=g)


def _ket(case, seed, n):
    """A normalised Ket's amplitudes, rounded to the case's type."""
    v = _gauss(seed, n)
    return (v / torch.linalg.vector_norm(v)).to(_t_dtype(case))


def _kets(case, seed, Ls):
    """Normalised Kets of 2^L amplitudes one after another in one tensor."""
    parts = torch.split(_gauss(seed, sum(1 << L for L in Ls)), [1 << L for L in Ls])
    return torch.cat([v / torch.linalg.vector_norm(v) for v in parts]).to(_t_dtype(case))


class _Part:
    """A state inside a larger DeviceArray, as Batch.bind reads it."""

    def __init__(self, d, first, n):
        self.d, self.n, self.dtype = d, n, d.dtype
        self.ptr = C.c_void_p(d.ptr.value + first * d.dtype.itemsize)


def _parts(d, Ls):
    first = np.cumsum([0] + [1 << L for L in Ls])
    return [_Part(d, int(f), 1 << L) for f, L in zip(first, Ls)]


def _rho(case, seed, n):
    """A Ginibre density matrix of trace 1, rounded to the case's type."""
    G = _gauss(seed, n, n)
    r = G @ G.conj().T.contiguous()
    return (r / torch.diagonal(r).sum().real).to(_t_dtype(case))


def _colmajor(M):
    return M.T.contiguous().reshape(-1)


def _hermitian(rng, d):
    X = rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d))
    return (X + X.conj().T) / 2


def _generic(dims):
    return Q.tensor(*[Q.GenericBasis(d) for d in dims])


def _dims(case):
    return [int(d) for d in case["dims"].split(",")]


def _lengths(case):
    return [int(L) for L in W.tfim_batch_lengths(case["n"], case["lmin"], case["lmax"])]


def _chain_seed(seed):
    return seed % (1 << 30) + 1


def _modes(case):
    """Basis and dense site matrices of two Fock modes and a spin."""
    B = Q.tensor(Q.FockBasis(case["na"]), Q.FockBasis(case["nb"]), Q.SpinBasis(case["spin2"] / 2))
    return B, _destroy(case["na"] + 1), _destroy(case["nb"] + 1), _raise(case["spin2"])


def _destroy(n):
    return np.diag(np.sqrt(np.arange(1, n)), 1).astype(complex)


def _raise(spin2):
    s = spin2 / 2
    m = [s - k for k in range(spin2 + 1)]
    return np.diag([math.sqrt(s * (s + 1) - x * (x + 1)) for x in m[1:]], 1).astype(complex)


def _coupling(seed):
    return float(W.rng(_chain_seed(seed)).uniform(0, 1))


def _lazy_modes(case, seed):
    """a^dag a + b^dag b + g (a b^dag s+ + h.c.) as a LazySum."""
    B, a, b, sp = _modes(case)
    fa, fb, s = B.bases
    A, Ad, N = (Q.SparseOperator(fa, fa, m) for m in (a, a.conj().T, a.conj().T @ a))
    Bb, Bd, M = (Q.SparseOperator(fb, fb, m) for m in (b, b.conj().T, b.conj().T @ b))
    P, D = (Q.SparseOperator(s, s, m) for m in (sp, sp.conj().T))
    g = _coupling(seed)
    return Q.LazySum(B, B, [1.0, 1.0, g, g],
                     (Q.LazyTensor(B, B, (1,), (N,)), Q.LazyTensor(B, B, (2,), (M,)),
                      Q.LazyTensor(B, B, (1, 2, 3), (A, Bd, P)), Q.LazyTensor(B, B, (1, 2, 3), (Ad, Bb, D))))


def _cavity(case, seed):
    """Hamiltonian and jump matrices of a driven, damped cavity with a spin."""
    rng = np.random.default_rng(seed)
    n, s = case["n"] + 1, case["spin2"] + 1
    a = np.kron(np.eye(s), _destroy(n))
    sp = np.kron(_raise(case["spin2"]), np.eye(n))
    delta, g, drive = rng.uniform(0, 1, 3)
    H = delta * a.conj().T @ a + g * (a @ sp + a.conj().T @ sp.conj().T) + drive * (a + a.conj().T)
    return H, [a, sp.conj().T], rng.uniform(0.1, 1, 2)


def _chain(case, seed):
    if case["kind"] == "measure":
        return W.tfim_chain(case["L"], _chain_seed(seed))
    return W.spin_chain(case["L"], _chain_seed(seed))


def prepare(case, seed):
    kind, dt = case["kind"], _np_dtype(case)
    st = dict(case=case)
    if kind in ("chain", "measure"):
        spec = _chain(case, seed)
        n = len(spec.basis)
        State = Q.Bra if case.get("op") == "bra" else Q.Ket
        st["H"] = spec.build()
        st["psi"] = State(spec.basis, _upload(_ket(case, seed, n), dt))
        if kind == "chain":
            st["out"] = State(spec.basis, Q.DeviceArray(n, dt))
            st["view"] = _view(st["out"].data)
    elif kind == "batch":
        Ls = _lengths(case)
        st["batch"] = Q.Batch([W.tfim_chain(L, _chain_seed(seed) + j).build() for j, L in enumerate(Ls)], dt)
        x = _kets(case, seed, Ls)
        st["in"], st["out"] = _upload(x, dt), Q.DeviceArray(x.numel(), dt)
        st["batch"].bind(0, _parts(st["in"], Ls), _parts(st["out"], Ls))
        st["view"] = _view(st["out"])
    elif kind == "fock":
        if case["form"] == "sparse":
            spec = W.fock_fock_spin(case["na"], case["spin2"] / 2, _chain_seed(seed))
            B, st["H"] = spec.basis, Q.SparseOperator(spec.basis, spec.basis, spec.H)
        else:
            st["H"] = _lazy_modes(case, seed)
            B = st["H"].basis_l
        _density(st, case, seed, B, dt)
    elif kind == "lt":
        dims, rng = _dims(case), np.random.default_rng(seed)
        B = _generic(dims)
        ops = tuple(Q.DenseOperator(b, b, _hermitian(rng, len(b))) for b in B.bases)
        st["H"] = Q.LazyTensor(B, B, tuple(range(1, len(dims) + 1)), ops)
        _density(st, case, seed, B, dt)
        if case["op"] == "both":
            st["Hd"] = Q.dagger(st["H"])
            st["tmp"] = Q.Operator(B, B, Q.DeviceArray(len(B) ** 2, dt))
    elif kind in ("dense", "denseket"):
        n = case["n"]
        B = Q.GenericBasis(n)
        G = _gauss(seed + 1, n, n)
        st["H"] = Q.Operator(B, B, _upload(_colmajor((G + G.conj().T) / 2).to(_t_dtype(case)), dt))
        if kind == "dense":
            _density(st, case, seed, B, dt)
        else:
            v = _ket(case, seed, n)
            st["ket"], st["bra"] = Q.Ket(B, _upload(v, dt)), Q.Bra(B, _upload(v.conj().resolve_conj(), dt))
            st["kout"], st["bout"] = Q.Ket(B, Q.DeviceArray(n, dt)), Q.Bra(B, Q.DeviceArray(n, dt))
            st["views"] = [_view(st["kout"].data), _view(st["bout"].data)]
    elif kind == "lazyket":
        st["H"] = _lazy_modes(case, seed)
        B = st["H"].basis_l
        st["psi"] = Q.Ket(B, _upload(_ket(case, seed, len(B)), dt))
        st["out"] = Q.Ket(B, Q.DeviceArray(len(B), dt))
        st["view"] = _view(st["out"].data)
    else:  # lindblad
        B = Q.tensor(Q.FockBasis(case["n"]), Q.SpinBasis(case["spin2"] / 2))
        H, J, rates = _cavity(case, seed)
        st["H"] = Q.liouvillian(Q.SparseOperator(B, B, H), [Q.SparseOperator(B, B, j) for j in J], rates)
        _density(st, case, seed, B, dt)
    torch.cuda.synchronize()
    return st


def _density(st, case, seed, B, dt):
    n = len(B)
    st["rho"] = Q.Operator(B, B, _upload(_colmajor(_rho(case, seed, n)), dt))
    st["out"] = Q.Operator(B, B, Q.DeviceArray(n * n, dt))
    st["view"] = _view(st["out"].data)


# --------------------------------------------------------------------- run
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "chain":
        if case["op"] == "step":
            Q.mul_(st["out"], st["H"], st["psi"], -1j * DT, 0.0)
            Q.axpy_(st["out"], 1.0, st["psi"])
        elif case["op"] == "bra":
            Q.mul_(st["out"], st["psi"], st["H"])
        else:
            Q.mul_(st["out"], st["H"], st["psi"])
        return st["view"]
    if kind == "batch":
        st["batch"].apply(0, -1j * DT, 0.0, 1.0)
        return st["view"]
    if kind in ("fock", "dense"):
        Q.mul_(st["out"], st["H"], st["rho"], -1j, 0.0)
        Q.mul_(st["out"], st["rho"], st["H"], 1j, 1.0)
        return st["view"]
    if kind == "lt":
        if case["op"] == "left":
            Q.mul_(st["out"], st["H"], st["rho"])
        else:
            Q.mul_(st["tmp"], st["H"], st["rho"])
            Q.mul_(st["out"], st["tmp"], st["Hd"])
        return st["view"]
    if kind == "denseket":
        Q.mul_(st["kout"], st["H"], st["ket"])
        Q.mul_(st["bout"], st["bra"], st["H"])
        return st["views"]
    if kind == "lazyket":
        Q.mul_(st["out"], st["H"], st["psi"])
        return st["view"]
    if kind == "lindblad":
        Q.mul_(st["out"], st["H"], st["rho"])
        return st["view"]
    return np.array([Q.expect(st["H"], st["psi"]), Q.variance(st["H"], st["psi"]), Q.norm(st["psi"])], dtype=np.complex128)


# -------------------------------------------------------------------- work
def work(case):
    """Bytes: each input read once, each output written once; flops: 8 per
    complex multiply-add of the operator's stored or implied entries."""
    kind, es = case["kind"], _esize(case)
    if kind == "chain":
        D = 1 << case["L"]
        return dict(bytes=2 * es * D, flops=8 * (2 * case["L"] - 1) * D)
    if kind == "batch":
        Ls = _lengths(case)
        return dict(bytes=sum(2 * es << L for L in Ls), flops=sum(8 * (2 * L - 1) << L for L in Ls))
    if kind == "fock":
        N = (case["na"] + 1) * (case["nb"] + 1) * (case["spin2"] + 1)
        return dict(bytes=2 * es * N * N, flops=2 * 8 * 3 * N * N)
    if kind == "lt":
        dims = _dims(case)
        N = math.prod(dims)
        return dict(bytes=2 * es * N * N, flops=8 * N * N * sum(dims) * (2 if case["op"] == "both" else 1))
    if kind == "dense":
        n = case["n"]
        return dict(bytes=3 * es * n * n, flops=2 * 8 * n**3)
    if kind == "denseket":
        n = case["n"]
        return dict(bytes=2 * es * n * n, flops=2 * 8 * n * n)
    if kind == "lazyket":
        N = (case["na"] + 1) * (case["nb"] + 1) * (case["spin2"] + 1)
        return dict(bytes=2 * es * N, flops=8 * 4 * N)
    if kind == "lindblad":
        d = (case["n"] + 1) * (case["spin2"] + 1)
        nnz = 9 * d * d
        return dict(bytes=2 * es * d * d + nnz * (es + 4), flops=8 * nnz)
    D = 1 << case["L"]
    return dict(bytes=es * D, flops=2 * 8 * (2 * case["L"] - 1) * D)


# ------------------------------------------------------------------- exact
def _chain_apply(spec, x):
    """H x for a chain of Pauli terms (x a complex128 device vector)."""
    D = x.numel()
    i = torch.arange(D, device=x.device)
    y = torch.zeros_like(x)
    for coef, sites, facs in spec.terms:
        mask, sign = 0, torch.ones(D, dtype=torch.float64, device=x.device)
        for s, f in zip(sites, facs):
            if f[0, 0] == 0:  # sigma_x
                mask |= 1 << (s - 1)
            else:             # sigma_z: +1 on the first state of a site, -1 on the second
                sign *= 1.0 - 2.0 * ((i >> (s - 1)) & 1)
        y += coef * (sign * x)[i ^ mask] if mask else coef * sign * x
    return y


def _device(M):
    return torch.as_tensor(M, dtype=torch.complex128, device="cuda")


def _modes_apply(case, seed, x):
    """H x with the first axis of x (N, ...) the basis index, site 1 fastest."""
    _, a, b, sp = _modes(case)
    g = _coupling(seed)
    a, b, sp = _device(a), _device(b), _device(sp)
    shape = x.shape
    t = x.reshape(sp.shape[0], b.shape[0], a.shape[0], -1)

    def on(M, t, axis):
        return torch.movedim(torch.tensordot(M, t, dims=([1], [axis])), 0, axis)

    def dag(M):
        return M.conj().T.contiguous()
    y = on(dag(a) @ a, t, 2) + on(dag(b) @ b, t, 1)
    y = y + g * on(sp, on(dag(b), on(a, t, 2), 1), 0)
    y = y + g * on(dag(sp), on(b, on(dag(a), t, 2), 1), 0)
    return y.reshape(shape)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("chain", "measure"):
        spec = _chain(case, seed)
        x = _ket(case, seed, 1 << case["L"]).to(torch.complex128)
        y = _chain_apply(spec, x)  # the chains' matrices are real and symmetric: <psi| H has the same entries
        if kind == "measure":
            e = torch.sum(x.conj() * y)
            v = torch.sum(x.conj() * _chain_apply(spec, y)) - e * e
            return np.array([e.item(), v.item(), torch.linalg.vector_norm(x).item()], dtype=np.complex128)
        return x - 1j * DT * y if case["op"] == "step" else y
    if kind == "batch":
        Ls, out = _lengths(case), []
        for j, x in enumerate(torch.split(_kets(case, seed, Ls).to(torch.complex128), [1 << L for L in Ls])):
            out.append(x - 1j * DT * _chain_apply(W.tfim_chain(Ls[j], _chain_seed(seed) + j), x))
        return torch.cat(out)
    if kind == "fock":
        n = (case["na"] + 1) * (case["nb"] + 1) * (case["spin2"] + 1)
        r = _rho(case, seed, n).to(torch.complex128)
        left = _modes_apply(case, seed, r)
        right = _modes_apply(case, seed, r.T.contiguous()).T  # H is real and symmetric: rho H = (H rho^T)^T
        return _colmajor(-1j * left + 1j * right)
    if kind == "lt":
        dims, rng = _dims(case), np.random.default_rng(seed)
        facs = [_device(_hermitian(rng, d)) for d in dims]
        r = _rho(case, seed, math.prod(dims)).to(torch.complex128)

        def on_rows(M):
            t = M.reshape(*dims[::-1], -1)
            for k, f in enumerate(facs):
                ax = len(dims) - 1 - k
                t = torch.movedim(torch.tensordot(f, t, dims=([1], [ax])), 0, ax)
            return t.reshape(M.shape)
        y = on_rows(r)
        if case["op"] == "both":
            y = on_rows(y.conj().T.contiguous()).conj().T.resolve_conj()  # y U^dagger = (U y^dagger)^dagger
        return _colmajor(y)
    if kind in ("dense", "denseket"):
        n = case["n"]
        G = _gauss(seed + 1, n, n)
        H = ((G + G.conj().T) / 2).to(_t_dtype(case)).to(torch.complex128)
        if kind == "dense":
            r = _rho(case, seed, n).to(torch.complex128)
            return _colmajor(-1j * (H @ r) + 1j * (r @ H))
        v = _ket(case, seed, n).to(torch.complex128)
        return [H @ v, H.T.contiguous() @ v.conj().resolve_conj()]
    if kind == "lazyket":
        n = (case["na"] + 1) * (case["nb"] + 1) * (case["spin2"] + 1)
        return _modes_apply(case, seed, _ket(case, seed, n).to(torch.complex128))
    H, J, rates = _cavity(case, seed)
    r = _rho(case, seed, H.shape[0]).to(torch.complex128)
    H = _device(H)
    y = -1j * (H @ r - r @ H)
    for j, k in zip(J, rates):
        j = _device(j)
        jd = j.conj().T.contiguous()
        y = y + k * (j @ r @ jd - 0.5 * (jd @ j @ r + r @ jd @ j))
    return _colmajor(y)
