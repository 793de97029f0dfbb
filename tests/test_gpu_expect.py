"""Fused expect / variance (src/operators.jl:119, 139-143,
src/operators_sparse.jl:36-45, src/operators_dense.jl:219-230) on the GPU:
single-pass forms against the oracle's dense algebra, against the plain
two-pass path, and the fallbacks for operators without a fused form."""
import numpy as np
import pytest
import scipy.sparse as sp

import qob_oracle as O
import qobhip as Q
from qobhip import _lib
from qobhip import workloads as W
from test_gpu_parity import to_q
from test_gpu_qubit import build_pair, random_pauli_sum

pytestmark = pytest.mark.gpu


def _ev(M, psi):
    return np.vdot(psi, M @ psi)


def _var(M, psi):
    x = M @ psi
    return np.vdot(psi, M @ x) - np.vdot(psi, x) ** 2


@pytest.mark.parametrize("qubit", [1, 0])
@pytest.mark.parametrize("dtype,tol", [(np.complex128, 1e-12), (np.complex64, 1e-5)])
def test_expect_variance_ket_qubit_sum(qubit, dtype, tol):
    g = np.random.default_rng(90)
    L = 10
    Hq, Ho, B = build_pair(L, random_pauli_sum(g, L, 18))
    M = O.dense_of(Ho)
    psi = g.standard_normal(2 ** L) + 1j * g.standard_normal(2 ** L)
    psi /= np.linalg.norm(psi)
    if dtype == np.complex64:
        psi = psi.astype(np.complex64).astype(np.complex128)
    _lib.call("qob_tune_set", b"qubit_enable", qubit)
    try:
        k = Q.Ket(B, psi, dtype)
        e, v = Q.expect(Hq, k), Q.variance(Hq, k)
        assert abs(e - _ev(M, psi)) <= tol * max(1.0, abs(_ev(M, psi)))
        assert abs(v - _var(M, psi)) <= tol * max(1.0, abs(_var(M, psi)))
        ctx = Q.context()
        ctx.set_mode(Q.QOB_MODE_PLAIN)
        try:
            ep, vp = Q.expect(Hq, k), Q.variance(Hq, k)
        finally:
            ctx.set_mode(Q.QOB_MODE_FUSED)
        assert abs(e - ep) <= tol * max(1.0, abs(e)) and abs(v - vp) <= tol * max(1.0, abs(v))
    finally:
        _lib.call("qob_tune_set", b"qubit_enable", 1)


def test_expect_ket_fock_lazy_and_dense_fallback():
    spec = W.fock_fock_spin(4, 1.5, 3)
    lz = W.fock_fock_spin_lazy(spec)
    M = spec.H.toarray()
    g = np.random.default_rng(5)
    D = M.shape[0]
    psi = g.standard_normal(D) + 1j * g.standard_normal(D)
    k = Q.Ket(spec.basis, psi)
    assert abs(Q.expect(lz, k) - _ev(M, psi)) < 1e-12 * abs(_ev(M, psi))
    assert abs(Q.variance(lz, k) - _var(M, psi)) < 1e-11 * abs(_var(M, psi))
    # a dense LazyTensor has no fused form: the two-pass path answers
    lt = W.dense_lazytensor((4, 6), 2)
    Md = O.dense_of(O.OLazyTensor((4, 6), (4, 6), (1, 2), tuple(O.ODense(f) for f in W.dense_lazytensor_factors((4, 6), 2)), 1.0))
    p2 = g.standard_normal(24) + 1j * g.standard_normal(24)
    k2 = Q.Ket(lt.basis_l, p2)
    assert abs(Q.expect(lt, k2) - _ev(Md, p2)) < 1e-12 * abs(_ev(Md, p2))
    assert abs(Q.variance(lt, k2) - _var(Md, p2)) < 1e-11 * abs(_var(Md, p2))


@pytest.mark.parametrize("adj", [False, True])
@pytest.mark.parametrize("dtype,tol", [(np.complex128, 1e-12), (np.complex64, 1e-5)])
def test_expect_rho_sparse_and_lazy(adj, dtype, tol):
    spec = W.fock_fock_spin(5, 1.5, 4)
    n = spec.H.shape[0]
    g = np.random.default_rng(6)
    A = g.standard_normal((n, n)) + 1j * g.standard_normal((n, n))
    rho = A @ A.conj().T
    rho /= np.trace(rho)
    if dtype == np.complex64:
        rho = rho.astype(np.complex64).astype(np.complex128)
    Hs = Q.SparseOperator(spec.basis, spec.basis, spec.H)
    M = spec.H.toarray()
    if adj:
        Hs = Q.dagger(Hs)
        M = M.conj().T
    R = Q.Operator(spec.basis, spec.basis, rho, dtype)
    want = np.trace(M @ rho)
    assert abs(Q.expect(Hs, R) - want) <= tol * max(1.0, abs(want))
    lz = W.fock_fock_spin_lazy(spec)
    want = np.trace(spec.H.toarray() @ rho)
    got = Q.expect(lz, R)
    assert abs(got - want) <= tol * max(1.0, abs(want))
    ctx = Q.context()
    ctx.set_mode(Q.QOB_MODE_PLAIN)
    try:
        gp = Q.expect(lz, R)
    finally:
        ctx.set_mode(Q.QOB_MODE_FUSED)
    assert abs(gp - got) <= tol * max(1.0, abs(got))


def test_expect_follows_device_coefficients():
    spec = W.spin_chain(8, 2)
    ops = spec.build().operators
    coefs = [(lambda t, k=k: np.cos(t + k)) for k in range(len(ops))]
    H = Q.TimeDependentSum(coefs, ops, init_time=0.0)
    D = 2 ** 8
    g = np.random.default_rng(2)
    psi = g.standard_normal(D) + 1j * g.standard_normal(D)
    k = Q.Ket(spec.basis, psi)
    Q.expect(H, k)  # plans built
    for t in [0.3, 1.7]:
        H.set_time_(t)
        sh = spec.basis.shape
        Ho = O.OLazySum(D, D, H.eval_coefficients(t),
                        [O.OLazyTensor(sh, sh, tuple(i), tuple(O.OSparse.from_scipy(f) for f in fs), 1.0)
                         for _, i, fs in spec.terms])
        M = O.dense_of(Ho)
        assert abs(Q.expect(H, k) - _ev(M, psi)) < 1e-12 * max(1, abs(_ev(M, psi)))


@pytest.mark.parametrize("dtype,tol", [(np.complex128, 1e-12), (np.complex64, 1e-5)])
def test_variance_rho_sparse_lazy_dense(dtype, tol):
    """variance(op, rho) = tr(op op rho) - tr(op rho)^2 for a SparseOperator,
    its LazySum form and a dense operator, against dense algebra."""
    spec = W.fock_fock_spin(5, 1.5, 4)
    n = spec.H.shape[0]
    g = np.random.default_rng(8)
    A = g.standard_normal((n, n)) + 1j * g.standard_normal((n, n))
    rho = A @ A.conj().T
    rho /= np.trace(rho)
    if dtype == np.complex64:
        rho = rho.astype(np.complex64).astype(np.complex128)
    M = spec.H.toarray()
    R = Q.Operator(spec.basis, spec.basis, rho, dtype)
    want = np.trace(M @ M @ rho) - np.trace(M @ rho) ** 2
    scale = max(1.0, abs(np.trace(M @ M @ rho)))
    for op in (Q.SparseOperator(spec.basis, spec.basis, spec.H), W.fock_fock_spin_lazy(spec),
               Q.DenseOperator(spec.basis, spec.basis, M, dtype)):
        assert abs(Q.variance(op, R) - want) <= 10 * tol * scale, type(op).__name__


def test_time_dependent_sum_expect_variance_follow_time():
    """expect / variance of a TimeDependentSum are those of its static
    operator at the current time (src/time_dependent_operator.jl:76-80), on
    a Ket and on a density matrix."""
    from qobhip.timedependent import TimeDependentSum
    L = 6
    g = np.random.default_rng(12)
    terms = random_pauli_sum(g, L, 8)
    Hq, _, B = build_pair(L, terms)
    coefs = [lambda t, k=k: np.cos(0.3 * k * t) + 0.1j * k for k in range(len(Hq.operators))]
    tds = TimeDependentSum(list(zip(coefs, Hq.operators)))
    D = 2 ** L
    psi = g.standard_normal(D) + 1j * g.standard_normal(D)
    psi /= np.linalg.norm(psi)
    rho = np.outer(psi, psi.conj())
    k, R = Q.Ket(B, psi), Q.Operator(B, B, rho)
    for t in (0.0, 0.7, 2.5):
        tds.set_time_(t)
        c = [f(t) for f in coefs]
        M = sum(ci * O.dense_of(to_o) for ci, to_o in zip(c, _oracle_terms(Hq)))
        assert abs(Q.expect(tds, k) - _ev(M, psi)) < 1e-12 * max(1, abs(_ev(M, psi)))
        assert abs(Q.variance(tds, k) - _var(M, psi)) < 1e-11 * max(1, abs(_var(M, psi)))
        want_e = np.trace(M @ rho)
        want_v = np.trace(M @ M @ rho) - want_e ** 2
        assert abs(Q.expect(tds, R) - want_e) < 1e-12 * max(1, abs(want_e))
        assert abs(Q.variance(tds, R) - want_v) < 1e-11 * max(1, abs(want_v))


def _oracle_terms(Hq):
    """The oracle LazyTensors of a qobhip LazySum of qubit LazyTensors."""
    out = []
    for lt in Hq.operators:
        sh = tuple(lt.basis_l.shape)
        out.append(O.OLazyTensor(sh, sh, tuple(lt.indices),
                                 tuple(O.OSparse.from_scipy(sp.csc_matrix(f.csc)) for f in lt.operators),
                                 lt.factor))
    return out


@pytest.mark.parametrize("qubit", [1, 0])
@pytest.mark.parametrize("L", [1, 4, 9, 10, 11, 17])
def test_variance_one_pass_matches_plain(L, qubit):
    """Both sums of a variance from one pass over the state, against the dot
    products of the plain path: FP64 sums of 2^L products, rounding below
    2^L eps of the sums' magnitude (<= 2e-11 at 17 sites)."""
    g = np.random.default_rng(300 + L)
    H, _, B = build_pair(L, random_pauli_sum(g, L, 6))
    psi = g.standard_normal(2 ** L) + 1j * g.standard_normal(2 ** L)
    k = Q.Ket(B, psi / np.linalg.norm(psi), np.complex128)
    ctx = Q.context()
    _lib.call("qob_tune_set", b"qubit_enable", qubit)
    try:
        e, v = Q.expect(H, k), Q.variance(H, k)
        ctx.set_mode(Q.QOB_MODE_PLAIN)
        ep, vp = Q.expect(H, k), Q.variance(H, k)
    finally:
        ctx.set_mode(Q.QOB_MODE_FUSED)
        _lib.call("qob_tune_set", b"qubit_enable", 1)
    scale = max(1.0, abs(ep) ** 2, abs(vp))
    assert abs(e - ep) <= 2e-11 * scale and abs(v - vp) <= 2e-11 * scale


def test_scalars_on_many_streams_and_behind_a_long_queue():
    """Scalar results of threads with a stream each, more calls than result
    slots, and a result that is waited for behind milliseconds of queued work."""
    import concurrent.futures as cf
    import ctypes as C

    ctx = Q.context()
    g = np.random.default_rng(7)
    n = 4099
    xs = [g.standard_normal(n) + 1j * g.standard_normal(n) for _ in range(8)]
    dev = [Q.DeviceArray.from_numpy(x) for x in xs]

    def one(i):
        s = C.c_void_p()
        _lib.call("qob_stream_create", ctx.h, C.byref(s))
        try:
            got = []
            for _ in range(100):
                nrm, d = C.c_double(), _lib.qob_c64()
                _lib.call("qob_norm", ctx.h, Q.QOB_C64, n, dev[i].ptr, C.byref(nrm), s)
                _lib.call("qob_dot", ctx.h, Q.QOB_C64, n, dev[i].ptr, dev[(i + 1) % 8].ptr, C.byref(d), s)
                got.append((nrm.value, complex(d.re, d.im)))
            return got
        finally:
            _lib.call("qob_stream_destroy", ctx.h, s)

    with cf.ThreadPoolExecutor(8) as ex:
        for i, got in enumerate(ex.map(one, range(8))):
            want_n, want_d = np.linalg.norm(xs[i]), np.vdot(xs[i], xs[(i + 1) % 8])
            for a, b in got:
                assert abs(a - want_n) <= 1e-12 * want_n and abs(b - want_d) <= 1e-12 * want_n ** 2

    big = [Q.DeviceArray(1 << 24, np.complex128) for _ in range(2)]
    for _ in range(30):  # about 0.1 ms each
        _lib.call("qob_copy", ctx.h, Q.QOB_C64, 1 << 24, big[0].ptr, big[1].ptr, None)
    nrm = C.c_double()
    _lib.call("qob_norm", ctx.h, Q.QOB_C64, n, dev[0].ptr, C.byref(nrm), None)
    assert abs(nrm.value - np.linalg.norm(xs[0])) <= 1e-12 * nrm.value


@pytest.mark.parametrize("L", [1, 5, 9, 10, 11, 12])
@pytest.mark.parametrize("kind", ["hermitian", "pairs", "one_way", "phase"])
@pytest.mark.parametrize("dtype,tol", [(np.complex128, 1e-12), (np.complex64, 1e-5)])
def test_variance_of_hermitian_and_other_sums(L, kind, dtype, tol):
    """Real combinations of Pauli strings and of sigma_+ sigma_- with its
    adjoint (one pass over the state), and sums that only look like them: a
    sigma_+ without its adjoint, a complex coefficient, and coefficients that
    become complex on the device.  Against sparse algebra in ComplexF64."""
    from test_gpu_qubit import PAULI

    g = np.random.default_rng(1000 + L)
    terms = []
    for i in range(L):
        terms.append((float(g.standard_normal()), (i + 1,), [PAULI[g.choice(list("xyzn"))]]))
        if i + 1 < L:
            terms.append((float(g.standard_normal()), (i + 1, i + 2), [PAULI[g.choice(list("xyz"))] for _ in range(2)]))
            if kind != "hermitian":
                c = float(g.standard_normal())
                terms.append((c, (i + 1, i + 2), [PAULI["p"], PAULI["m"]]))
                terms.append((c, (i + 1, i + 2), [PAULI["m"], PAULI["p"]]))
    if kind == "one_way":
        terms.append((0.7, (1,), [PAULI["p"]]))
    if kind == "phase":
        terms.append((0.3 + 0.4j, (L,), [PAULI["x"]]))
    H, Ho, B = build_pair(L, terms)
    psi = g.standard_normal(2 ** L) + 1j * g.standard_normal(2 ** L)
    psi = (psi / np.linalg.norm(psi)).astype(dtype)
    k = Q.Ket(B, psi, dtype)
    psi = psi.astype(complex)
    M = sp.csr_matrix(O.dense_of(Ho)) if L <= 10 else None
    if M is None:
        M = sp.csr_matrix((2 ** L, 2 ** L), dtype=complex)
        for c, sites, mats in terms:
            K = sp.identity(1, format="csr")
            for s in range(1, L + 1):
                K = sp.kron(mats[sites.index(s)] if s in sites else sp.identity(2), K, format="csr")
            M = M + c * K
    want = _var(M, psi)
    scale = max(1.0, np.linalg.norm(M @ psi) ** 2)
    assert abs(Q.variance(H, k) - want) <= tol * scale
    # the same operator with one coefficient made complex on the device
    fac = np.array([c for c, _, _ in terms], dtype=complex)
    fac[0] *= 1j
    c, sites, mats = terms[0]
    K = sp.identity(1, format="csr")
    for s in range(1, L + 1):
        K = sp.kron(mats[sites.index(s)] if s in sites else sp.identity(2), K, format="csr")
    M2 = M + (fac[0] - c) * K
    d = Q.DeviceArray.from_numpy(fac)
    H.set_factors_device(d)
    got = Q.variance(H, k)
    assert abs(got - _var(M2, psi)) <= tol * max(1.0, np.linalg.norm(M2 @ psi) * np.linalg.norm(M2.conj().T @ psi))


@pytest.mark.parametrize("n", [1, 255, 256, 257, 2049, 8192, 8193, 70001])
@pytest.mark.parametrize("dtype,eps", [(np.complex128, 1e-13), (np.complex64, 1e-13)])
def test_scalars_of_few_and_many_workgroups(n, dtype, eps):
    """norm, dot and trace whose sums the host adds (up to eight workgroups) and
    those a second kernel adds: FP64 sums of products that are exact in FP64
    for ComplexF32 inputs."""
    g = np.random.default_rng(n)
    x = (g.standard_normal(n) + 1j * g.standard_normal(n)).astype(dtype)
    y = (g.standard_normal(n) + 1j * g.standard_normal(n)).astype(dtype)
    B = Q.GenericBasis(n)
    kx, ky = Q.Ket(B, x, dtype), Q.Ket(B, y, dtype)
    x, y = x.astype(complex), y.astype(complex)
    nx = np.linalg.norm(x)
    assert abs(Q.norm(kx) - nx) <= eps * nx
    assert abs(Q.dot(kx, ky) - np.vdot(x, y)) <= eps * nx * np.linalg.norm(y)
    if n <= 2049:
        M = np.zeros((n, n), dtype)
        M[np.arange(n), np.arange(n)] = y
        assert abs(Q.tr(Q.Operator(B, B, M, dtype)) - y.sum()) <= eps * abs(y).sum()


@pytest.mark.parametrize("mode", ["fused", "plain"])
@pytest.mark.parametrize("kind", ["sparse_dense", "wide", "three", "sum"])
@pytest.mark.parametrize("dtype,eps", [(np.complex128, 2.0 ** -52), (np.complex64, 2.0 ** -23)])
def test_variance_ket_of_several_passes(kind, mode, dtype, eps):
    """variance on a Ket of operators whose application goes through a
    temporary of its own: mode chains (a sparse factor beside a dense one,
    factors wider than a site group takes) of two and three steps, and a sum
    whose second term is applied over the first term's result.  An application
    of factors of widths d rounds by less than 3/2 (sum d + 4) eps |M| |psi| per
    element (complex products and sums, 3 for the modulus of both parts)."""
    shape = {"sparse_dense": (6, 5), "wide": (70, 70), "three": (12, 45, 7), "sum": (41, 44)}[kind]
    g = np.random.default_rng(41)
    bases = [Q.GenericBasis(d) for d in shape]
    B = Q.tensor(*bases)

    def factors(sparse):
        ms, fs = [], []
        for i, (d, b) in enumerate(zip(shape, bases)):
            m = (g.standard_normal((d, d)) + 1j * g.standard_normal((d, d))) / d
            if i in sparse:
                m = m * (g.random((d, d)) < 0.4)
            m = m + np.diag(1 + g.random(d))
            ms.append(m)
            fs.append(Q.SparseOperator(b, b, sp.csc_matrix(m)) if i in sparse else Q.DenseOperator(b, b, m))
        return ms, tuple(fs)

    def dense(ms):
        K = np.ones((1, 1))
        for m in ms:  # the first site is the fastest
            K = np.kron(m, K)
        return K

    sites = tuple(range(1, len(shape) + 1))
    if kind == "sum":
        (ma, fa), (mb, fb) = factors(()), factors((0,))
        op = Q.LazySum(B, B, [0.7, -1.3j], (Q.LazyTensor(B, B, sites, fa), Q.LazyTensor(B, B, sites, fb)))
        M = 0.7 * dense(ma) - 1.3j * dense(mb)
        absM = 0.7 * abs(dense(ma)) + 1.3 * abs(dense(mb))
    else:
        ms, fs = factors({"sparse_dense": (0,), "three": (2,)}.get(kind, ()))
        op, M = Q.LazyTensor(B, B, sites, fs), dense(ms)
        absM = abs(M)
    psi = g.standard_normal(len(B)) + 1j * g.standard_normal(len(B))
    psi = (psi / np.linalg.norm(psi)).astype(dtype)
    k = Q.Ket(B, psi, dtype)
    want = _var(M, psi.astype(complex))
    a = abs(psi.astype(complex))
    bound = 3 * (sum(shape) + 4) * eps * (a @ (absM @ (absM @ a)) + (a @ (absM @ a)) ** 2)
    ctx = Q.context()
    ctx.set_mode(Q.QOB_MODE_PLAIN if mode == "plain" else Q.QOB_MODE_FUSED)
    try:
        got = Q.variance(op, k)
    finally:
        ctx.set_mode(Q.QOB_MODE_FUSED)
    assert abs(got - want) <= bound


@pytest.mark.parametrize("shape", [(15, 17), (16, 16), (1, 257), (510, 514), (512, 512), (513, 512)])
@pytest.mark.parametrize("dtype,eps", [(np.complex128, 2.0 ** -52), (np.complex64, 2.0 ** -23)])
def test_expect_and_variance_of_sparse_sums_by_length(shape, dtype, eps):
    """Around one workgroup of 256 elements and the largest grid (2^18 elements):
    the sum alone (expect) and with conj(psi) op psi beside it (variance).  An
    element of op psi is a sum of at most 5 complex products of up to 3 factors:
    less than 12 eps |M| |psi|."""
    g = np.random.default_rng(sum(shape))
    ba, bb = (Q.GenericBasis(d) for d in shape)
    B = Q.tensor(ba, bb)

    def factor(d):
        m = sp.diags([g.standard_normal(d - 1) + 0.5j, g.standard_normal(d) + 0j], [1, 0] if d > 1 else [0], shape=(d, d)) \
            if d > 1 else sp.csc_matrix([[0.8 + 0.3j]])
        return sp.csc_matrix(m).astype(complex)
    a, b, c, d = factor(shape[0]), factor(shape[1]), factor(shape[0]), factor(shape[1])
    S = lambda bas, m: Q.SparseOperator(bas, bas, m)
    co = [0.7, -0.4 + 0.2j, 1.1j]
    op = Q.LazySum(B, B, co, (Q.LazyTensor(B, B, (1,), (S(ba, a),)), Q.LazyTensor(B, B, (2,), (S(bb, b),)),
                              Q.LazyTensor(B, B, (1, 2), (S(ba, c), S(bb, d)))))
    parts = (sp.kron(sp.identity(shape[1]), a), sp.kron(b, sp.identity(shape[0])), sp.kron(d, c))
    M = sum(z * m for z, m in zip(co, parts)).tocsr()
    W = sum(abs(z) * abs(m) for z, m in zip(co, parts)).tocsr()
    psi = g.standard_normal(len(B)) + 1j * g.standard_normal(len(B))
    psi = (psi / np.linalg.norm(psi)).astype(dtype)
    k, x = Q.Ket(B, psi, dtype), psi.astype(complex)
    r = abs(x)
    e, e2 = np.vdot(x, M @ x), np.vdot(x, M @ (M @ x))
    assert abs(Q.expect(op, k) - e) <= 12 * eps * (r @ (W @ r))
    assert abs(Q.variance(op, k) - (e2 - e * e)) <= 30 * eps * (r @ (W @ (W @ r)) + (r @ (W @ r)) ** 2)


def test_scalars_of_many_threads_and_streams_word_by_word():
    """Scalar results of four threads in turn over states whose sums are whole
    numbers: every result is exactly its own (a word of another call, or of the
    slot's last one, would change it), by one workgroup's sums, several, and two
    launches, one sum and two."""
    import ctypes as C
    import threading

    from qobhip.serve import new_stream
    g = np.random.default_rng(8)
    L = 6
    Hq, _, B = build_pair(L, [(1.0, (i + 1,), [np.diag([1.0 + 0j, -1.0])]) for i in range(L)])
    Hq._handle()
    ctx, errors = Q.context(), []

    def work(seed):
        r = np.random.default_rng(seed)
        st = new_stream()
        try:
            xs = []
            for n in (3, 300, 2048, 5000):
                x = (r.integers(-9, 10, n) + 1j * r.integers(-9, 10, n)).astype(complex)
                y = (r.integers(-9, 10, n) + 1j * r.integers(-9, 10, n)).astype(complex)
                xs.append((n, Q.DeviceArray.from_numpy(x), Q.DeviceArray.from_numpy(y), np.vdot(x, y)))
            p = (r.integers(-9, 10, 2 ** L) + 1j * r.integers(-9, 10, 2 ** L)).astype(complex)
            z = L - 2 * np.array([bin(i).count("1") for i in range(2 ** L)])
            pd, e, e2 = Q.DeviceArray.from_numpy(p), (abs(p) ** 2 * z).sum(), (abs(p) ** 2 * z ** 2).sum()
            e, e2 = round(e), round(e2)
            Q.synchronize()
            out = _lib.qob_c64()
            for _ in range(300):
                for n, x, y, want in xs:
                    _lib.call("qob_dot", ctx.h, x.qdt, n, x.ptr, y.ptr, C.byref(out), st)
                    if complex(out.re, out.im) != want:
                        errors.append((seed, n, out.re, out.im, want))
                _lib.call("qob_expect_ket", ctx.h, pd.qdt, Hq._handle(), pd.ptr, 2 ** L, C.byref(out), st)
                if complex(out.re, out.im) != e:
                    errors.append((seed, "expect", out.re, out.im, e))
                _lib.call("qob_variance_ket", ctx.h, pd.qdt, Hq._handle(), pd.ptr, 2 ** L, C.byref(out), st)
                if complex(out.re, out.im) != e2 - e * e:
                    errors.append((seed, "variance", out.re, out.im, e2 - e * e))
        finally:
            _lib.call("qob_stream_destroy", ctx.h, st)
    ts = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors[:5]
