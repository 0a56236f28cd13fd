"""Products with compressed matrices at the sizes where the kernels of
csrc/hip/tlr.hip change course: row strips of 16, 32 and 64, tiles that are
no multiple of 16 or 64 rows, ranks around the 16- and 32-column groups and
the 64-column pieces of an entry, one right-hand side (lane sums) and more
(MFMA, groups of 16), dense tiles and their transposes."""
import ctypes as C
from fractions import Fraction

import numpy as np
import pytest

import starsh_hip as S

pytestmark = pytest.mark.gpu


def _array(a):
    A = C.POINTER(S.Array)()
    assert S.lib().array_from_buffer(
        C.byref(A), C.c_int(2), (C.c_int*2)(*a.shape), C.c_char(b"d"),
        C.c_char(b"F"), a.ctypes.data_as(C.c_void_p)) == 0
    return A


def _ints(v):
    libc = C.CDLL(None)
    libc.malloc.restype = C.c_void_p
    a = (S.STARSH_int*max(1, len(v)))(*v)
    p = libc.malloc(C.c_size_t(C.sizeof(a)))
    C.memmove(p, a, C.sizeof(a))
    return C.cast(p, C.POINTER(S.STARSH_int))


def _operator(N, nb, symm, ranks, rng):
    """A BLRM of random factors; ranks cycle over the tiles, -1: dense.
    Returns it, the dense matrix and what has to stay alive."""
    p = S.TLRProblem("spatial", N, 2, nb, symm=symm, kernel="exp",
                     points=rng.random((2, N)))
    st, sz = p.cluster_ranges()
    A = np.zeros((N, N))
    far, near, U, V, D, rk, keep = [], [], [], [], [], [], [p]
    for t, (i, j) in enumerate(p.tiles()):
        r = ranks[t % len(ranks)]
        ri, rj = slice(st[i], st[i]+sz[i]), slice(st[j], st[j]+sz[j])
        if r < 0:
            d = np.asfortranarray(rng.standard_normal((sz[i], sz[j])))
            keep.append(d)
            near += [i, j]
            D.append(_array(d))
            block = d
        else:
            r = min(r, sz[i], sz[j])
            u = np.asfortranarray(rng.standard_normal((sz[i], r)))
            v = np.asfortranarray(rng.standard_normal((sz[j], r)))
            keep += [u, v]
            far += [i, j]
            rk.append(r)
            U.append(_array(u))
            V.append(_array(v))
            block = u @ v.T
        A[ri, rj] = block
        if symm == "S" and i != j:
            A[rj, ri] = block.T
    F = C.POINTER(S.BLRF)()
    assert S.lib().starsh_blrf_new_from_coo(
        C.byref(F), p.P, C.c_char(symm.encode()), p.C, p.C,
        S.STARSH_int(len(rk)), _ints(far), S.STARSH_int(len(D)),
        _ints(near), C.c_int(p.F.contents.type)) == 0
    M = S.BLRM()
    PA = C.POINTER(S.Array)
    M.format = F
    M.far_rank = (C.c_int*max(1, len(rk)))(*rk)
    M.far_U = (PA*max(1, len(U)))(*U)
    M.far_V = (PA*max(1, len(V)))(*V)
    M.near_D = (PA*max(1, len(D)))(*D)
    M.onfly = 0
    return M, A, keep


@pytest.mark.parametrize("N,nb,symm,ranks", [
    (40, 40, "S", [3]),
    (37, 15, "N", [1, 0, 15, -1]),
    (331, 47, "S", [16, 17, -1, 0, 1]),
    (1030, 250, "S", [31, 32, 33, -1]),
    (1030, 250, "N", [64, 65, 15, -1, 100]),
    (500, 100, "S", [0]),
    (17000, 2048, "S", [5, 40, 1]),
    (33000, 1601, "N", [2, 18]),
    (33000, 1601, "N", [30])])
def test_products(N, nb, symm, ranks):
    L = S.lib()
    rng = np.random.default_rng(N)
    if N > 5000:
        # too large to hold densely: products of the factors instead
        M, apply, keep = _large(N, nb, symm, ranks, rng)
    else:
        M, A, keep = _operator(N, nb, symm, ranks, rng)

        def apply(X):
            return A @ X
    for nrhs in ([1, 3] if N > 5000 else [1, 2, 15, 16, 17, 33]):
        print(f"N={N} nb={nb} {symm} ranks {ranks} nrhs {nrhs}", flush=True)
        X = np.asfortranarray(rng.standard_normal((N, nrhs)))
        Y = np.asfortranarray(rng.standard_normal((N, nrhs)))
        ref = 1.5*apply(X)-0.25*Y
        dp = C.POINTER(C.c_double)
        assert L.starsh_blrm__dmml_hip(
            C.cast(C.byref(M), C.c_void_p), nrhs, 1.5, X.ctypes.data_as(dp),
            N, -0.25, Y.ctypes.data_as(dp), N) == 0
        # sums of at most N products of up to 100 terms each
        scale = max(np.max(np.abs(ref)), 1.0)
        assert np.max(np.abs(Y-ref)) <= 1e-13*scale*np.sqrt(N)


def _large(N, nb, symm, ranks, rng):
    p = S.TLRProblem("spatial", N, 2, nb, symm=symm, kernel="exp",
                     points=rng.random((2, N)))
    st, sz = p.cluster_ranges()
    parts, U, V, rk, keep = [], [], [], [], [p]
    for t, (i, j) in enumerate(p.tiles()):
        r = ranks[t % len(ranks)]
        u = np.asfortranarray(rng.standard_normal((sz[i], r)))
        v = np.asfortranarray(rng.standard_normal((sz[j], r)))
        parts.append((slice(st[i], st[i]+sz[i]), slice(st[j], st[j]+sz[j]),
                      u, v, symm == "S" and i != j))
        keep += [u, v]
        rk.append(r)
        U.append(_array(u))
        V.append(_array(v))
    M = S.BLRM()
    PA = C.POINTER(S.Array)
    M.format = p.F
    M.far_rank = (C.c_int*len(rk))(*rk)
    M.far_U = (PA*len(U))(*U)
    M.far_V = (PA*len(V))(*V)
    M.onfly = 0

    def apply(X):
        Y = np.zeros_like(X)
        for ri, rj, u, v, both in parts:
            Y[ri] += u @ (v.T @ X[rj])
            if both:
                Y[rj] += v @ (u.T @ X[ri])
        return Y
    return M, apply, keep

@pytest.mark.parametrize("nrhs", [1, 2])
def test_long_sums_go_in_blocks(nrhs):
    """Sums of 1700 products that start with 1 and go on with values below
    half a unit of it, which a single chain of additions loses one by one:
    dense tiles, transposed dense tiles and coefficients.  Every kernel adds
    at most 32 products to one partial sum, and then the partial sums (at
    most 28 per wave, and four waves): the error is at most that many units
    of rounding."""
    L = S.lib()
    n = 1700
    t = 0.99*2.0**-54
    exact = float(Fraction(1)+(n-1)*Fraction(t))
    u = 2.0**-53
    col = np.full(n, t)
    col[0] = 1.0
    ones = np.ones((n, 1))
    p = S.TLRProblem("spatial", 2*n, 2, n, symm="S", kernel="exp",
                     points=np.random.default_rng(0).random((2, 2*n)))
    tiles = [tuple(x) for x in p.tiles()]
    assert sorted(tiles) == [(0, 0), (1, 0), (1, 1)]
    dense = np.asfortranarray(np.tile(col, (n, 1)))
    by_rows = np.asfortranarray(np.tile(col[:, None], (1, n)))
    lowrank = (ones, np.asfortranarray(col[:, None]))
    none = (np.zeros((n, 0), order="F"), np.zeros((n, 0), order="F"))
    # what each block row of y = A (1, ..., 1) starts its sums with
    for name, blocks, where in (
            ("dense", {(0, 0): dense, (1, 0): none, (1, 1): none}, 0),
            ("transposed", {(0, 0): none, (1, 0): by_rows, (1, 1): none}, 0),
            ("coefficients", {(0, 0): lowrank, (1, 0): none,
                              (1, 1): none}, 0),
            ("twin's coefficients", {(0, 0): none, (1, 0): lowrank[::-1],
                                     (1, 1): none}, 0)):
        near = [q for q in tiles if not isinstance(blocks[q], tuple)]
        far = [q for q in tiles if isinstance(blocks[q], tuple)]
        F = C.POINTER(S.BLRF)()
        assert L.starsh_blrf_new_from_coo(
            C.byref(F), p.P, C.c_char(b"S"), p.C, p.C,
            S.STARSH_int(len(far)), _ints([x for q in far for x in q]),
            S.STARSH_int(len(near)), _ints([x for q in near for x in q]),
            C.c_int(p.F.contents.type)) == 0
        PA = C.POINTER(S.Array)
        M = S.BLRM()
        M.format = F
        rk = [blocks[q][0].shape[1] for q in far]
        one = np.ones((n, 1), order="F")
        UV = [[_array(f if f.shape[1] else one) for f in blocks[q]]
              for q in far]
        M.far_rank = (C.c_int*max(1, len(far)))(*rk)
        M.far_U = (PA*max(1, len(far)))(*[x[0] for x in UV])
        M.far_V = (PA*max(1, len(far)))(*[x[1] for x in UV])
        M.near_D = (PA*max(1, len(near)))(*[_array(blocks[q]) for q in near])
        M.onfly = 0
        X = np.ones((2*n, nrhs), order="F")
        Y = np.zeros((2*n, nrhs), order="F")
        dp = C.POINTER(C.c_double)
        assert L.starsh_blrm__dmml_hip(
            C.cast(C.byref(M), C.c_void_p), nrhs, 1.0, X.ctypes.data_as(dp),
            2*n, 0.0, Y.ctypes.data_as(dp), 2*n) == 0
        got = Y[where*n:(where+1)*n]
        err = np.max(np.abs(got-exact))/u
        print(name, nrhs, "error", err, "units", flush=True)
        assert err <= 32+28+4


def test_uploads_from_two_threads():
    """Two operators uploaded at the same time (the second finds the pinned
    ring taken): both hold the same factors, so their products are the
    same, bit for bit."""
    import threading
    L = S.lib()
    N = 20000
    M, apply, keep = _large(N, 1000, "N", [10, 20], np.random.default_rng(1))
    T = [C.c_void_p(), C.c_void_p()]
    info = [None, None]

    def make(q):
        info[q] = L.starsh_hip_tlr_new(C.byref(T[q]), C.byref(M))

    threads = [threading.Thread(target=make, args=(q,)) for q in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert info == [0, 0]
    X = np.random.default_rng(2).standard_normal(N)
    out = []
    d = [C.c_void_p(), C.c_void_p()]
    for x in d:
        assert L.starsh_hip_malloc(C.byref(x), C.c_size_t(8*N)) == 0
    vp = C.c_void_p
    assert L.starsh_hip_memcpy_h2d(d[0], X.ctypes.data_as(vp),
                                   C.c_size_t(8*N)) == 0
    for t in T:
        Y = np.zeros(N)
        assert L.starsh_hip_tlr_dmml(t, C.c_int(1), C.c_double(1.0), d[0],
                                     C.c_int(N), C.c_double(0.0), d[1],
                                     C.c_int(N)) == 0
        assert L.starsh_hip_memcpy_d2h(Y.ctypes.data_as(vp), d[1],
                                       C.c_size_t(8*N)) == 0
        out.append(Y)
        L.starsh_hip_tlr_free(t)
    for x in d:
        L.starsh_hip_free(x)
    assert np.array_equal(out[0], out[1])
    ref = apply(X[:, None])[:, 0]
    assert np.max(np.abs(out[0]-ref)) <= 1e-13*np.max(np.abs(ref))*np.sqrt(N)


@pytest.mark.parametrize("total", [(1 << 20)+1, 1 << 21, (1 << 21)+1,
                                   3*(1 << 21)+5, 11*(1 << 21)+7])
def test_upload_sizes(total):
    """Arrays of odd lengths, empty ones among them, whose sum sits at the
    edges of the pinned ring's slots: one slot, its growth, and more slots
    than it holds, from a ring that starts empty."""
    L = S.lib()
    if total == (1 << 20)+1:
        assert L.starsh_hip_set_option(b"release_workspace",
                                       C.c_double(0.0)) == 0
    data = np.random.default_rng(total).random(total)
    cuts = np.sort(np.random.default_rng(1).integers(0, total, 40))
    cuts[5] = cuts[6]
    parts = [np.ascontiguousarray(x) for x in np.split(data, cuts)]
    src = (C.c_void_p*len(parts))(*[x.ctypes.data for x in parts])
    size = (C.c_int64*len(parts))(*[len(x) for x in parts])
    d = C.c_void_p()
    assert L.starsh_hip_malloc(C.byref(d), C.c_size_t(8*total)) == 0
    assert L.hip_upload_segments(d, C.c_int64(len(parts)), src, size) == 0
    back = np.zeros(total)
    assert L.starsh_hip_memcpy_d2h(back.ctypes.data_as(C.c_void_p), d,
                                   C.c_size_t(8*total)) == 0
    L.starsh_hip_free(d)
    assert np.array_equal(back, data)


@pytest.mark.parametrize("nrhs", [1, 3])
def test_cg_solves(nrhs):
    """Random columns, and one that is an eigenvector and converges at once,
    against the dense solution."""
    N = 700
    fn = S.init("HIP", oversample=16)
    rng = np.random.default_rng(3)
    p = S.TLRProblem("spatial", N, 2, 100, kernel="exp", beta=0.1,
                     noise=0.5, points=rng.random((2, N)))
    assert p.approximate(60, 1e-9, 0, fn) == 0
    A = p.dmml(np.eye(N))
    X = rng.standard_normal((N, nrhs))
    if nrhs > 1:
        X[:, 1] = np.linalg.eigh(0.5*(A+A.T))[1][:, -1]
    B = A @ X
    it, Y = p.cg(B, np.zeros_like(B), 1e-10)
    print("iterations", it, flush=True)
    assert 0 < it < N
    # |x - x'| <= cond |r|/|b| |x|, cond below |A|/noise
    cond = np.linalg.norm(A, 2)/0.5
    for q in range(nrhs):
        assert np.linalg.norm(Y[:, q]-X[:, q]) <= 2e-10*cond*np.linalg.norm(
            X[:, q])
    p.free_matrix()


def _covariance(N=700):
    fn = S.init("HIP", oversample=16)
    rng = np.random.default_rng(3)
    p = S.TLRProblem("spatial", N, 2, 100, kernel="exp", beta=0.1,
                     noise=0.01, points=rng.random((2, N)))
    assert p.approximate(60, 1e-9, 0, fn) == 0
    return p, p.dmml(np.eye(N)), rng


def _cg(A, b, tol):
    """The reference's iteration for one column: the index at which |r| <
    tol |r_0|, the solution, and |r|/(tol |r_0|) of the last two."""
    x, r = np.zeros_like(b), b.copy()
    p, rs = r.copy(), b @ b
    check = tol*np.sqrt(rs)
    ratio = [np.inf, 1.0/tol]
    for it in range(len(b)):
        q = A @ p
        a = rs/(p @ q)
        x += a*p
        r -= a*q
        new = r @ r
        ratio = [ratio[1], np.sqrt(new)/check]
        if ratio[1] < 1.0:
            return it, x, ratio
        p = r+new/rs*p
        rs = new
    raise AssertionError("no convergence")


def test_cg_columns_stop_on_their_own():
    """Columns of one block that converge at different iterations, between
    the ones at which the states are read back, at a tolerance so loose that
    more iterations would change them visibly.  A block of four copies of one
    column takes the same steps for it, bit for bit, and ends with it: each
    column of the mixed block equals that, and the index returned is the last
    one's.  (Another summation order is no measure: 23 iterations of CG carry
    a rounding error of the product to 1e-4 of the solution here.)"""
    p, A, rng = _covariance()
    N, tol = len(A), 1e-2
    base = rng.standard_normal((N, 4))
    X = np.stack([base[:, 0], A @ base[:, 1], A @ (A @ base[:, 2]),
                  np.linalg.eigh(0.5*(A+A.T))[1][:, -3:] @ [1.0, 2.0, 3.0]],
                 axis=1)
    B = A @ X
    ref = [_cg(A, B[:, q], tol) for q in range(4)]
    its = [r[0] for r in ref]
    print("iterations", its, "residuals at them", [r[2] for r in ref],
          flush=True)
    assert len(set(its)) == 4
    # no column sits at the edge of the rule, where rounding would decide
    assert all(r[2][0] > 1.01 and r[2][1] < 0.99 for r in ref)
    it, Y = p.cg(B, np.zeros_like(B), tol)
    assert it == max(its)
    for q in range(4):
        four = np.repeat(B[:, q:q+1], 4, axis=1)
        one, y = p.cg(four, np.zeros_like(four), tol)
        assert one == its[q]
        assert np.array_equal(Y[:, q], y[:, q])
        # one right-hand side goes through other kernels
        assert p.cg(B[:, q:q+1], np.zeros((N, 1)), tol)[0] == its[q]
    # ... and more steps of the columns that stop early would be seen
    for q in (1, 2):
        more = _cg(A, B[:, q], tol*0.2)[1]
        assert np.linalg.norm(more-ref[q][1]) > 1e-6*np.linalg.norm(more)
    p.free_matrix()


def test_cg_leaves_columns_of_a_negative_rule_alone():
    """A negative tolerance gives every column a negative check value: the
    reference skips such columns and never converges."""
    p, A, rng = _covariance(300)
    B = rng.standard_normal((len(A), 2))
    X0 = rng.standard_normal(B.shape)
    it, X = p.cg(B, X0, -0.5)
    assert it == -1 and np.array_equal(X, X0)
    p.free_matrix()
