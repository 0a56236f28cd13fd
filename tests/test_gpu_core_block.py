"""Block Jacobi of the cores beyond LDS (csrc/hip/core_block.hip): tiles of
known singular values whose core sizes sit at the edges of the 16-column
blocks, the 16-row fragments and the even block count, against the spectrum
they were built from; and the early verdict on a rank above the limit
against the same tiles run to convergence."""
import ctypes as C

import numpy as np
import pytest

import starsh_hip as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _tile(m, n, s, seed):
    rng = np.random.default_rng(seed)
    U, _ = np.linalg.qr(rng.standard_normal((m, len(s))))
    V, _ = np.linalg.qr(rng.standard_normal((n, len(s))))
    return U*s @ V.T


def _lowrank(engine, tiles, maxrank, os_, tol, want_s):
    L = S.lib()
    m = np.array([t.shape[0] for t in tiles], dtype=np.int32)
    n = np.array([t.shape[1] for t in tiles], dtype=np.int32)
    off = np.cumsum([0]+[t.size for t in tiles])[:-1].astype(np.int64)
    flat = np.concatenate([t.T.ravel() for t in tiles])
    d = C.c_void_p()
    assert L.starsh_hip_malloc(C.byref(d), C.c_size_t(flat.nbytes)) == 0
    vp = C.c_void_p
    ptr = lambda a: a.ctypes.data_as(vp)  # noqa: E731
    assert L.starsh_hip_memcpy_h2d(d, ptr(flat), C.c_size_t(flat.nbytes)) == 0
    uoff = np.cumsum([0]+[int(x)*maxrank for x in m])[:-1].astype(np.int64)
    voff = np.cumsum([0]+[int(x)*maxrank for x in n])[:-1].astype(np.int64)
    mn = np.minimum(m, n)
    soff = np.cumsum([0]+[int(x) for x in mn])[:-1].astype(np.int64)
    U, V = np.zeros(int(m.sum())*maxrank), np.zeros(int(n.sum())*maxrank)
    Sv = np.zeros(int(mn.sum()))
    rank = np.zeros(len(tiles), dtype=np.int32)
    info = L.starsh_hip_dense_lowrank(
        C.c_int(engine), C.c_int(len(tiles)), ptr(m), ptr(n), d, ptr(off),
        C.c_int(maxrank), C.c_int(os_), C.c_double(tol), ptr(rank), ptr(U),
        ptr(uoff), ptr(V), ptr(voff), ptr(Sv) if want_s else None,
        ptr(soff) if want_s else None)
    L.starsh_hip_free(d)
    assert info == 0
    out = []
    for t, A in enumerate(tiles):
        r = max(int(rank[t]), 0)
        u = U[uoff[t]:uoff[t]+m[t]*r].reshape(r, m[t]).T
        v = V[voff[t]:voff[t]+n[t]*r].reshape(r, n[t]).T
        out.append((int(rank[t]), u, v, Sv[soff[t]:soff[t]+mn[t]]))
    return out


def _dsvfr(s, tol):
    limit = tol*tol*np.sum(s*s)
    tail = np.cumsum((s*s)[::-1])[::-1]
    return int(np.sum(tail > limit))


@pytest.mark.parametrize("spectrum", ["square", "cluster", "graded"])
def test_core_sizes(spectrum):
    sizes = [129, 144, 160, 161, 191, 192, 193, 257, 400, 527]
    tol = 1e-3
    tiles, spectra = [], []
    for q, p in enumerate(sizes):
        i = np.arange(p)
        s = {"square": 1.0/(1.0+i)**2,
             "cluster": np.where(i < 40, 3.0, 1e-4),
             "graded": 10.0**(-7.5*i/p)}[spectrum]
        spectra.append(s)
        tiles.append(_tile(p+40, p+30, s, 10+q))
    print(f"cores {sizes} {spectrum}", flush=True)
    for (r, u, v, sv), A, s, p in zip(
            _lowrank(1, tiles, max(sizes)+20, 16, tol, True), tiles, spectra,
            sizes):
        # rounding of the sketch, the projection and the rotations: each a
        # few units of p eps of the largest singular value
        bound = 20*p*np.finfo(float).eps*s[0]
        assert np.max(np.abs(sv[:p]-s)) <= bound, (p, spectrum)
        want = _dsvfr(s, tol)
        assert r == (want if want < min(A.shape)//2 else -1), (p, spectrum)
        if r > 0:
            best = np.sqrt(np.sum(s[r:]**2))
            err = np.linalg.norm(A-u @ v.T)
            assert abs(err-best) <= np.sqrt(p)*bound+1e-9*best, (p, spectrum)
            g = u.T @ u
            assert np.max(np.abs(g-np.eye(r))) <= 100*p*np.finfo(float).eps


def test_early_verdict_on_the_rank():
    """Without singular values asked for, a tile may end as soon as its rank
    is certainly above maxrank: the verdicts equal those of the converged
    singular values, also one value to either side of the limit."""
    maxrank, os_, tol = 140, 10, 1e-2
    n, k = 300, 150
    base = np.where(np.arange(k) < 100, 1.0, 0.1)
    # energy beyond maxrank against tol^2 of the total: far above, just
    # above and just below the limit
    tiles = [_tile(n, n, np.ones(k), 1), _tile(n, n, base, 2)]
    for q, f in enumerate((1.01, 0.99)):
        s = np.r_[np.ones(maxrank), np.zeros(k-maxrank)]
        s[maxrank:] = f*tol*np.sqrt(maxrank/(k-maxrank))
        tiles.append(_tile(n, n, s, 3+q))
    tiles.append(_tile(n, n, 0.9**np.arange(k), 5))
    with_s = [x[0] for x in _lowrank(0, tiles, maxrank, os_, tol, True)]
    without = [x[0] for x in _lowrank(0, tiles, maxrank, os_, tol, False)]
    ref = [O.dlrrsdd(A, maxrank, os_, tol)[0] for A in tiles]
    print(with_s, without, ref, flush=True)
    assert without == with_s == ref
    assert ref[:3] == [-1, -1, -1] and ref[3] == maxrank


def test_many_cores_on_both_sides_of_a_launch():
    """More than 512 tiles with cores from 0 (a zero tile) to 128 rows go in
    two launches, up to 64 rows and above: every tile has its spectrum and
    rank, as in a batch of few tiles (one launch)."""
    sizes = [0, 1, 2, 63, 64, 65, 66, 127, 128]+[5, 20, 40, 70, 100]*102
    tol = 1e-3
    tiles, spectra = [], []
    for q, p in enumerate(sizes):
        s = 0.9**np.arange(p)
        spectra.append(s)
        tiles.append(_tile(p+9, p+5, s, q) if p else np.zeros((30, 20)))
    print(len(tiles), "tiles", flush=True)
    got = _lowrank(0, tiles, 140, 10, tol, True)
    few = _lowrank(0, tiles[:20], 140, 10, tol, True)
    for t, ((r, u, v, sv), s, p) in enumerate(zip(got, spectra, sizes)):
        # rounding of the sketch, the projection and the rotations: each a
        # few units of p eps of the largest singular value
        bound = 20*max(p, 1)*np.finfo(float).eps
        assert r == _dsvfr(s, tol), (t, p)
        assert np.max(np.abs(sv[:p]-s), initial=0.0) <= bound, (t, p)
        if t < len(few):
            assert few[t][0] == r
            assert np.max(np.abs(few[t][3]-sv)) <= 2*bound, (t, p)
