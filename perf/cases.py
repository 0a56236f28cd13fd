"""Workloads of the tile low-rank (TLR) compressor, through its public entry
points: compression of kernel matrices (both forms of the randomized engine,
the exact SVD engine, a batch of problems), products and conjugate gradients
with the compressed matrix, and the Morton sort of the points.

A compression hands out factors that are unique only up to signs and bases,
so each compression case goes on to what such a factorization is made for:
the product of the compressed matrix with a block of vectors.  It returns the
ranks of the tiles and that product.

listed() are the cases, draw(rng) gives one more of the same ranges,
prepare(case, seed) makes what a program holds before the call, run(state) is
one pass, work(case) the bytes and operations a pass cannot do without, and
exact(case, seed) the same outputs in plain 64-bit torch.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(
    os.path.abspath(__file__))), "stars-h_amd"))
import starsh_hip as S  # noqa: E402


def listed():
    return [
        # The smallest compression of the test suite (2D exponential
        # covariance, 55 tiles of 250, tight tolerance): latency and the
        # number of launches count.
        dict(name="compress small exp", kind="compress", form="plain",
             kernel="exp", ndim=2, N=2500, nb=250, maxrank=100, os=10,
             tol=1e-9, beta=0.1, nu=0.5, nrhs=1),
        # The headline matrix of the benchmark, FP64 form: geostatistics on
        # 64000 sites, 820 tiles of 1600.
        dict(name="compress 64k plain", kind="compress", form="plain",
             kernel="sqrexp", ndim=2, N=64000, nb=1600, maxrank=400, os=16,
             tol=1e-7, beta=0.1, nu=0.5, nrhs=1),
        # The same matrix in the mixed form.
        dict(name="compress 64k mixed", kind="compress", form="mixed",
             kernel="sqrexp", ndim=2, N=64000, nb=1600, maxrank=400, os=16,
             tol=1e-7, beta=0.1, nu=0.5, nrhs=1),
        # Tiles of slowly decaying spectrum (3D Matern covariance, ranks up
        # to 512, some tiles not low-rank at all) at half the benchmark's
        # point count: the largest compression.
        dict(name="compress matern mixed", kind="compress", form="mixed",
             kernel="matern", ndim=3, N=65536, nb=2048, maxrank=512, os=16,
             tol=1e-7, beta=0.1, nu=1.5, nrhs=4),
        # Boundary-element-like points on spheres, oscillating kernel,
        # ragged last tile, FP64 form.
        dict(name="compress sin plain", kind="compress", form="plain",
             kernel="sin", ndim=3, N=25000, nb=1536, maxrank=384, os=16,
             tol=1e-6, beta=0.1, nu=0.5, nrhs=1),
        # A likelihood sweep: many problems of different sizes and
        # correlation lengths in one call, tiles of 900 to 2800.
        dict(name="batch of 12 exp", kind="batch", form="mixed",
             kernel="exp", ndim=2, N=20000, problems=12, maxrank=384, os=16,
             tol=1e-7, nrhs=1),
        # The exact engine (STARSH_LRENGINE=SVD) on an odd-sized problem.
        dict(name="compress svd exp", kind="compress", form="svd",
             kernel="exp", ndim=2, N=9973, nb=1000, maxrank=150, os=10,
             tol=1e-7, beta=0.1, nu=0.5, nrhs=1),
        # Repeated products with a small operator: latency.
        dict(name="product small", kind="product", symm="S", N=2500, nb=250,
             rank=30, near=0, nrhs=1),
        # Products with the compressed 64000-point matrix, one vector (an
        # iterative solver's step): bandwidth.
        dict(name="product 64k", kind="product", symm="S", N=64000, nb=1600,
             rank=31, near=0, nrhs=1),
        # A block of vectors, ragged nonsymmetric tiling, some dense tiles.
        dict(name="product block", kind="product", symm="N", N=30000,
             nb=1700, rank=90, near=12, nrhs=10),
        # Conjugate gradients on a compressed covariance with a nugget, from
        # host arrays: kriging weights.
        dict(name="cg 10k", kind="cg", kernel="exp", ndim=2, N=10000,
             nb=1000, maxrank=300, os=16, tol=1e-9, beta=0.1, nu=0.5,
             noise=0.01, nrhs=1),
        # Morton order of a million points, the input step of a large
        # problem whose points are on the GPU already.
        dict(name="zsort 1m", kind="zsort", N=1000000, ndim=3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["compress"]*6+["batch", "product", "product",
                                      "product", "cg", "zsort"])
    if kind == "zsort":
        return dict(kind=kind, N=_log_int(rng, 1000, 2000000),
                    ndim=rng.randint(1, 4))
    if kind == "product":
        N = _log_int(rng, 1000, 64000)
        nb = max(100, min(2048, int(math.sqrt(40.0*N)*rng.uniform(0.7, 1.3))))
        symm = rng.choice("SSN")
        return dict(kind=kind, symm=symm, N=N, nb=nb,
                    rank=_log_int(rng, 4, max(5, nb//12)),
                    near=rng.choice([0, 0, 3, 11]),
                    nrhs=rng.choice([1, 1, 2, 3, 4, 7, 16]))
    if kind == "cg":
        N = _log_int(rng, 1500, 12000)
        return dict(kind=kind, kernel="exp", ndim=2, N=N,
                    nb=max(150, min(1200, int(math.sqrt(100.0*N)))),
                    maxrank=300, os=16, tol=1e-9,
                    beta=rng.uniform(0.05, 0.2), nu=0.5,
                    noise=rng.choice([0.003, 0.01, 0.1]),
                    nrhs=rng.choice([1, 1, 2, 5]))
    if kind == "batch":
        return dict(kind=kind, form=rng.choice(["mixed", "mixed", "plain"]),
                    kernel="exp", ndim=2, N=_log_int(rng, 4000, 20000),
                    problems=rng.randint(2, 12), maxrank=384, os=16,
                    tol=1e-7, nrhs=1)
    kernel = rng.choice(["sqrexp", "sqrexp", "exp", "exp", "matern",
                         "coulomb", "sin"])
    ndim = 2 if kernel in ("sqrexp", "exp") else 3
    form = rng.choice(["plain", "plain", "mixed", "mixed", "mixed", "svd",
                       "rrqr"])
    exact_engine = form in ("svd", "rrqr")
    if kernel in ("matern", "coulomb", "sin"):
        N = _log_int(rng, 3000, 8000 if exact_engine else 40000)
        nb = max(500, min(2048, int(math.sqrt(64.0*N)*rng.uniform(0.8,
                                                                  1.25))))
        tol = 1e-6 if kernel in ("coulomb", "sin") else \
            rng.choice([1e-6, 1e-7])
        maxrank = nb//4
    else:
        N = _log_int(rng, 2000, 12000 if exact_engine else 64000)
        nb = max(200, min(3000, int(math.sqrt(40.0*N)*rng.uniform(0.7,
                                                                  1.6))))
        tol = rng.choice([1e-5, 1e-7, 1e-7, 1e-9])
        maxrank = max(100, nb//4)
    return dict(kind="compress", form=form, kernel=kernel, ndim=ndim, N=N,
                nb=nb, maxrank=min(maxrank, 512), os=rng.choice([10, 16]),
                tol=tol, beta=rng.uniform(0.05, 0.3), nu=rng.choice(
                    [0.5, 1.5, 2.5]), nrhs=rng.choice([1, 1, 4]))


# ---- points, in Morton order

def _morton(x):
    """The points (ndim x n) in Morton order: dimension ndim-1's bit first
    at every level, coordinates scaled to 32 bits."""
    nd, n = x.shape
    bits = 63//nd if nd > 1 else 32
    bits = min(bits, 32)
    lo = x.min(axis=1, keepdims=True)
    rng = x.max(axis=1, keepdims=True)-lo
    u = ((x-lo)/rng*4294967295.0).astype(np.uint64) >> np.uint64(32-bits)
    key = np.zeros(n, dtype=np.uint64)
    for b in range(bits):
        for d in range(nd):
            key |= (u[d] >> np.uint64(b) & np.uint64(1)) << np.uint64(
                b*nd+d)
    return np.ascontiguousarray(x[:, np.argsort(key, kind="stable")])


def _points(kernel, ndim, N, seed):
    """Jittered grid in 2D, uniform in 3D, points on spheres for the
    particle kernels."""
    rng = np.random.default_rng(seed)
    if kernel in ("coulomb", "sin"):
        per = 500
        ns = -(-N//per)
        c = np.repeat(rng.uniform(0, 1, (3, ns)), per, axis=1)[:, :N]
        v = rng.standard_normal((3, N))
        return _morton(c+0.02*v/np.sqrt((v*v).sum(axis=0)))
    if ndim == 2:
        side = math.isqrt(N-1)+1
        g = np.arange(side*side)[:N]
        x = np.stack([g % side, g//side])+0.5
        return _morton((x+rng.uniform(-0.4, 0.4, (2, N)))/side)
    return _morton(rng.uniform(0, 1, (ndim, N)))


def _batch_specs(case):
    """Sizes, tiles and correlation lengths of a batch: the sizes spread
    over a factor of ten up to N, the tile from the size."""
    q = case["problems"]
    out = []
    for i in range(q):
        f = (i+1)/q
        N = int(round(case["N"]*10.0**(f-1.0)))
        out.append((N, 64*max(4, round(math.sqrt(400.0*N)/64)),
                    0.05+0.25*((i*7) % q)/q))
    return out


BACKEND = {"plain": ("HIP", "RSVD"), "mixed": ("HIP_MIXED", "RSVD"),
           "svd": ("HIP", "SVD"), "rrqr": ("HIP", "RRQR")}


def _problem(case, N, nb, beta, pts, noise=0.0):
    kernel = case["kernel"]
    spatial = kernel not in ("coulomb", "sin", "cos")
    return S.TLRProblem("spatial" if spatial else kernel, N, case["ndim"],
                        nb, symm="S", points=pts, kernel=kernel, beta=beta,
                        nu=case.get("nu", 0.5), noise=noise, wave_k=50.0,
                        diag=1.0)


def _vectors(n, nrhs, seed):
    return np.asfortranarray(np.random.default_rng(seed+77)
                             .standard_normal((n, nrhs)))


class Operator:
    """A device-resident compressed matrix (starsh_hip_tlr)."""

    def __init__(self, M):
        self.T = C.c_void_p()
        assert S.lib().starsh_hip_tlr_new(C.byref(self.T), M) == 0

        self.free = S.lib().starsh_hip_tlr_free

    def __del__(self):
        if self.T:
            self.free(self.T)


def _layout(case):
    """Tiles (i, j) of a product case with their ranks, dense tiles having
    rank -1, and the block sizes: off-diagonal ranks fall with the distance
    from the diagonal, as compression leaves them."""
    N, nb = case["N"], case["nb"]
    size = [min(nb, N-s) for s in range(0, N, nb)]
    tiles = []
    for i in range(len(size)):
        for j in range(i+1 if case["symm"] == "S" else len(size)):
            r = max(3, int(case["rank"]/(1.0+0.08*abs(i-j))))
            tiles.append([i, j, min(r, size[i], size[j])])
    step = max(1, len(tiles)//case["near"]) if case["near"] else 0
    for q in range(case["near"]):
        if q*step < len(tiles):
            tiles[q*step][2] = -1
    return size, tiles


def _factors(case, seed):
    """U, V (graded columns) of the low-rank tiles and the dense tiles, as
    one array and the tiles' offsets into it."""
    size, tiles = _layout(case)
    off, at = [], 0
    for i, j, r in tiles:
        off.append(at)
        at += (size[i]+size[j])*r if r >= 0 else size[i]*size[j]
    data = np.random.default_rng(seed).random(at)
    data -= 0.5
    data = torch.from_numpy(data)
    for (i, j, r), o in zip(tiles, off):
        if r >= 0:
            m, n = size[i], size[j]
            data[o:o+m*r] *= math.sqrt(12.0/m)
            v = data[o+m*r:o+(m+n)*r].view(r, n)
            v *= torch.pow(10.0, torch.linspace(0, -7, r,
                                                dtype=torch.float64))[:, None]
    return size, tiles, off, data


def _operator(case, seed):
    """The operator of a product case: the tile lists and factors as a
    caller that has them from elsewhere passes them to the library."""
    L = S.lib()
    size, tiles, off, data = _factors(case, seed)
    N, nb = case["N"], case["nb"]
    p = S.TLRProblem("spatial", N, 2, nb, symm=case["symm"], kernel="exp",
                     points=_points("exp", 2, N, seed))
    libc = C.CDLL(None)
    libc.malloc.restype = C.c_void_p

    def ints(v):
        a = (S.STARSH_int*max(1, len(v)))(*v)
        ptr = libc.malloc(C.c_size_t(C.sizeof(a)))
        C.memmove(ptr, a, C.sizeof(a))
        return C.cast(ptr, C.POINTER(S.STARSH_int))

    far = [t for t in tiles if t[2] >= 0]
    near = [t for t in tiles if t[2] < 0]
    F = C.POINTER(S.BLRF)()
    info = L.starsh_blrf_new_from_coo(
        C.byref(F), p.P, C.c_char(case["symm"].encode()), p.C, p.C,
        S.STARSH_int(len(far)), ints([x for t in far for x in t[:2]]),
        S.STARSH_int(len(near)), ints([x for t in near for x in t[:2]]),
        C.c_int(p.F.contents.type))
    assert info == 0, info
    base = data.data_ptr()

    def array(o, rows, cols):
        A = C.POINTER(S.Array)()
        assert L.array_from_buffer(C.byref(A), C.c_int(2),
                                   (C.c_int*2)(rows, cols), C.c_char(b"d"),
                                   C.c_char(b"F"),
                                   C.c_void_p(base+8*o)) == 0
        return A

    PA = C.POINTER(S.Array)
    U, V, D = [], [], []
    for (i, j, r), o in zip(tiles, off):
        m, n = size[i], size[j]
        if r >= 0:
            U.append(array(o, m, r))
            V.append(array(o+m*r, n, r))
        else:
            D.append(array(o, m, n))
    M = S.BLRM()
    M.format = F
    M.far_rank = (C.c_int*max(1, len(far)))(*[t[2] for t in far])
    M.far_U = (PA*max(1, len(U)))(*U)
    M.far_V = (PA*max(1, len(V)))(*V)
    M.near_D = (PA*max(1, len(D)))(*D)
    M.onfly = 0
    return Operator(C.byref(M))


# ---- one pass

def prepare(case, seed):
    kind = case["kind"]
    if kind == "compress":
        fn = S.init(*BACKEND[case["form"]][:1], oversample=case["os"],
                    lrengine=BACKEND[case["form"]][1])
        pts = _points(case["kernel"], case["ndim"], case["N"], seed)
        p = _problem(case, case["N"], case["nb"], case["beta"], pts)
        return dict(case=case, fn=fn, p=p,
                    X=_vectors(case["N"], case["nrhs"], seed))
    if kind == "batch":
        S.init(*BACKEND[case["form"]][:1], oversample=case["os"],
               lrengine=BACKEND[case["form"]][1])
        ps, X = [], []
        for q, (N, nb, beta) in enumerate(_batch_specs(case)):
            pts = _points(case["kernel"], case["ndim"], N, seed*100+q)
            ps.append(_problem(case, N, nb, beta, pts))
            X.append(_vectors(N, case["nrhs"], seed*100+q))
        return dict(case=case, ps=ps, X=X)
    if kind == "product":
        gen = torch.Generator().manual_seed(int(seed)+77)
        X = torch.randn(case["nrhs"], case["N"], dtype=torch.float64,
                        generator=gen).cuda()
        return dict(case=case, op=_operator(case, seed), X=X,
                    Y=torch.zeros_like(X))
    if kind == "cg":
        fn = S.init("HIP", oversample=case["os"])
        pts = _points(case["kernel"], case["ndim"], case["N"], seed)
        p = _problem(case, case["N"], case["nb"], case["beta"], pts,
                     noise=case["noise"])
        assert p.approximate(case["maxrank"], case["tol"], 0, fn) == 0
        B = _vectors(case["N"], case["nrhs"], seed)
        return dict(case=case, p=p, B=B, X0=np.zeros_like(B))
    gen = torch.Generator().manual_seed(int(seed))
    x = torch.rand(case["ndim"], case["N"], dtype=torch.float64,
                   generator=gen).cuda()
    return dict(case=case, x=x, y=torch.empty_like(x),
                order=torch.empty(case["N"], dtype=torch.int64,
                                  device="cuda"))


def _fresh_format(p):
    """The plain tile low-rank format of a problem: a compression rewrites
    it, so a program that compresses again makes a new one."""
    L = S.lib()
    if p.F:
        L.starsh_blrf_free(p.F)
    p.F = C.POINTER(S.BLRF)()
    assert L.starsh_blrf_new_tlr(C.byref(p.F), p.P,
                                 C.c_char(p.symm.encode()), p.C, p.C) == 0


def _ranks(p):
    """Ranks of the lower triangle's tiles, -1 for the dense ones."""
    M = p.M.contents
    F = M.format.contents
    nfar, nb = F.nblocks_far, F.nbrows
    out = np.full((nb, nb), -1, dtype=np.int64)
    if nfar > 0:
        ij = np.ctypeslib.as_array(F.block_far, (nfar, 2))
        out[ij[:, 0], ij[:, 1]] = np.ctypeslib.as_array(M.far_rank, (nfar,))
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "compress":
        p = state["p"]
        _fresh_format(p)
        assert p.approximate(case["maxrank"], case["tol"], 0,
                             state["fn"]) == 0
        out = {"ranks": _ranks(p), "y": p.dmml(state["X"])}
        p.free_matrix()
        return out
    if kind == "batch":
        ps = state["ps"]
        for p in ps:
            _fresh_format(p)
        assert S.approximate_batch(ps, case["maxrank"], case["tol"]) == 0
        out = {"ranks": [_ranks(p) for p in ps],
               "y": [p.dmml(X) for p, X in zip(ps, state["X"])]}
        for p in ps:
            p.free_matrix()
        return out
    if kind == "product":
        N = case["N"]
        assert S.lib().starsh_hip_tlr_dmml(
            state["op"].T, C.c_int(case["nrhs"]), C.c_double(1.0),
            C.c_void_p(state["X"].data_ptr()), C.c_int(N), C.c_double(0.0),
            C.c_void_p(state["Y"].data_ptr()), C.c_int(N)) == 0
        return {"y": state["Y"]}
    if kind == "cg":
        it, X = state["p"].cg(state["B"], state["X0"], 1e-11)
        assert it >= 0
        return {"x": X}
    x = state["x"]
    assert S.lib().starsh_hip_zsort(
        C.c_void_p(x.data_ptr()), C.c_int64(case["N"]),
        C.c_int(case["ndim"]), C.c_void_p(state["y"].data_ptr()),
        C.c_void_p(state["order"].data_ptr())) == 0
    return {"y": state["y"], "order": state["order"]}


# ---- what a pass cannot do without

# average rank of the compressed tiles by kernel (measured on the listed
# sizes): enough for the bytes of the factors
RANK = {"sqrexp": 20, "exp": 60, "matern": 140, "coulomb": 56, "sin": 56}


def _tlr_work(N, nb, rank, os, nrhs, ndim):
    nt = -(-N//nb)
    area = 0.5*N*(N+nb)
    # random sketch and projection of width rank + oversample, an
    # orthogonalisation, the factors written, then the product
    width = rank+os
    fac = nt*(nt+1)*nb*rank
    return {"bytes": 8.0*(ndim*N+2*nrhs*N+2*fac),
            "flops": 4.0*area*width+8.0*area*ndim+4.0*fac*width +
            8.0*fac*nrhs}


def work(case):
    kind = case["kind"]
    if kind == "compress":
        return _tlr_work(case["N"], case["nb"], min(RANK[case["kernel"]],
                                                    case["nb"]//4),
                         case["os"], case["nrhs"], case["ndim"])
    if kind == "batch":
        w = [_tlr_work(N, nb, min(RANK[case["kernel"]], nb//4), case["os"],
                       case["nrhs"], case["ndim"])
             for N, nb, _ in _batch_specs(case)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    if kind == "product":
        size, tiles = _layout(case)
        cells = twice = 0
        for i, j, r in tiles:
            c = (size[i]+size[j])*r if r >= 0 else size[i]*size[j]
            cells += c
            twice += 2*c if case["symm"] == "S" and i != j else c
        return {"bytes": 8.0*(cells+2*case["N"]*case["nrhs"]),
                "flops": 2.0*twice*case["nrhs"]}
    if kind == "cg":
        # the factors uploaded once and read once; a product per iteration,
        # of which a well-conditioned system needs a few tens
        w = _tlr_work(case["N"], case["nb"], RANK[case["kernel"]],
                      case["os"], case["nrhs"], case["ndim"])
        return {"bytes": w["bytes"], "flops": 50*w["bytes"]/4*case["nrhs"]}
    return {"bytes": 8.0*case["N"]*(2*case["ndim"]+1), "flops": 0.0}


# ---- the same outputs in plain 64-bit torch

def _dense_rows(case, pts, rows, beta, noise):
    """Rows `rows` of the dense kernel matrix."""
    x = pts[:, rows]
    d2 = torch.zeros(x.shape[1], pts.shape[1], dtype=torch.float64,
                     device=pts.device)
    for d in range(pts.shape[0]):
        d2 += (x[d][:, None]-pts[d][None, :])**2
    kernel = case["kernel"]
    if kernel == "sqrexp":
        A = torch.exp(-d2/(2.0*beta*beta))
    elif kernel == "exp":
        A = torch.exp(-torch.sqrt(d2)/beta)
    elif kernel == "matern":
        nu = case["nu"]
        t = torch.sqrt(d2)*(math.sqrt(2.0*nu)/beta)
        poly = {0.5: 1.0, 1.5: 1.0+t, 2.5: 1.0+t+t*t/3.0}[nu]
        A = poly*torch.exp(-t)
    else:
        r = torch.sqrt(d2)
        zero = r == 0
        A = (1.0 if kernel == "coulomb" else torch.sin(50.0*r))/torch.where(
            zero, torch.ones_like(r), r)
        A[zero] = 0.0 if kernel == "coulomb" else 1.0
    if noise:
        A[d2 == 0] += noise
    return A


def _dense_apply(case, pts, beta, X, noise=0.0):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p = torch.from_numpy(pts).to(dev)
    X = torch.from_numpy(np.ascontiguousarray(X)).to(dev)
    n = p.shape[1]
    out = torch.empty_like(X)
    step = max(1, 100000000//n)
    for a in range(0, n, step):
        rows = slice(a, min(n, a+step))
        A = _dense_rows(case, p, rows, beta, noise)
        for q in range(X.shape[1]):
            out[rows, q] = torch.mv(A, X[:, q].contiguous())
    return out.cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "compress":
        pts = _points(case["kernel"], case["ndim"], case["N"], seed)
        return {"ranks": None,
                "y": _dense_apply(case, pts, case["beta"],
                                  _vectors(case["N"], case["nrhs"], seed))}
    if kind == "batch":
        y = []
        for q, (N, nb, beta) in enumerate(_batch_specs(case)):
            pts = _points(case["kernel"], case["ndim"], N, seed*100+q)
            y.append(_dense_apply(case, pts, beta,
                                  _vectors(N, case["nrhs"], seed*100+q)))
        return {"ranks": None, "y": y}
    if kind == "product":
        size, tiles, off, data = _factors(case, seed)
        start = np.concatenate([[0], np.cumsum(size)])
        gen = torch.Generator().manual_seed(int(seed)+77)
        X = torch.randn(case["nrhs"], case["N"], dtype=torch.float64,
                        generator=gen)
        Y = torch.zeros_like(X)
        for (i, j, r), o in zip(tiles, off):
            m, n = size[i], size[j]
            ri = slice(int(start[i]), int(start[i+1]))
            rj = slice(int(start[j]), int(start[j+1]))
            both = case["symm"] == "S" and i != j
            if r >= 0:
                U = data[o:o+m*r].view(r, m)
                V = data[o+m*r:o+(m+n)*r].view(r, n)
                Y[:, ri] += (X[:, rj] @ V.T.contiguous()) @ U
                if both:
                    Y[:, rj] += (X[:, ri] @ U.T.contiguous()) @ V
            else:
                D = data[o:o+m*n].view(n, m)
                Y[:, ri] += X[:, rj] @ D
                if both:
                    Y[:, rj] += X[:, ri] @ D.T.contiguous()
        return {"y": Y}
    if kind == "cg":
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        pts = torch.from_numpy(_points(case["kernel"], case["ndim"],
                                       case["N"], seed)).to(dev)
        A = _dense_rows(case, pts, slice(0, case["N"]), case["beta"],
                        case["noise"])
        B = torch.from_numpy(np.ascontiguousarray(
            _vectors(case["N"], case["nrhs"], seed)))
        return {"x": torch.linalg.solve(A.cpu(), B)}
    gen = torch.Generator().manual_seed(int(seed))
    x = torch.rand(case["ndim"], case["N"], dtype=torch.float64,
                   generator=gen).numpy()
    return {"y": _morton(x), "order": None}
