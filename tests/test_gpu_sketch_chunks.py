"""The plain form's sketch in chunks of columns (csrc/hip/gen_gemm.hip):
widths on either side of every rule, with tiles that exhaust their range in
the first chunk, in a later one and not at all, against forced column blocks
(whose chunks lie elsewhere): the same ranks and products."""
import ctypes as C
import os

import numpy as np
import pytest

import starsh_hip as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _option(name, value):
    assert S.lib().starsh_hip_set_option(name, C.c_double(value)) == 0


@pytest.mark.parametrize("kernel,beta", [("sqrexp", 0.5), ("sqrexp", 0.05),
                                         ("exp", 0.1)])
@pytest.mark.parametrize("width", [64, 65, 128, 129, 256, 257, 330, 416, 470,
                                   520, 600])
def test_chunks(kernel, beta, width):
    N, nb = 1817, 607
    fn = S.init("HIP", oversample=10)
    rng = np.random.default_rng(5)
    pts = rng.random((2, N))
    X = rng.standard_normal((N, 2))
    got = []
    for bn in (0, 64, 256):
        p = S.TLRProblem("spatial", N, 2, nb, kernel=kernel, beta=beta,
                         points=pts)
        _option(b"gemm_bn", bn)
        try:
            assert p.approximate(width-10, 1e-9, 0, fn) == 0
        finally:
            _option(b"gemm_bn", 0)
        far = [(i, j) for i, j in p.tiles()]
        got.append((dict(zip(far, p.ranks().tolist())), p.dmml(X)))
        p.free_matrix()
    print(kernel, beta, width, sorted(got[0][0].values())[-3:], flush=True)
    for ranks, y in got[1:]:
        assert ranks == got[0][0]
        # the same columns in other blocks: rounding only, and what the rank
        # rule leaves out is the same to first order
        assert np.max(np.abs(y-got[0][1])) <= 1e-12*np.max(np.abs(y))


def test_dump_holds_every_column(tmp_path):
    """STARSH_HIP_DEBUG_DUMP writes the whole sketch of tile (0, 0), Y = A
    Omega, also the columns past its range that are otherwise never
    computed."""
    print("case: dump of the sketch, 2D sqexp N=2400 nb=800", flush=True)
    os.environ["STARSH_HIP_DEBUG_DUMP"] = str(tmp_path)
    try:
        fn = S.init("HIP", oversample=16)
        p = S.TLRProblem("spatial", 2400, 2, 800, symm="S", seed=4,
                         kernel="sqrexp", beta=0.1)
        assert p.approximate(400, 1e-7, 0, fn) == 0
    finally:
        del os.environ["STARSH_HIP_DEBUG_DUMP"]
    Y = np.fromfile(tmp_path/"Y.bin").reshape(416, 800).T
    st, sz = p.cluster_ranges()
    rows = np.arange(st[0], st[0]+sz[0])
    A = O.kernel_block(O.kernel("sqrexp", 2, beta=0.1), p.points(),
                       p.points(), rows, rows)
    om = O.omega(800, 416)
    # rounding of 800 products and of the entries (a few ulp)
    bound = 800*np.finfo(float).eps*(np.abs(A) @ np.abs(om))
    assert np.all(np.abs(Y-A @ om) <= bound)
    p.free_matrix()
