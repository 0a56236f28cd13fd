"""Block Gram-Schmidt (csrc/hip/qr.hip) at the edges of its blocks (64, then
32 columns), panels (8 and 4), 16-row fragments, 128-row strips and register
classes (1024, 2048 rows): tiles of a prescribed range, whose dimension lies
below, at and above the sketch width, give the spectrum they were built from
and orthonormal factors."""
import ctypes as C

import numpy as np
import pytest

import starsh_hip as S
from test_gpu_core_block import _lowrank, _tile

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _check(tiles, spectra, panel):
    L = S.lib()
    assert L.starsh_hip_set_option(b"qr_panel", C.c_double(panel)) == 0
    try:
        got = _lowrank(1, tiles, 160, 16, 1e-2, True)
    finally:
        assert L.starsh_hip_set_option(b"qr_panel", C.c_double(0)) == 0
    for (r, u, v, sv), A, s in zip(got, tiles, spectra):
        k = max(len(s), 1)
        # rounding of sketch, projection and rotations, each a few units of
        # k eps of the largest singular value
        assert np.max(np.abs(sv[:k]-s)) <= 20*k*EPS*s[0], (A.shape, k)
        if r > 0:
            g = u.T @ u
            assert np.max(np.abs(g-np.eye(r))) <= 100*k*EPS, (A.shape, k)


@pytest.mark.parametrize("panel", [0, 4])
def test_widths(panel):
    tiles, spectra = [], []
    for q, p in enumerate([1, 2, 3, 4, 5, 8, 11, 16, 31, 32, 33, 60, 62, 63,
                           64, 65, 67, 68, 95, 96, 97, 100, 127, 128, 129]):
        s = 1.0/(1.0+np.arange(p))**1.5
        # the range within the tile, and the tile's smaller side equal to it
        for m, n in ((p+37, p+90), (p, p+3)):
            tiles.append(_tile(m, n, s, 100+q))
            spectra.append(s)
    print(len(tiles), "tiles, panel", panel, flush=True)
    _check(tiles, spectra, panel)


@pytest.mark.parametrize("rows", [15, 17, 127, 129, 255, 1023, 1024, 1025,
                                  2047, 2048, 2049, 4096])
def test_rows(rows):
    tiles, spectra = [], []
    for q, p in enumerate([7, 70, 101]):
        p = min(p, rows)
        s = 0.93**np.arange(p)
        tiles += [_tile(rows, p+150, s, q), _tile(p+150, rows, s, 10+q)]
        spectra += [s, s]
    print("rows", rows, flush=True)
    _check(tiles, spectra, 0)


def _free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert S.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_workspace_of_tiles_of_unlike_widths():
    """2080 tiles of 64 with a sketch 20 wide and 3 tiles of 1100 with one
    1010 wide in one batch: the device memory kept afterwards stays within
    the budget (workspace_gb) and the rounding of the pools, whatever the
    widest tile of the batch is."""
    L = S.lib()
    budget = 0.45*2**30
    rng = np.random.default_rng(0)
    S.init("HIP", oversample=10)

    def problems():
        return [S.TLRProblem("spatial", N, 2, nb, kernel="exp", beta=0.1,
                             points=rng.random((2, N)))
                for N, nb in ((4096, 64), (3300, 1100))]
    assert L.starsh_hip_set_option(b"workspace_gb",
                                   C.c_double(budget/2**30)) == 0
    try:
        # code objects, streams and pinned memory first
        assert S.approximate_batch(problems()[:1], [10], 1e-3) == 0
        assert L.starsh_hip_set_option(b"release_workspace",
                                       C.c_double(0)) == 0
        before = _free_bytes()
        ps = problems()
        assert S.approximate_batch(ps, [10, 1000], 1e-3) == 0
        used = before-_free_bytes()
        print("used MiB", used/2**20, "tiles", [len(p.tiles()) for p in ps],
              flush=True)
        for p in ps:
            p.free_matrix()
    finally:
        assert L.starsh_hip_set_option(b"workspace_gb", C.c_double(96)) == 0
        assert L.starsh_hip_set_option(b"release_workspace",
                                       C.c_double(0)) == 0
    # five pools of 64 MiB units at most
    assert used <= budget+5*2**26
