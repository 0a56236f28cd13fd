"""Block Gram-Schmidt (csrc/hip/qr.hip) at the edges of its blocks (64, then
32 columns), panels (8 and 4), 16-row fragments, 128-row strips and register
classes (1024, 2048 rows): tiles of a prescribed range, whose dimension lies
below, at and above the sketch width, give the spectrum they were built from
and orthonormal factors."""
import numpy as np
import pytest

import starsh_hip as S
from test_gpu_core_block import _lowrank, _tile

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _check(tiles, spectra, panel):
    import ctypes as C
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
