"""Gram-Schmidt panels as one captured hipGraph (starsh_hip_set_option
"qr_graph" 1) against the default host-launched panels: the same ranks and
the same error, bit for bit, in both forms, on a first call (capture) and a
second one (replay of the kept graph)."""
import ctypes as C

import pytest

import starsh_hip as S

pytestmark = pytest.mark.gpu


def _opt(name, value):
    assert S.lib().starsh_hip_set_option(name.encode(),
                                         C.c_double(value)) == 0, name


@pytest.mark.parametrize("backend", ["HIP", "HIP_MIXED"])
def test_graph_panels_match_host_launches(backend):
    print(f"case: qr_graph {backend} 2D sqexp N=12800 nb=1600", flush=True)
    res = {}
    try:
        for g in (0, 1):
            _opt("qr_graph", g)
            fn = S.init(backend, oversample=16)
            out = []
            for _ in range(2):
                p = S.TLRProblem("spatial", 12800, 2, 1600, symm="S", seed=1,
                                 kernel="sqrexp", beta=0.1)
                assert p.approximate(400, 1e-7, 0, fn) == 0
                out.append((p.ranks().tolist(), p.dfe()))
                p.free_matrix()
            res[g] = out
    finally:
        _opt("qr_graph", 0)
    for (r0, e0), (r1, e1) in zip(res[0], res[1]):
        assert r0 == r1
        assert e0 == e1


def test_sketch_statistics_count_what_was_computed():
    """N=3300 in tiles of 800, 800, 800, 800, 100: with the panels launched
    by the host the chunks past a tile's range are not computed (128 columns
    of 416 for these tiles), with a captured graph all are."""
    print("case: qr_graph sketch statistics", flush=True)
    size = [800]*4+[100]
    pairs = [(size[i], size[j]) for i in range(5) for j in range(i+1)]
    st = {}
    for g in (0, 1):
        _opt("qr_graph", g)
        try:
            fn = S.init("HIP", oversample=16)
            p = S.TLRProblem("spatial", 3300, 2, 800, symm="S", seed=1,
                             kernel="sqrexp", beta=0.5)
            assert p.approximate(400, 1e-7, 0, fn) == 0
            st[g] = S.stats()
            p.free_matrix()
        finally:
            _opt("qr_graph", 0)
    full = sum(2.0*m*n*min(416, m, n) for m, n in pairs)
    first = sum(2.0*m*n*min(128, m, n) for m, n in pairs)
    assert st[1].sketch_bytes_or_flops == full
    assert st[0].sketch_bytes_or_flops == first
    assert st[1].dominant_kernel_launches == 3       # 128, 256, 32 columns
    # the block after the last one that had work may have been queued before
    # the host saw that none was left
    assert 1 <= st[0].dominant_kernel_launches <= 2
