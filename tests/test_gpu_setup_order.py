"""balanceOctree returns a finished octree, which the set-up of a hierarchy reads
on a second stream: the library's stream is idle after the call, and every
level's DA of an overlapped set-up is that of the level's octree built by
itself, also where the helper is idle when a level is handed to it (hierarchies
that coarsen past the requested levels)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# octrees that lack splits, with one and with four leaves per thread, and one that lacks none
@pytest.mark.parametrize("dist,n,m,again", [(2, 30000, 1, False), (2, 400000, 1, False), (2, 400000, 1, True)])
def test_balance_is_done_when_it_returns(dgx, dist, n, m, again):
    ou = dgx.points2octree(dgx.gen_points(dist, 17, n, n_gauss=4, lo=0.2, hi=0.8, sig_lo=0.02), 30, m)
    if again:
        ou = dgx.balance_octree(ou)
    query = dgx.load_library().hipStreamQuery  # of the HIP runtime that the library is linked with
    query.argtypes = [ctypes.c_void_p]
    for _ in range(20):
        ob = dgx.balance_octree(ou)
        assert query(dgx.stream()) == 0
        ob.free()


@pytest.mark.parametrize("n,nlevels", [(60000, 1), (60000, 2), (20000, 5)])
@pytest.mark.parametrize("curve", [0, 1])
def test_levels_of_an_overlapped_set_up(dgx, oracle, n, nlevels, curve):
    pts = dgx.gen_points(2, 5 + n, n, n_gauss=4, lo=0.2, hi=0.8, sig_lo=0.02)
    oracle.set_ordering(curve == 0)
    try:
        ob = dgx.balance_octree(dgx.points2octree(pts, 30, 1, curve))
        t = ob.treenodes()
        for _ in range(3):  # later rounds find the helper's stream and the blocks of the first
            mg = dgx.MG(ob, nlevels=nlevels)
            assert nlevels > 2 or mg.nlevels > nlevels
            level = t
            for k in range(mg.nlevels):
                got, want = mg.level_da(k).maps(), dgx.DA(dgx.import_treenodes(level, 30, curve)).maps()
                for a, b in zip(got, want):
                    assert np.array_equal(a, b), k
                level = oracle.balance(oracle.coarsen(level))
            mg.free()
    finally:
        oracle.set_ordering(True)
