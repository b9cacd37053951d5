"""The coarse solver's analysis in a hierarchy, whose matrix graph is built on the
device, against the host analysis of the oracle's element maps: the same graph
in the same order gives the same interior nodes, fronts, tree and sizes."""
import numpy as np
import pytest

from test_direct_plan import element_data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,curve", [(40, 1, 0), (900, 1, 1), (9000, 1, 0), (9000, 1, 1), (30000, 8, 0)])
def test_device_graph_gives_the_host_plan(dgx, oracle, n, m, curve):
    pts = dgx.gen_points(1, 40 + n, n)
    oracle.set_ordering(curve == 0)
    try:
        conn, cn, meta, bd, xyz = element_data(oracle, pts, m)
    finally:
        oracle.set_ordering(True)
    P = dgx.direct_plan(conn, meta, bd, xyz, leaf=128, dense=4096)  # as library hierarchies take them
    mg = dgx.MG(dgx.balance_octree(dgx.points2octree(pts, 30, m, curve)), nlevels=1)
    assert mg.nlevels == 1
    want = {"interior": P["interior"], "fronts": P["fronts"], "tree_levels": P["levels"], "max_front": P["max_m"],
            "max_separator": P["max_s"], "front_entries": P["entries"]}
    print(want, flush=True)
    assert mg.coarse == want and (n < 9000 or P["fronts"] > 8)
    mg.free()
