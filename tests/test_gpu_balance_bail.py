"""balanceOctree of complete octrees that lack so many splits that the levels are
rebuilt after all (a fine plane against coarse leaves, a line), and of octrees
whose leaves lie on two neighbouring levels and lack none: the same octants as
level by level (which any other order of the leaves takes), and no multiple of
its time."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _line(n, seed=1):
    t = np.random.default_rng(seed).random((n, 1))
    return np.array([0.1, 0.2, 0.15]) + t * np.array([0.7, 0.5, 0.6])


def _plane(n, seed=1):
    p = np.random.default_rng(seed).random((n, 3))
    p[:, 0] = 0.5 - 1e-3 * p[:, 0]
    return p


def _other_order(dgx, ou, curve=0):
    return dgx.import_treenodes(np.ascontiguousarray(ou.treenodes()[::-1]), ou.max_depth, curve, sort=False)


@pytest.mark.parametrize("kind,n", [("line", 300), ("line", 5000), ("line", 40000), ("plane", 5000), ("plane", 60000)])
@pytest.mark.parametrize("curve", [0, 1])
def test_same_octants(dgx, oracle, kind, n, curve):
    ou = dgx.points2octree({"line": _line, "plane": _plane}[kind](n), 30, 1, curve)
    fast, slow = dgx.balance_octree(ou), dgx.balance_octree(_other_order(dgx, ou, curve))
    t = fast.treenodes()
    assert np.array_equal(t, slow.treenodes()) and fast.stats() == slow.stats()
    if len(t) < 200000:
        oracle.set_ordering(curve == 0)
        try:
            assert np.array_equal(t, oracle.balance(ou.treenodes()))
        finally:
            oracle.set_ordering(True)


# 40^3 points: cells of levels 5 and 6 in every workgroup of leaves; 16^3: one level
@pytest.mark.parametrize("k", [16, 40])
@pytest.mark.parametrize("curve", [0, 1])
def test_two_neighbouring_levels(dgx, oracle, k, curve):
    a = (np.arange(k) + 0.5) / k
    ou = dgx.points2octree(np.stack(np.meshgrid(a, a, a), -1).reshape(-1, 3), 30, 1, curve)
    t = ou.treenodes()
    assert np.ptp(t[:, 3]) <= 1
    ob = dgx.balance_octree(ou)
    assert np.array_equal(ob.treenodes(), t) and ob.stats()[:2] == [0, 0]
    # one leaf far finer than the rest: all of them count again
    pts = np.concatenate([np.stack(np.meshgrid(a, a, a), -1).reshape(-1, 3), [[0.3, 0.3, 0.3], [0.3 + 2.0 ** -12, 0.3, 0.3]]])
    ou = dgx.points2octree(pts, 30, 1, curve)
    oracle.set_ordering(curve == 0)
    try:
        assert np.array_equal(dgx.balance_octree(ou).treenodes(), oracle.balance(ou.treenodes()))
    finally:
        oracle.set_ordering(True)


@pytest.mark.parametrize("kind,n", [("line", 300000), ("plane", 1000000)])
def test_time_beside_level_by_level(dgx, kind, n):
    """Giving up costs little: within 1.6 times the level-by-level step (2.5 to 3
    when every workgroup went to its end first)."""
    ou = dgx.points2octree({"line": _line, "plane": _plane}[kind](n), 30, 1)
    other = _other_order(dgx, ou)

    def best(o):
        t = []
        for _ in range(6):
            dgx.synchronize()
            t0 = time.perf_counter()
            dgx.balance_octree(o)
            dgx.synchronize()
            t.append(time.perf_counter() - t0)
        return min(t[1:])

    a, b = best(ou), best(other)
    print(f"{kind} {len(ou)} leaves: {a * 1e6:.0f} us, level by level {b * 1e6:.0f} us", flush=True)
    assert a < 1.6 * b
