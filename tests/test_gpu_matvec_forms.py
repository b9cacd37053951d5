"""Every form of the matvec that a V-cycle uses (both precisions, Dirichlet rows,
the Jacobi sweep in place, the residual) on DAs of at most 256 element blocks,
one per workgroup, and of more, against the kernel for large blocks: the node
sums are the same integers and the updates the same expressions, so single
products and whole solves agree to the last bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,curve", [(60, 1, 0), (3000, 1, 1), (17000, 1, 0), (60000, 1, 1)])
def test_forms_agree(dgx, n, m, curve, monkeypatch):
    ob = dgx.balance_octree(dgx.points2octree(dgx.gen_points(0, n, n), 30, m, curve))
    mg = dgx.MG(ob, nlevels=3)
    nn = mg.n_nodes
    blocks = [-(-e // 512) for e in mg.level_octants]
    print(f"n={n} blocks {blocks}", flush=True)
    assert blocks[-1] <= 256
    rng = np.random.default_rng(n)
    x = rng.standard_normal(nn)
    got = []
    for blocked in ("0", "1"):
        monkeypatch.setenv("DGX_MATVEC_BLOCKED", blocked)
        out = [mg.da.matvec_host(x), mg.da.matvec_dirichlet_host(x)]
        x32, y32 = dgx.DeviceArray.from_host(x.astype(np.float32)), dgx.DeviceArray((nn,), np.float32)
        mg.da.matvec(x32, y32)
        out.append(y32.to_host())
        b = dgx.DeviceArray((nn,), np.float64)
        mg.rhs(dgx.DeviceArray.from_host(x), b)
        for fp32 in (False, True):
            u = dgx.DeviceArray((nn,), np.float64)
            mg.solve(b, u, fp32=fp32, maxit=3, rtol=1e-12, graph=False)
            out.append(u.to_host())
        got.append(out)
    for a, c in zip(*got):
        assert np.array_equal(a, c)
    mg.free()
