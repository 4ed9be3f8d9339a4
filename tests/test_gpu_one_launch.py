"""Meshes of several orders: the captured step's passes over all orders in one launch give the bits of the
separate launches (steps without a graph), in every form, at the smallest and largest orders it takes and
beyond (orders 11 and 12 keep separate launches), with few workgroups (atomic residual) and many, after
another upload and after another boundary state."""
import numpy as np
import pytest

from horses2d_amd import cases as C

pytestmark = pytest.mark.gpu


def _case(nx, ny, orders, viscous, scheme, seed=5):
    q = tuple(C.freestream_state(0.3))
    far, wall = C.Zone(C.BC_FARFIELD, q=q), C.Zone(C.BC_VISCOUSWALL, isothermal=1, Tw=1.0)
    zones = [far if viscous == "none" else wall, far, far, far]
    mesh = C.channel(nx, ny, 3.0, 2.0, zones, skew=0.4)
    N = np.random.Generator(np.random.PCG64(seed)).choice(orders, mesh.K).astype(np.int32)
    return C.Case("orders", mesh, N, 0.3, 0.0 if viscous == "none" else 300.0, 0.72, viscous != "none", riemann="roe",
                  viscous=viscous, ip_method="sipg", sigma0=1.0, cfl=0.02, scheme=scheme,
                  ic=C.isentropic_vortex(0.3, 1.0, 1.4, 0.9))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nx, ny, orders, viscous, scheme", [
    (3, 2, [1, 2], "none", "euler"), (9, 7, [2, 4, 7], "none", "rk5"), (9, 7, [1, 10], "br1", "rk3"),
    (40, 41, [3, 5], "none", "rk3"), (9, 7, [3, 6, 8], "br1", "rk5"), (9, 7, [2, 5, 7], "ip", "rk3"),
    (36, 31, [7, 8], "ip", "rk3"), (5, 4, [4, 11, 12], "none", "rk3")])
def test_graph_steps_equal_direct_steps(nx, ny, orders, viscous, scheme, precision):
    from horses2d_amd import gpu
    case = _case(nx, ny, orders, viscous, scheme)
    a, b = gpu.DGSEM(case, precision), gpu.DGSEM(case, precision)
    b.set_graph(False)
    Q0 = a.state()
    dt = a.estimate_dt(case.dt_max, case.cfl)
    half = Q0.reshape(-1, 4) * np.array([1.0, 1.0, 1.0, 1.1])

    def same(steps):
        for k in range(steps):
            for s in (a, b):
                s.rk_step(0.0, dt * (1.0 + 0.1 * k))
            np.testing.assert_array_equal(a.residuals(), b.residuals())
        np.testing.assert_array_equal(a.state(), b.state())
        assert np.all(np.isfinite(a.state()))
    same(3)
    for s in (a, b):
        s.upload(half.reshape(-1))
    same(2)
    for s in (a, b):
        n = len(s.boundary_nodes(2))
        s.set_boundary_state(2, np.tile(C.freestream_state(0.31), (n, 1)))
    same(2)
