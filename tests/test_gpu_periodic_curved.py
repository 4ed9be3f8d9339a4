"""A periodic pair of a straight and a curved edge: viscous traces stored along the normal would be along
different normals on the two sides, also where the first nodes' happen to be opposite."""
import numpy as np
import pytest

from horses2d_amd import cases as C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bend", [0.0, 0.3])
@pytest.mark.parametrize("N", [3, 5])
@pytest.mark.parametrize("viscous", ["br1", "ip"])
def test_straight_against_curved_matches_oracle(N, viscous, bend):
    """The left edges are cubics, the right ones straight (pairs are matched by one coordinate of their ends);
    at bend 0 the cubic's slope vanishes at the edge's first node.  FP64 bar: 1e-12 of the max-norm after
    three RK3 steps."""
    from horses2d_amd import gpu
    from oracle.oracle import Oracle
    wall = C.Zone(C.BC_VISCOUSWALL)
    nx, ny = 6, 5
    mesh = C.channel(nx, ny, 2.0, 1.0, [wall, C.Zone(C.BC_PERIODIC, direction=1, partner=4), wall,
                                        C.Zone(C.BC_PERIODIC, direction=1, partner=2)])
    s1 = 0.5 + 0.5 * np.polynomial.legendre.leggauss(N + 1)[0][0]
    c = s1 + s1 * (1.0 - s1) / (1.0 - 2.0 * s1) + bend
    s = 0.5 - 0.5 * np.cos(np.pi * np.arange(4) / 3.0)
    edges, xy = [], []
    for j in range(ny):
        a, b = mesh.points[j], mesh.points[j + 1]
        x = a[None] + s[:, None] * (b - a)[None]
        x[:, 0] += 0.15 * s * (1.0 - s) * (s - c)
        edges.append((j, j + 1))
        xy.append(x)
    mesh.cedges, mesh.cxy = np.array(edges, np.int32), np.array(xy)
    case = C.Case("bent", mesh, np.full(mesh.K, N, np.int32), 0.3, 200.0, 0.72, True, riemann="roe", viscous=viscous,
                  cfl=0.05, ic=C.isentropic_vortex(0.3, 1.0, 1.0, 0.5))
    orc = Oracle(case)
    Q0 = case.initial_state(orc.coords())
    orc.set_state(Q0)
    dt = orc.estimate_dt(case.dt_max, case.cfl)
    dg = gpu.DGSEM(case, "fp64", apply_ic=False)
    dg.upload(Q0)
    for _ in range(3):
        orc.step(0.0, dt, case.scheme)
        dg.rk_step(0.0, dt)
    ref = orc.state()
    assert np.max(np.abs(dg.state() - ref)) <= 1e-12 * np.max(np.abs(ref))
