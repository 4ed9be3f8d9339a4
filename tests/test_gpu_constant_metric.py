"""Elements of constant metric (parallelograms) in the FP64 viscous forms: the gradient's traces come
from the reference derivatives along and across the face, the nodal gradient takes the metric out of
its sums.

A sheared channel (near the origin and moved far from it, where the mesh's rounding is larger) and the
same with one vertex moved, which takes the general kernels: all match the oracle within the FP64 bar
(1e-12 of the max-norm after three RK3 steps)."""
import numpy as np
import pytest

from horses2d_amd import cases as C

pytestmark = pytest.mark.gpu


def _channel(N, viscous, kind):
    q = C.freestream_state(0.3)
    far = C.Zone(C.BC_FARFIELD, q=tuple(q))
    zones = [C.Zone(C.BC_VISCOUSWALL), far, C.Zone(C.BC_VISCOUSWALL, isothermal=1, wall_velocity=(0.1, 0.0)), far]
    mesh = C.channel(7, 5, 2.0, 1.0, zones)
    if kind == "bent":
        mesh.points[6 * 3 + 2] += [0.03, -0.02]
    mesh.points[:] = mesh.points @ np.array([[1.0, -0.2], [0.3, 0.9]])
    if kind == "far":
        mesh.points[:] += [40.0, -30.0]
    centre = (41.0, -30.0) if kind == "far" else (1.0, 0.2)
    return C.Case(kind, mesh, np.full(mesh.K, N, np.int32), 0.3, 200.0, 0.72, True, riemann="roe", viscous=viscous,
                  cfl=0.05, ic=C.isentropic_vortex(0.3, 1.0, *centre))


@pytest.mark.parametrize("kind", ["shear", "far", "bent"])
@pytest.mark.parametrize("N", [1, 2, 3, 5, 6, 7, 10, 12])
@pytest.mark.parametrize("viscous", ["br1", "ip"])
def test_constant_metric_matches_oracle(N, viscous, kind):
    from horses2d_amd import gpu
    from oracle.oracle import Oracle
    case = _channel(N, viscous, kind)
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


@pytest.mark.parametrize("slant", [0.0, 0.15])
@pytest.mark.parametrize("N", [2, 5, 6])
@pytest.mark.parametrize("viscous", ["br1", "ip"])
def test_periodic_viscous_trace_matches_oracle(N, viscous, slant):
    """Viscous traces stored along the normal, and per direction where a periodic pair (matched by one
    coordinate of its ends) is not parallel: both within the FP64 bar."""
    from horses2d_amd import gpu
    from oracle.oracle import Oracle
    wall = C.Zone(C.BC_VISCOUSWALL)
    mesh = C.channel(6, 5, 2.0, 1.0, [wall, C.Zone(C.BC_PERIODIC, direction=1, partner=4), wall,
                                      C.Zone(C.BC_PERIODIC, direction=1, partner=2)])
    mesh.points[:, 0] *= 1.0 + slant * mesh.points[:, 1]
    case = C.Case("slanted", mesh, np.full(mesh.K, N, np.int32), 0.3, 200.0, 0.72, True, riemann="roe",
                  viscous=viscous, cfl=0.05, ic=C.isentropic_vortex(0.3, 1.0, 1.0, 0.5))
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
