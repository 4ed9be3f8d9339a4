"""The metric stored per line of nodes (straight-sided elements, FP64 form).

A mesh of general straight quads takes it, and one with curved edges does not; both match the oracle
within the FP64 bar (1e-12 of the max-norm after three RK3 steps; the stored lines and the Jacobian
formed from them are the mesh builder's own bits)."""
import numpy as np
import pytest

from horses2d_amd import cases as C

pytestmark = pytest.mark.gpu


def _channel(N, viscous):
    q = C.freestream_state(0.3)
    far = C.Zone(C.BC_FARFIELD, q=tuple(q))
    mesh = C.channel(7, 5, 2.0, 1.0, [far, far, far, far], skew=0.6)
    return C.Case("skewed", mesh, np.full(mesh.K, N, np.int32), 0.3, 0.0 if viscous == "none" else 200.0, 0.72,
                  viscous != "none", riemann="roe", viscous=viscous, cfl=0.05,
                  ic=C.isentropic_vortex(0.3, 1.0, 1.0, 0.5))


@pytest.mark.parametrize("N", [1, 3, 6, 7, 12])
@pytest.mark.parametrize("viscous", ["none", "br1", "ip", "curved"])
def test_line_metric_matches_oracle(N, viscous):
    from horses2d_amd import gpu
    from oracle.oracle import Oracle
    case = C.ns_cylinder_case(3, 12, N=max(N, 3)) if viscous == "curved" else _channel(N, viscous)
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
