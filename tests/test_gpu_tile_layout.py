"""The padded LDS layout of the element tiles at every compiled order: both workgroup tiles, a
mesh whose last tile is partial, node arrays of all three forms (Euler, BR1, interior penalty).

Bar: 1e-12 of the oracle's max-norm after two RK3 steps (the FP64 bar of the parity tests; each
step's rounding is ~1e-15), and the two tiles bit for bit, QDot included.
"""
import numpy as np
import pytest

from horses2d_amd import cases as C

pytestmark = pytest.mark.gpu


def _case(N, viscous):
    if viscous == "none":
        case = C.euler_vortex_case(5, N)
    else:
        case = C.ns_tgv_case(5, N, riemann="roe", viscous=viscous)
    case.mesh = C.periodic_rectangle(5, 5, 0.0, 2.0 * np.pi, 0.0, 5.0) if viscous != "none" else case.mesh
    case.cfl = 0.05
    return case


@pytest.mark.parametrize("viscous", ["none", "br1", "ip"])
@pytest.mark.parametrize("N", list(range(1, 13)))
def test_every_order_and_tile(N, viscous):
    from horses2d_amd import gpu
    from oracle.oracle import Oracle
    case = _case(N, viscous)
    orc = Oracle(case)
    Q0 = case.initial_state(orc.coords())
    orc.set_state(Q0)
    dt = orc.estimate_dt(case.dt_max, case.cfl)
    for _ in range(2):
        orc.step(0.0, dt, case.scheme)
    ref = orc.state()
    got = []
    for tile in (0, 1):
        dg = gpu.DGSEM(case, "fp64", apply_ic=False)
        dg.set_tiles(tile, tile)
        dg.upload(Q0)
        qdot = dg.time_derivative()
        for _ in range(2):
            dg.rk_step(0.0, dt)
        got.append((dg.state(), qdot, dg.residuals()))
        assert np.max(np.abs(got[-1][0] - ref)) <= 1e-12 * np.max(np.abs(ref))
        dg.close()
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)
