"""The residual maxima at the edges of their three reductions: atomics (up to 256 workgroups of the
last stage), one workgroup over the partials (up to 8192), two passes.

After a time derivative the residual is max |QDot| per equation bit for bit; after a step it is
compared with the oracle (1e-12 of the largest, the FP64 bar)."""
import numpy as np
import pytest

from horses2d_amd import cases as C

pytestmark = pytest.mark.gpu


def _case(nx, ny, N=1):
    mesh = C.periodic_rectangle(nx, ny, -5.0, 5.0, -5.0, 5.0)
    return C.Case("resid", mesh, np.full(mesh.K, N, np.int32), 0.5, cfl=0.1, ic=C.isentropic_vortex(0.5, 4.0, 0.3, -0.2))


@pytest.mark.parametrize("nx, ny", [(2, 2), (32, 64), (8, 257), (64, 1024), (8, 8193)])
def test_residual_is_the_derivatives_maximum(nx, ny):
    from horses2d_amd import gpu
    dg = gpu.DGSEM(_case(nx, ny), "fp64")
    dg.set_tiles(0, 0)          # eight elements per workgroup at N = 1
    q = dg.time_derivative().reshape(-1, 4)
    np.testing.assert_array_equal(dg.residuals(), np.abs(q).max(axis=0))


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("nx, ny", [(2, 2), (32, 64), (8, 257)])
def test_residual_of_a_step(nx, ny, graph):
    from horses2d_amd import gpu
    from oracle.oracle import Oracle
    case = _case(nx, ny)
    orc, dg = Oracle(case), gpu.DGSEM(case, "fp64")
    dg.set_tiles(0, 0)
    dg.set_graph(graph)
    Q0 = case.initial_state(orc.coords())
    orc.set_state(Q0)
    dt = orc.estimate_dt(case.dt_max, case.cfl)
    for _ in range(3):
        orc.step(0.0, dt, case.scheme)
        dg.rk_step(0.0, dt)
        ref = orc.residuals()
        assert np.max(np.abs(dg.residuals() - ref)) <= 1e-12 * np.max(ref)
    Q0[4 * 7 + 2] = np.nan      # a NaN stays, in every equation it reaches
    dg.upload(Q0)
    dg.rk_step(0.0, dt)
    assert np.isnan(dg.residuals()[2])
