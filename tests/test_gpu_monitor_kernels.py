"""The reductions behind the monitors at the edges of their rounds: the time-step scan (4096 elements
a round), the conservation sums (1024 partials a round), the probes at the smallest and largest order.

The scan's maxima and minimum are exact in any order; numpy's prefix maxima take the element side from
the mesh's extent, while the library subtracts corner coordinates (rounded at 5, over sides down to
0.04: 1e-13), hence 1e-12.  The sums are compared at 1e-13 of the sum of magnitudes (the unit rounding
times the depth of the additions), the probes at 1e-13 of the state (two interpolations of at most 13
products with weights below 4)."""
import numpy as np
import pytest

from horses2d_amd import cases as C

pytestmark = pytest.mark.gpu


def _solver(nx, ny, N):
    from horses2d_amd import gpu
    mesh = C.periodic_rectangle(nx, ny, -5.0, 5.0, -5.0, 5.0)
    return gpu.DGSEM(C.Case("m", mesh, np.full(mesh.K, N, np.int32), 0.5, cfl=0.1,
                            ic=C.isentropic_vortex(0.5, 4.0, 0.3, -0.2)), "fp64")


@pytest.mark.parametrize("nx, ny, N", [(2, 2, 3), (63, 65, 1), (64, 64, 1), (17, 241, 2), (128, 65, 1), (3, 5, 12)])
def test_scan_and_sums(nx, ny, N):
    dg = _solver(nx, ny, N)
    K, P = nx * ny, N + 1
    rng = np.random.Generator(np.random.PCG64(K))
    Q = dg.state().reshape(K, P * P, 4)
    Q[..., 3] *= 1.0 + 0.3 * rng.uniform(size=(K, 1))   # uneven elements: the running maxima matter
    dg.upload(Q.reshape(-1))
    u = np.hypot(Q[..., 1], Q[..., 2]) / Q[..., 0]
    a = np.sqrt(1.4 * 0.4 * (Q[..., 3] / Q[..., 0] - 0.5 * u * u))
    um, am = np.maximum.accumulate(u.max(1)), np.maximum.accumulate(a.max(1))
    dt = np.min(0.5 * np.sqrt(1.4) * 0.1 * min(10.0 / nx, 10.0 / ny) / (um + am) / P)
    assert dg.estimate_dt(1e30, 0.1) == pytest.approx(dt, rel=1e-12)
    again = np.min(0.5 * np.sqrt(1.4) * 0.1 * min(10.0 / nx, 10.0 / ny) / (um[-1] + am[-1]) / P)
    assert dg.estimate_dt(1e30, 0.1) == pytest.approx(again, rel=1e-12)   # the saved maxima
    w = 0.5 * np.polynomial.legendre.leggauss(P)[1]
    terms = Q * (np.outer(w, w).reshape(-1) * (100.0 / K))[None, :, None]
    got = dg.conservation_sums()
    assert np.all(np.abs(got - terms.sum((0, 1))) <= 1e-13 * np.abs(terms).sum((0, 1)))


@pytest.mark.parametrize("N", [1, 6, 12])
def test_probes_on_nodes_and_between(N):
    dg = _solver(5, 4, N)
    P = N + 1
    Q = dg.state().reshape(20, P, P, 4)
    x = 0.5 + 0.5 * np.polynomial.legendre.leggauss(P)[0]
    wb = np.array([1.0 / np.prod([x[i] - x[j] for j in range(P) if j != i]) for i in range(P)])
    rng = np.random.Generator(np.random.PCG64(N))
    el, xi, eta = rng.integers(0, 20, 70), rng.uniform(size=70), rng.uniform(size=70)

    def lag(s):
        c = wb / (s - x)
        return c / c.sum()
    dg.probes_set(el, xi, eta, [("rho", "rhou", "rhov", "rhoe")[k % 4] for k in range(70)])
    ref = np.array([lag(eta[k]) @ Q[el[k], :, :, k % 4] @ lag(xi[k]) for k in range(70)])
    assert np.max(np.abs(dg.probes_update() - ref)) <= 1e-13 * np.max(np.abs(Q))
