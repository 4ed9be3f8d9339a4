"""Which forms a mesh takes (hg_get_form), on the stand-in for the HIP runtime of test_transfer_runtime: the
meshes of the GPU tests of these forms, and the ones next to them that take the general form."""
from test_transfer_runtime import child  # noqa: F401 (fixture)

MESHES = """
q = tuple(C.freestream_state(0.3))
far, wall = C.Zone(C.BC_FARFIELD, q=q), C.Zone(C.BC_VISCOUSWALL)

def case(mesh, N, viscous="br1", riemann="roe", **more):
    ns = viscous != "none"
    return C.Case("f", mesh, np.broadcast_to(np.asarray(N, np.int32), (mesh.K,)).copy(), 0.3, 200.0 if ns else 0.0, 0.72,
                  ns, riemann=riemann, viscous=viscous, ip_method="sipg", sigma0=1.0, cfl=0.05, **more)

def sheared(bent=0.0, shift=0.0):
    m = C.channel(7, 5, 2.0, 1.0, [wall, far, wall, far])
    m.points[6 * 3 + 2] += [bent, -bent]
    m.points[:] = m.points @ np.array([[1.0, -0.2], [0.3, 0.9]]) + [shift, -0.75 * shift]
    return m

def form(c, precision="fp64"):
    dg = gpu.DGSEM(c, precision, apply_ic=False)
    f = dg.form()
    dg.close()
    return f["metric"], f["parallelograms"], f["trace"], f["one_launch"]
"""


def test_stored_metric_and_parallelograms(child):  # noqa: F811
    child(MESHES + """
for N in (1, 3, 6, 7, 12):
    for viscous in ("br1", "ip"):
        for shift in (0.0, 40.0, 1000.0):
            assert form(case(sheared(shift=shift), N, viscous)) == ("line", True, 3, False), (N, viscous, shift)
        for bent in (0.03, 1e-12):
            assert form(case(sheared(bent), N, viscous)) == ("line", False, 3, False), (N, viscous, bent)
        skewed = C.channel(7, 5, 2.0, 1.0, [far] * 4, skew=0.6)
        assert form(case(skewed, N, viscous)) == ("line", False, 3, False)
    assert form(case(C.channel(7, 5, 2.0, 1.0, [far] * 4), N, "none")) == ("line", False, 0, False)
    curved = C.ns_cylinder_case(3, 12, N=max(N, 3))
    assert form(curved) == ("node", False, 3, False)
    assert form(case(C.channel(7, 5, 2.0, 1.0, [far] * 4), N), "mixed") == ("element", False, 5, False)
    assert form(case(C.channel(7, 5, 2.0, 1.0, [far] * 4, skew=0.6), N), "mixed") == ("node", False, 5, False)
""")


def test_viscous_traces_of_periodic_pairs(child):  # noqa: F811
    child(MESHES + """
def periodic(slant=0.0, curved=False):
    m = C.channel(6, 5, 2.0, 1.0, [wall, C.Zone(C.BC_PERIODIC, direction=1, partner=4), wall,
                                   C.Zone(C.BC_PERIODIC, direction=1, partner=2)])
    m.points[:, 0] *= 1.0 + slant * m.points[:, 1]
    if curved:
        s = np.array([0.0, 0.25, 0.75, 1.0])
        g = 0.5 + 0.5 * np.polynomial.legendre.leggauss(4)[0][0]
        c = g + g * (1.0 - g) / (1.0 - 2.0 * g)          # the edge's slope vanishes at its first node
        bulge = np.stack([0.15 * s * (1.0 - s) * (s - c), 0.0 * s], 1)
        m.cedges = np.array([(j, j + 1) for j in range(5)], np.int32)
        m.cxy = np.array([m.points[j] + s[:, None] * (m.points[j + 1] - m.points[j]) + bulge for j in range(5)])
    return m
for viscous in ("br1", "ip"):
    assert form(case(periodic(), 3, viscous))[2] == 3
    assert form(case(periodic(slant=0.15), 3, viscous))[2] == 5
    assert form(case(periodic(curved=True), 3, viscous))[2] == 5
    assert form(case(periodic(), 3, viscous), "mixed")[2] == 5
""")


def test_one_launch_for_several_orders(child):  # noqa: F811
    child(MESHES + """
rng = np.random.default_rng(5)
mesh = C.channel(9, 7, 3.0, 2.0, [far] * 4, skew=0.4)
pick = lambda orders: rng.choice(orders, mesh.K)
for viscous in ("none", "br1", "ip"):
    trace = 0 if viscous == "none" else 3
    assert form(case(mesh, pick([1, 10]), viscous)) == ("line", False, trace, True)
    assert form(case(mesh, pick([2, 4, 7]), viscous, scheme="rk5")) == ("line", False, trace, True)
    assert not form(case(mesh, pick([4, 11]), viscous))[3]              # beyond the batched kernels' orders
    assert not form(case(mesh, 4, viscous))[3]                          # one order
    assert form(case(mesh, pick([2, 4]), viscous), "mixed")[3]
euler_wall = C.channel(9, 7, 3.0, 2.0, [C.Zone(C.BC_EULERWALL), far, far, far])
assert not form(case(euler_wall, pick([2, 4]), "none"))[3]              # a boundary kind of its own kernels
own = C.channel(9, 7, 3.0, 2.0, [C.Zone(C.BC_FARFIELD, q=q, riemann=C.RIEMANN["exact"]), far, far, far])
assert not form(case(own, pick([2, 4]), "none"))[3]                     # a zone with a solver of its own
""")
