"""What the host side asks of the HIP runtime when it moves data, on a stand-in for it (fake_hip.c, which
needs no GPU): each test runs a child process that loads the stand-in before the library."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PRELUDE = """
import ctypes, sys, threading
import numpy as np
F = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)
F.fake_host_flags.restype = F.fake_event_flags.restype = ctypes.c_uint
F.fake_count.restype = F.fake_pending.restype = F.fake_unwaited.restype = ctypes.c_long
F.fake_fail.argtypes = [ctypes.c_int, ctypes.c_long]
F.fake_pinned_most.restype = F.fake_largest_new.restype = ctypes.c_size_t
sys.path.insert(0, {root!r})
from horses2d_amd import gpu, cases as C
HOST_MALLOC, EVENT_CREATE, EVENT_RECORD, EVENT_SYNC, STREAM_SYNC, COPY_ASYNC, LAUNCH = range(7)

def solver(nx, ny, N, precision="fp64"):
    mesh = C.periodic_rectangle(nx, ny, -5.0, 5.0, -5.0, 5.0)
    return gpu.DGSEM(C.Case("t", mesh, np.full(mesh.K, N, np.int32), 0.5, cfl=0.1), precision, apply_ic=False)

def values(dg, seed):
    q = np.random.Generator(np.random.PCG64(seed)).uniform(0.5, 1.5, dg.ndof)
    q.reshape(-1, 4)[:, 3] += 3.0
    return q
"""


@pytest.fixture(scope="module")
def child(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "fake_hip.c"), "-lpthread"],
                   check=True)

    def run(code):
        r = subprocess.run([sys.executable, "-c", PRELUDE.format(so=so, root=os.path.dirname(HERE)) + code],
                           capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
    return run


def test_staging_memory_is_coherent_by_contract(child):
    """Kernels write the staging buffers and the host reads them after an event: coherent memory
    (hipHostMallocCoherent) and events that release to the system (hipEventReleaseToSystem), whatever the
    environment's defaults."""
    child("""
dg = solver(16, 16, 4)
q = values(dg, 1)
dg.upload(q)
assert (dg.state() == q).all()
assert F.fake_count(HOST_MALLOC) > 0 and F.fake_count(EVENT_CREATE) > 0
assert F.fake_host_flags() & 0x40000000, hex(F.fake_host_flags())
assert F.fake_event_flags() & 0x80000000, hex(F.fake_event_flags())
""")


@pytest.mark.parametrize("what, left", [("EVENT_RECORD", "a.state()"), ("STREAM_SYNC", "a.residuals()"),
                                        ("EVENT_SYNC", "a.state()")])
def test_failed_read_leaves_the_pool_clean(child, what, left):
    """A read of one handle that fails with its transfer still on the stream does not hand the buffer that
    transfer writes to another handle."""
    child(f"""
a, b = solver(16, 16, 4), solver(16, 16, 4)
qa, qb = values(a, 1), values(b, 2)
a.upload(qa); b.upload(qb)
assert (a.state() == qa).all() and (b.state() == qb).all()
F.fake_fail({what}, 1)
try:
    {left}
except RuntimeError:
    pass
else:
    raise SystemExit("the failure was not reported")
F.fake_fail({what}, 0)
assert (b.state() == qb).all()
assert (a.state() == qa).all()
""")


def test_failed_upload_leaves_the_one_before_it(child):
    """An upload that cannot wait for the buffer's last transfer does not write into the buffer."""
    child("""
a, b = solver(16, 16, 4), solver(16, 16, 4)
qa, qb = values(a, 1), values(b, 2)
a.upload(qa)
F.fake_fail(EVENT_SYNC, 1)
try:
    b.upload(qb)
except RuntimeError:
    pass
F.fake_fail(EVENT_SYNC, 0)
assert (a.state() == qa).all()
b.upload(qb)
assert (b.state() == qb).all()
""")


@pytest.mark.parametrize("what", ["HOST_MALLOC", "EVENT_CREATE"])
@pytest.mark.parametrize("nx, N", [(16, 4), (80, 5), (200, 6)])
def test_transfers_without_pinned_memory(child, nx, N, what):
    """Where pinned memory (or an event) is not to be had, the runtime's own path moves the data."""
    child(f"""
dg = solver({nx}, {nx}, {N})
q = values(dg, 1)
F.fake_fail({what}, -1)
dg.upload(q)
assert (dg.state() == q).all()
assert (dg.residuals() == 0.0).all() and dg.conservation_sums().shape == (4,)
F.fake_fail({what}, 0)
dg.upload(2.0 * q)
assert (dg.state() == 2.0 * q).all()
""")


def test_upload_of_the_mixed_form_needs_no_memory_of_its_own(child):
    """The mixed form's reference pressure is summed while the state is read: an array of the nodes'
    pressures cost a fifth of the upload's time at 90 k nodes (239 us against 195)."""
    child("""
dg = solver(60, 60, 4, "mixed")
q = values(dg, 1)
F.fake_largest_new()
dg.upload(q)
assert F.fake_largest_new() < 8 * dg.nodes
assert (dg.state() == q).all()
""")


def test_many_threads_share_a_bounded_pool(child):
    """Eight threads' reads, each of up to four shares, make at most eight staging sets (two buffers each)
    in all and free none in between; whoever finds none goes the runtime's way."""
    child("""
solvers = [solver(100, 90 + k, 6) for k in range(8)]
q = [values(s, k) for k, s in enumerate(solvers)]
wrong = []
def work(k):
    solvers[k].upload(q[k])
    for _ in range(6):
        if not (solvers[k].state() == q[k]).all():
            wrong.append(k)
for _ in range(2):
    threads = [threading.Thread(target=work, args=(k,)) for k in range(8)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not wrong
    assert F.fake_count(HOST_MALLOC) <= 16 and F.fake_pinned_most() <= 32 << 20, F.fake_count(HOST_MALLOC)
[s.close() for s in solvers]
last = solver(16, 16, 4)
assert (last.state() == 0.0).all() and F.fake_count(HOST_MALLOC) <= 18
""")


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_upload_returns_with_the_state_in_place(child, precision):
    """hg_upload_state waits for its copy and the traces it starts, at a short state, a long one and a mesh
    of two orders: their errors are its own, and nothing of it is left to a later call."""
    child(f"""
two = C.periodic_rectangle(6, 5, -5.0, 5.0, -5.0, 5.0)
two = gpu.DGSEM(C.Case("two", two, np.repeat([3, 3, 3, 5, 5, 3], 5).astype(np.int32), 0.5, cfl=0.1), {precision!r},
                apply_ic=False)
for dg in (solver(16, 16, 4, {precision!r}), solver(60, 60, 4, {precision!r}), two):
    q = values(dg, 1)
    dg.upload(q)
    assert F.fake_pending() == 0 and F.fake_unwaited() == 0, (F.fake_pending(), F.fake_unwaited())
    assert (dg.state() == q).all()
    dg.synchronize()
""")
