"""Transfers through the pinned staging pool: every route (one kernel-moved chunk, two, several chunks, two
to four threads) returns the bytes that went in, also from several threads on handles of their own,
after all handles are gone, and with the caller's array changed right after the upload."""
import threading

import numpy as np
import pytest

from horses2d_amd import cases as C

pytestmark = pytest.mark.gpu


def _solver(nx, ny, N):
    from horses2d_amd import gpu
    mesh = C.periodic_rectangle(nx, ny, -5.0, 5.0, -5.0, 5.0)
    return gpu.DGSEM(C.Case("t", mesh, np.full(mesh.K, N, np.int32), 0.5, cfl=0.1), "fp64", apply_ic=False)


def _round_trip(dg, seed):
    Q = np.random.Generator(np.random.PCG64(seed)).uniform(0.5, 1.5, dg.ndof)
    Q.reshape(-1, 4)[:, 3] += 3.0
    sent = Q.copy()
    dg.upload(sent)
    sent[:] = -1.0
    np.testing.assert_array_equal(dg.state(), Q)


# 512 B to 42 MB: 512 KiB = 16384 nodes, two chunks 32768, a thread's share 65536
@pytest.mark.parametrize("nx, ny, N", [(2, 2, 1), (64, 64, 1), (64, 65, 1), (64, 128, 1), (64, 129, 1), (128, 128, 1),
                                       (128, 129, 1), (256, 128, 1), (256, 129, 1), (96, 97, 5), (190, 191, 5)])
def test_round_trip(nx, ny, N):
    dg = _solver(nx, ny, N)
    for seed in (1, 2):
        _round_trip(dg, seed)


def test_values_follow_the_state():
    dg = _solver(16, 16, 3)
    Q = np.tile([1.0, 0.2, 0.1, 2.5], dg.ndof // 4)
    for f in (1.0, 2.0, 3.0):
        dg.upload(f * Q)
        np.testing.assert_allclose(dg.conservation_sums(), 100.0 * f * Q[:4], rtol=1e-13)


def test_threads_and_reopened_pool():
    for _ in range(2):
        solvers = [_solver(60, 50 + 17 * k, 4) for k in range(4)]
        errors = []

        def work(dg, k):
            try:
                for r in range(5):
                    _round_trip(dg, 100 * k + r)
            except BaseException as e:   # noqa: BLE001 (reported by the main thread)
                errors.append(e)
        th = [threading.Thread(target=work, args=(s, k)) for k, s in enumerate(solvers)]
        for t in th:
            t.start()
        for t in th:
            t.join()
        assert not errors, errors
        for s in solvers:
            s.close()                    # the last one frees the pool
