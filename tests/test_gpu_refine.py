"""Calls beside failures that are not their own, and refinement after its own."""
import numpy as np
import pytest

import taucs_amd as T

pytestmark = pytest.mark.gpu


def _system(side):
    A = T.mesh3d(side)
    perm, inv = T.order(A, "genmmd")
    return T.permute(A, perm, inv)


def test_calls_after_a_refused_allocation():
    """An allocation that the device refused, and that the program has dealt
    with, is no failure of the calls that follow: factorization, digest, solves
    (host, device and allocation-free; graphs and eager launches), refinement
    and the CCS solve give the bits that they gave before it."""
    PA = _system(9)
    b = np.random.default_rng(2).uniform(-1, 1, (PA.n, 3))

    def calls():
        out = []
        for prec in (T.FP64, T.FP32):
            print(f"case: calls beside a refused allocation, precision {prec}", flush=True)
            yield
            F = T.factor_llt_mf(PA, precision=prec)
            yield
            out.append(F.digest())
            yield
            out.append(F.solve(b))
            for method in (0, 1):
                yield
                x, info = F.solve_refined(PA, b, method=method)
                assert info.converged
                out.append(x)
            dB, dX = T.DeviceArray(b), T.DeviceArray(np.zeros_like(b))
            yield
            rc = T.lib.taucs_amd_supernodal_solve_many_device_noalloc(F.h, 3, dX.ptr, PA.n, dB.ptr, PA.n)
            assert rc == 0
            out.append(dX.get())
            try:
                T.lib.taucs_amd_set_graphs(0)
                yield
                assert F.numeric(PA, prec) == 0
                yield
                F.solve_device(dX.ptr, dB.ptr, PA.n, 3)
            finally:
                T.lib.taucs_amd_set_graphs(1)
            out.append(dX.get())
            if prec == T.FP64:
                L = F.to_ccs()
                yield
                out.append(L.solve_llt(b[:, 0]))
            dB.free()
            dX.free()
            F.free()
        results.append(out)

    results = []
    for refused in (False, True):
        for _ in calls():
            if refused:
                assert not T.lib.taucs_amd_device_malloc(1 << 46)  # 64 TiB
    for x0, x1 in zip(*results):
        assert np.array_equal(x0, x1)


@pytest.mark.parametrize("method", [0, 1])
def test_every_allocation_of_a_refined_solve_may_fail(method, tmp_path):
    """Each allocation of a factor's first refined solve fails in turn, the
    pinned block of the norms among them.  The call reports it, the ledger
    holds nothing of it once the factor is freed, and the factor's next calls,
    of fewer and of as many right-hand sides, give the bits of a factor that
    never failed."""
    print(f"case: induced failures of a refined solve, method {method}", flush=True)
    PA = _system(6)
    b = np.random.default_rng(4).uniform(-1, 1, (PA.n, 5))

    def both(F):
        return [F.solve_refined(PA, b[:, :k], method=method)[0] for k in (2, 5)]

    F = T.factor_llt_mf(PA, precision=T.FP32)
    ref = both(F)
    F.free()
    held = T.lib.taucs_amd_device_bytes_in_use()
    log = tmp_path / "log"
    T.lib.taucs_logfile(str(log).encode())
    failed = 0
    try:
        for i in range(60):
            F = T.factor_llt_mf(PA, precision=T.FP32)
            T.lib.taucs_allocation_induce_failure(i)
            try:
                F.solve_refined(PA, b, method=method)
            except RuntimeError:
                failed += 1
            ended = T.lib.taucs_allocation_attempts() <= i
            T.lib.taucs_allocation_induce_failure(-1)
            x = both(F)
            assert np.array_equal(x[0], ref[0]) and np.array_equal(x[1], ref[1])
            F.free()
            assert T.lib.taucs_amd_device_bytes_in_use() == held
            if ended:
                break
        assert ended and failed == i
    finally:
        T.lib.taucs_allocation_induce_failure(-1)
        T.lib.taucs_logfile(b"none")
    assert log.read_text().count("hipHostMalloc") == 1
