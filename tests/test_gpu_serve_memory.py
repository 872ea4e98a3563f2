"""Device memory that the job server's batch takes beside the jobs' footprints:
the volume-pass records, the work units and the emptiness pass's second list
stay within the running jobs' shares and what the budget has left (or the
fixed 262,144 records), whatever ran before."""
import ctypes

import numpy as np
import pytest
from conftest import problem
from test_gpu_knn import _Hip

pytestmark = pytest.mark.gpu

MB = 1 << 20
REC = 16 + 4 * 20  # a record at the automatic vertex cap of 17
CFG = dict(accum="f64", moments="robust", tet_k=20)


def _free(hip):
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.L.hipDeviceSynchronize() == 0
    assert hip.L.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
    return a.value


def _used(vdn, hip, budget, rounds, **cfg):
    """Device bytes with every job running, and the jobs' results."""
    free = _free(hip)
    with vdn.Server(budget_bytes=budget, **{**CFG, **cfg}) as s:
        ids = []
        for jobs in rounds:
            ids += [s.submit(*p, 8) for p in jobs]
            s.step()
            assert s.step() == (len(ids), 0)
        used = free - _free(hip)
        while s.step() != (0, 0):
            pass
        return used, [s.result(i) for i in ids]


def _job_bytes(vdn, p):
    with vdn.Server(**CFG) as s:
        s.submit(*p, 3)
        s.step()
        return s.bytes_in_use()


def _alone(vdn, p, n_iter):
    with vdn.Engine(**CFG) as e:
        e.set_mesh(*p[:2])
        e.set_sites(p[2])
        e.lloyd(n_iter)
        return e.sites()


@pytest.mark.parametrize("n,ns", [(30, 16200), (20, 2000)])
def test_records_of_a_lone_job_are_given_back(vdn, n, ns):
    hip = _Hip()
    jobs = [problem("cube", n, ns, seed) for seed in (3, 4)]
    budget = 2 * _job_bytes(vdn, jobs[0]) + MB
    together, want = _used(vdn, hip, budget, [jobs])
    after, got = _used(vdn, hip, budget, [jobs[:1], jobs[1:]])
    assert after <= together + 8 * MB
    for a, b, p in zip(got, want, jobs):
        alone = _alone(vdn, p, 8)
        np.testing.assert_array_equal(a, alone)
        np.testing.assert_array_equal(b, alone)


@pytest.mark.parametrize("n,ns", [(30, 16200), (20, 2000)])
def test_records_within_the_jobs_shares(vdn, n, ns):
    hip = _Hip()
    jobs = [problem("cube", n, ns, seed) for seed in (3, 4)]
    budget = 2 * _job_bytes(vdn, jobs[0]) + MB
    without, _ = _used(vdn, hip, budget, [jobs], site_records=-1)
    used, _ = _used(vdn, hip, budget, [jobs])
    share = sum(len(p[1]) for p in jobs) * CFG["tet_k"] // 10 * REC
    assert used - without <= share + 262144 * REC + 8 * MB


def test_given_records_are_kept(vdn):
    """A given number of records above the limit: taken as it is, with the same
    memory at each step."""
    hip = _Hip()
    p = problem("cube", 20, 2000)
    with vdn.Server(budget_bytes=_job_bytes(vdn, p) + MB, **{**CFG, "site_records": 900000}) as s:
        j = s.submit(*p, 8)
        s.step()
        held = _free(hip)
        for _ in range(6):
            s.step()
            assert _free(hip) == held
        assert s.step() == (0, 0)
        np.testing.assert_array_equal(s.result(j), _alone(vdn, p, 8))
