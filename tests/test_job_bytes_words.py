"""The admission estimate bounds what a job's context really allocates also where the bricks are
down to a few cells, each with many region atoms (staging words), from 200,000 atoms to a million."""
import pytest

from exanbody_amd import _lib
from exanbody_amd.serve import job_bytes, make_job, serve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rho,rcut,skin", [(500000, 0.8, 4.0, 0.4), (500000, 0.6, 4.0, 0.4), (500000, 0.6, 2.5, 0.3),
                                             (500000, 1.0, 3.2, 0.4), (200000, 0.5, 4.6, 0.6), (200000, 0.8, 4.0, 0.4),
                                             (1000000, 0.8, 4.0, 0.4)])
def test_estimate_bounds_the_peak(n, rho, rcut, skin):
    job = make_job(n, rho, 1.0, 3, _lib.PRECISION_MIXED, seed=5, rcut=rcut, skin=skin, dt=0.001)
    results, _ = serve([job])
    assert results[0]["status"] == 0
    print(results[0]["peak_device_bytes"] / job_bytes(job))
    assert 0 < results[0]["peak_device_bytes"] <= job_bytes(job)
