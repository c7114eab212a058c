"""Handles of several sizes built, solved, set up again and destroyed on
several threads, with the reserve released beside them: no call fails, and
every solution is bitwise the one of a single thread."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PARAMS = dict(solverType=1, tolerance=1e-10, maxIters=500, smootherType=1, preInnerIters=3, postInnerIters=3,
              topSize=64, aggregationRule=1, strengthThreshold=0.01, proOmega=0.5)
CASES = [(13, 0, 1), (19, 1, 5), (12, 2, 1), (16, 1, 2)]


def _run(fem, n, precision, k):
    xyz, conn = fem.meshgen.cube_mesh(n, seed=n)
    kappa = fem.meshgen.lognormal_kappa(n, conn.shape[0], 1.0)
    b = np.random.default_rng(n + k).standard_normal((n ** 3, k)).squeeze()
    s = fem.FEMSolver.from_arrays(3, xyz, conn, kappa=kappa, mass_coeff=0.1)
    s.set_params(precision=precision, **PARAMS)
    out = []
    for i in range(3):
        x, info = s.solve(b)
        assert info["status"] == 0
        out.append(x)
        s.update_kappa(kappa * (1.5 + i))
    s.close()
    return out


def test_threads(gpu, fem):
    want = [_run(fem, *c) for c in CASES]

    def work(t):
        done = 0
        for j in range(6):
            i = (t + j) % len(CASES)
            assert all(np.array_equal(a, w) for a, w in zip(_run(fem, *CASES[i]), want[i]))
            done += 1
        return done

    def release(_):
        for _ in range(40):
            fem.release_cached_memory()
        return 0

    with ThreadPoolExecutor(4) as pool:
        jobs = [pool.submit(work, t) for t in range(3)] + [pool.submit(release, 0)]
        assert sum(j.result() for j in jobs) == 18
    fem.release_cached_memory()
