"""Device blocks that come back to the reserve: from a hierarchy that a setup
replaces, from destroyed handles (also on another thread), and reused by
handles of other sizes and precisions.  Every solve is bitwise the one of
freshly allocated memory."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PARAMS = dict(solverType=1, tolerance=1e-10, maxIters=500, smootherType=1, preInnerIters=3, postInnerIters=3,
              topSize=64, aggregationRule=1, strengthThreshold=0.01, proOmega=0.5)


def _run(fem, n, precision, k, between=None):
    xyz, conn = fem.meshgen.cube_mesh(n, seed=n)
    k0 = fem.meshgen.lognormal_kappa(n, conn.shape[0], 1.0)
    b = np.random.default_rng(n + k).standard_normal((n ** 3, k)).squeeze()
    s = fem.FEMSolver.from_arrays(3, xyz, conn, kappa=k0, mass_coeff=0.1)
    s.set_params(precision=precision, **PARAMS)
    out = [s.solve(b)[0]]
    for i in range(3):  # replaced hierarchies
        s.update_kappa(k0 * (1.5 + i))
        if between:
            between()
        out.append(s.solve(b)[0])
    s.close()
    return out


@pytest.mark.parametrize("threads", [0, 3])
def test_reused_blocks(gpu, fem, threads):
    cases = [(17, 0, 1), (21, 1, 5), (12, 2, 1), (17, 1, 1)]
    fresh = []
    for c in cases:
        fem.release_cached_memory()
        fresh.append(_run(fem, *c))
    bad = []

    def check(order):
        for i in order:
            for a, w in zip(_run(fem, *cases[i]), fresh[i]):
                if not np.array_equal(a, w):
                    bad.append(cases[i])

    if threads:
        ts = [threading.Thread(target=check, args=([(t + j) % 4 for j in range(6)],)) for t in range(threads)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    else:
        check([0, 1, 2, 3, 3, 1, 0])
    assert not bad
    fem.release_cached_memory()
