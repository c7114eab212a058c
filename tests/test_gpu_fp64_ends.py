"""FP64 PCG whose update takes the level-0 smoother's first step and whose last
smoothing step takes r.z: the iterate after a fixed number of iterations
against PCG on the host with the host statement of the V-cycle.  Row counts off
the 64-row slices and the blocks of them, both smoothers, one to three steps on
each side and none (where the separate kernels run), one column and column
counts at and between the groups of four."""
import numpy as np
import pytest

from vcycle_host import HostVCycle

pytestmark = pytest.mark.gpu
ITERS = 4


def _host_pcg(A, host, b):
    x, r = np.zeros_like(b), b.copy()
    z = host.vcycle(0, r)
    p, rz = z.copy(), r @ z
    for _ in range(ITERS):
        q = A @ p
        alpha = rz / (p @ q)
        x += alpha * p
        r -= alpha * q
        z = host.vcycle(0, r)
        rz, old = r @ z, rz
        p = z + (rz / old) * p
    return x


@pytest.mark.parametrize("dim,n,smoother,pre,post,k", [
    (3, 9, 1, 2, 2, 1), (3, 13, 1, 1, 1, 1), (3, 21, 0, 1, 1, 1), (3, 33, 1, 3, 3, 1), (2, 33, 0, 2, 3, 1),
    (2, 90, 1, 3, 2, 1), (3, 13, 1, 0, 2, 1), (3, 13, 1, 2, 0, 1), (3, 13, 1, 2, 2, 3), (3, 21, 0, 1, 2, 4),
    (3, 21, 1, 3, 1, 9), (2, 33, 1, 1, 1, 17), (3, 13, 0, 0, 2, 5), (3, 13, 1, 2, 0, 5)])
def test_iterates(gpu, fem, dim, n, smoother, pre, post, k):
    mg = fem.meshgen
    xyz, conn = mg.square_mesh(n, seed=5) if dim == 2 else mg.cube_mesh(n, seed=5)
    s = fem.FEMSolver.from_arrays(dim, xyz, conn, mass_coeff=1.0)
    s.set_params(precision=0, smootherType=smoother, preInnerIters=pre, postInnerIters=post, topSize=64,
                 aggregationRule=1, strengthThreshold=0.01, proOmega=0.5, solverType=1, maxIters=ITERS,
                 tolerance=1e-14)
    s.setup()
    host, perm = HostVCycle(s), s.permutation()
    b = np.random.default_rng(n + k).normal(size=(perm.size, k))
    want = np.empty_like(b)
    for c in range(k):
        want[perm, c] = _host_pcg(host.A[0], host, b[perm, c])
    got, info = s.solve(b[:, 0] if k == 1 else b)
    got = got.reshape(b.shape)
    assert info["iterations"] == ITERS
    # four iterations of some hundred FP64 operations per entry, in another
    # order on the host: 1e-14 each at the most, times the condition number of
    # the preconditioned operator (below 1e3 with one-sided smoothing too)
    err = np.linalg.norm(got - want, axis=0) / np.linalg.norm(want, axis=0)
    assert np.all(err <= 1e-10), err.max()
    s.close()
