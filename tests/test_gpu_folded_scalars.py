"""One-column PCG whose update and p kernels sum the partials of p.q and r.z
themselves: the iterate after a fixed number of iterations against PCG on the
host with the library's own preconditioner, below, at and above the row limit
(131,072), where the finish kernels run, in every precision."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ITERS = 4


@pytest.mark.parametrize("dim,shape,precision,cycle", [
    (2, (5, 5), 0, 0), (2, (33, 31), 0, 0), (3, (13, 12, 11), 1, 0), (2, (362, 362), 0, 0), (2, (362, 363), 0, 0),
    (2, (512, 256), 1, 0), (2, (513, 256), 1, 0), (3, (21, 20, 19), 2, 0), (3, (13, 13, 13), 0, 1)])
def test_iterates(gpu, fem, dim, shape, precision, cycle):
    g = np.meshgrid(*[np.arange(m) / (m - 1.0) for m in shape], indexing="ij")
    xyz = np.stack([c.ravel() for c in g], 1)
    if dim == 2:
        i, j = np.meshgrid(*[np.arange(m - 1) for m in shape], indexing="ij")
        a = (i * shape[1] + j).ravel()
        conn = np.concatenate([np.stack([a, a + shape[1], a + shape[1] + 1], 1),
                               np.stack([a, a + shape[1] + 1, a + 1], 1)]).astype(np.int32)
        xyz = np.concatenate([xyz, np.zeros((xyz.shape[0], 1))], 1)
    else:
        s1, s2 = shape[1] * shape[2], shape[2]
        i, j, k = np.meshgrid(*[np.arange(m - 1) for m in shape], indexing="ij")
        a = (i * s1 + j * s2 + k).ravel()
        steps = (s1, s2, 1)
        conn = np.concatenate([np.stack([a, a + steps[p], a + steps[p] + steps[q], a + s1 + s2 + 1], 1)
                               for p in range(3) for q in range(3) if p != q]).astype(np.int32)
    s = fem.FEMSolver.from_arrays(dim, xyz, conn, mass_coeff=1.0)
    s.set_params(precision=precision, smootherType=1, preInnerIters=2, postInnerIters=2, topSize=64,
                 aggregationRule=1, strengthThreshold=0.01, proOmega=0.5, solverType=1, maxIters=ITERS,
                 cycleType=cycle, tolerance=1e-14)
    s.setup()
    A = s.get_matrix_scipy()
    b = np.random.default_rng(shape[0]).normal(size=A.shape[0])
    x, r = np.zeros_like(b), b.copy()
    z = s.apply_preconditioner(r)
    p, rz = z.copy(), r @ z
    for _ in range(ITERS):
        q = A @ p
        alpha = rz / (p @ q)
        x += alpha * p
        r -= alpha * q
        z = s.apply_preconditioner(r)
        rz, old = r @ z, rz
        p = z + (rz / old) * p
    got, info = s.solve(b)
    # the same preconditioner, so only the order of FP64 sums differs; an FP32
    # V-cycle turns last-bit differences of r into FP32 rounding of z
    tol = 1e-10 if precision == 0 else 1e-4
    if info["iterations"] == ITERS:
        assert np.linalg.norm(got - x) <= tol * np.linalg.norm(x)
    else:  # the whole problem is on the coarsest level: solved at once
        assert np.linalg.norm(A @ got - b) <= 1e-12 * np.linalg.norm(b)
    s.close()
