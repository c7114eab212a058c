"""Several right-hand sides: column counts at and between the kernels' groups
of four, one and two chunks of staged columns, ragged rows, short and long
rows.  The operator against scipy in FP64; the solve's columns against
one-column solves, zero columns among them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PARAMS = dict(solverType=1, tolerance=1e-11, maxIters=500, smootherType=1, preInnerIters=3, postInnerIters=3,
              topSize=64, aggregationRule=1, strengthThreshold=0.01, proOmega=0.5)


def _solver(fem, dim, n):
    mg = fem.meshgen
    xyz, conn = mg.square_mesh(n, seed=3) if dim == 2 else mg.cube_mesh(n, seed=3)
    kappa = mg.lognormal_kappa(3, conn.shape[0], 0.5)
    return fem.FEMSolver.from_arrays(dim, xyz, conn, kappa=kappa, mass_coeff=1.0)


@pytest.mark.parametrize("k", [2, 3, 4, 5, 8, 9, 12, 13, 16, 17, 24, 33, 64])
def test_operator_columns(gpu, fem, k):
    s = _solver(fem, 3, 21)
    x = np.random.default_rng(k).standard_normal((s.getMatrixRows(), k))
    A = s.get_matrix_scipy()
    m = int(np.diff(A.indptr).max())
    bound = (m + 4) * 2.0 ** -53 * (abs(A) @ abs(x))
    assert np.all(abs(s.apply_operator(x) - A @ x) <= bound)  # CSR, before a setup
    s.set_params(precision=0, **PARAMS)
    s.setup()
    assert np.all(abs(s.apply_operator(x) - A @ x) <= bound)  # the staged copy
    s.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("dim,n,k", [(3, 17, 2), (3, 33, 5), (3, 41, 12), (2, 150, 3), (2, 61, 20), (3, 9, 64)])
def test_solve_columns(gpu, fem, dim, n, k, precision):
    s = _solver(fem, dim, n)
    s.set_params(precision=precision, **PARAMS)
    rng = np.random.default_rng(10 * n + k)
    b = rng.standard_normal((s.getMatrixRows(), k))
    b[:, 1] = 0.0
    x, info = s.solve(b)
    assert info["status"] == 0
    assert np.all(x[:, 1] == 0.0)
    A = s.get_matrix_scipy()
    r = np.linalg.norm(b - A @ x, axis=0)
    # the library's own test is the same residual to 1e-11; FP64 rounding of this one on top
    slack = 2.0 ** -53 * 30 * np.linalg.norm(abs(A) @ abs(x), axis=0)
    assert np.all(r <= 1.01e-11 * np.linalg.norm(b, axis=0) + slack)
    for c in (0, k - 1):
        xc, _ = s.solve(np.ascontiguousarray(b[:, c]))
        assert np.linalg.norm(xc - x[:, c]) <= 1e-8 * max(np.linalg.norm(xc), 1e-300)
    s.close()
