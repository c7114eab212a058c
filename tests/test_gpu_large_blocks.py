"""Operators of more than 2^20 rows, whose staged copies take blocks of eight
slices for one column (and blocks of two beside them for several): row sums,
smoothing steps and solves, with a ragged last block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 1027  # 1,054,729 rows: 16,481 slices, the last block of one slice, its last slice ragged
U = {0: 2.0 ** -53, 1: 2.0 ** -24}


@pytest.fixture(scope="module")
def problem(fem):
    mg = fem.meshgen
    xyz, conn = mg.square_mesh(N, seed=1)
    kappa = mg.lognormal_kappa(1, conn.shape[0], 0.5)
    s = fem.FEMSolver.from_arrays(2, xyz, conn, kappa=kappa, mass_coeff=1.0)
    s.set_params(solverType=1, tolerance=1e-9, maxIters=200, smootherType=1, preInnerIters=3, postInnerIters=3,
                 topSize=64, aggregationRule=1, strengthThreshold=0.01, proOmega=0.5)
    yield s, s.get_matrix_scipy()
    s.close()


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_rows_steps_and_solves(gpu, problem, precision):
    s, A = problem
    s.set_params(precision=precision)
    s.setup()
    rng = np.random.default_rng(precision)
    m = int(np.diff(A.indptr).max())
    perm = s.permutation()
    n = perm.size
    for k in (1, 2, 3, 12, 17):
        x = rng.standard_normal((n, k)).squeeze()
        assert np.all(abs(s.apply_operator(x) - A @ x) <= (m + 4) * U[0] * (abs(A) @ abs(x)))
    Ai = A[perm][:, perm]
    dinv = 1.0 / Ai.diagonal()
    u = U[min(precision, 1)]
    x, b, d = rng.standard_normal((3, n))
    absAx = abs(Ai) @ abs(x)
    y = s.apply_level(0, 0, x)
    assert np.all(abs(y - Ai @ x) <= (m + 4) * u * absAx)
    y, dn = s.smoother_step(0, 1, 0.37, 0.81, x, b, d)
    d_ref = 0.37 * d + 0.81 * dinv * (b - Ai @ x)
    bound = (m + 8) * u * (abs(x) + abs(0.37 * d) + 0.81 * dinv * (abs(b) + absAx))
    assert np.all(abs(dn - d_ref) <= bound) and np.all(abs(y - x - d_ref) <= bound)
    counts = set()
    for k in (1, 2, 5):
        b = rng.standard_normal((n, k)).squeeze()
        x, info = s.solve(b)
        assert info["status"] == 0
        counts.add(info["iterations"])
        r = np.linalg.norm(b - A @ x, axis=0)
        slack = U[0] * 30 * np.linalg.norm(abs(A) @ abs(x), axis=0)
        assert np.all(r <= 1.01e-9 * np.linalg.norm(b, axis=0) + slack)
    assert max(counts) <= 45
