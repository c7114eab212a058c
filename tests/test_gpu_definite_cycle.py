"""The V-cycle as a preconditioner of strongly varying coefficients: the
smoothers' intervals reach the largest eigenvalue of every level, the cycle is
positive in the direction where it would first lose that, and PCG converges in
a count that depends on neither the precision nor the number of columns."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

pytestmark = pytest.mark.gpu

TUNED = dict(solverType=1, smootherType=1, preInnerIters=3, postInnerIters=3, postRelaxes=1, aggregationRule=1,
             strengthThreshold=0.01, proOmega=0.5, maxIters=1000)


def _problem(fem, dim, n, sigma, seed):
    mg = fem.meshgen
    xyz, conn = mg.square_mesh(n, seed=seed) if dim == 2 else mg.cube_mesh(n, seed=seed)
    kappa = mg.lognormal_kappa(seed, conn.shape[0], sigma)
    s = fem.FEMSolver.from_arrays(dim, xyz, conn, kappa=kappa, mass_coeff=1.0 if dim == 2 else 1e-2)
    s.set_params(topSize=64 if dim == 2 else 300, **TUNED)
    return s, xyz.shape[0]


@pytest.mark.parametrize("dim,n,sigma,seed", [(3, 25, 1.0, 1), (3, 33, 1.0, 2), (3, 33, 2.0, 3), (3, 41, 1.5, 4),
                                             (2, 120, 1.0, 5), (2, 200, 2.0, 6), (3, 6, 1.0, 7), (3, 4, 2.0, 8)])
def test_intervals_reach_the_top(gpu, fem, dim, n, sigma, seed):
    s, rows = _problem(fem, dim, n, sigma, seed)
    s.set_params(topSize=8)
    s.setup()
    perm = s.permutation()
    for l in range(s.num_levels() - 1):
        rp, ci, v, _ = s.level_matrix(l)
        A = sp.csr_matrix((v, ci, rp))
        d = A.diagonal()
        S = sp.diags(d ** -0.5) @ A @ sp.diags(d ** -0.5)
        if S.shape[0] > 400:
            lam, vec = spla.eigsh(S, k=1, which="LA", tol=1e-8)
            lam, vec = lam[0], vec[:, 0]
        else:
            w, V = np.linalg.eigh(S.toarray())
            lam, vec = w[-1], V[:, -1]
        sm = s.level_smoother(l)
        assert lam < sm["lmax"] + sm["lmin"], (l, lam, sm)
        assert sm["lmax"] < 1.2 * lam, (l, lam, sm)
        if l == 0:
            # the residual of the error vec: r.Mr, in user numbering
            e = vec / np.sqrt(d)
            r = np.empty(rows)
            r[perm] = A @ e
            z = s.apply_preconditioner(r)
            assert r @ z > 0.0
    s.close()


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("dim,n,sigma,most", [(3, 57, 1.0, 30), (3, 61, 1.0, 30), (2, 450, 1.0, 45)])
def test_iteration_counts(gpu, fem, dim, n, sigma, most, precision):
    for seed in (1, 2):
        s, rows = _problem(fem, dim, n, sigma, seed)
        s.set_params(precision=precision, tolerance=1e-9)
        b = np.random.default_rng(seed).standard_normal((rows, 5))
        for k in (1, 5):
            x, info = s.solve(np.ascontiguousarray(b[:, :k]).squeeze())
            assert info["status"] == 0 and info["iterations"] <= most, (seed, k, info)
        s.close()
