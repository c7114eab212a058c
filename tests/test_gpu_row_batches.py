"""Row sums in batches of entries: every level's operator, prolongator and
restriction against scipy in FP64, in hierarchies whose rows end at every
remainder of the batches, with one and several lanes per row in the sliced and
the row-wise copies; the smoothing steps' vector entries are loaded before the
sum.  An infinite entry of x reaches the rows that hold its column and no other."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


# 2D 841: restriction of 38,000 rows, two lanes each; 3D 97: of 43,000, eight
@pytest.mark.parametrize("precision,dim,n", [(0, 2, 65), (1, 2, 230), (0, 2, 841), (1, 2, 841), (0, 3, 13), (1, 3, 29),
                                             (0, 3, 41), (1, 3, 97)])
def test_levels(gpu, fem, precision, dim, n):
    mg = fem.meshgen
    xyz, conn = mg.square_mesh(n, seed=4) if dim == 2 else mg.cube_mesh(n, seed=4)
    s = fem.FEMSolver.from_arrays(dim, xyz, conn, mass_coeff=1.0)
    s.set_params(precision=precision, smootherType=1, preInnerIters=3, postInnerIters=3, topSize=64,
                 aggregationRule=1, strengthThreshold=0.01, proOmega=0.5, solverType=1)
    s.setup()
    u = 2.0 ** -53 if precision == 0 else 2.0 ** -24
    rng = np.random.default_rng(n)
    for l in range(s.num_levels() - 1):
        rp, ci, v, _ = s.level_matrix(l)
        A = sp.csr_matrix((v, ci, rp))
        prp, pci, pv = s.level_prolongator(l)
        P = sp.csr_matrix((pv, pci, prp), shape=(A.shape[0], s.level_matrix(l + 1)[0].size - 1))
        for which, M in ((0, A), (1, P), (2, P.T.tocsr())):
            x = rng.standard_normal(M.shape[1])
            # products and sums of the longest row, the roundings of M and x
            m = int(np.diff(M.indptr).max())
            assert np.all(abs(s.apply_level(l, which, x) - M @ x) <= (m + 6) * u * (abs(M) @ abs(x))), (l, which)
            j = int(rng.integers(M.shape[1]))
            x[j] = np.inf
            y = s.apply_level(l, which, x)
            hit = np.zeros(M.shape[0], bool)
            hit[M[:, j].nonzero()[0]] = True
            stored = np.zeros(M.shape[0], bool)  # explicit zeros may or may not carry it
            stored[np.repeat(np.arange(M.shape[0]), np.diff(M.indptr))[M.indices == j]] = True
            assert not np.isfinite(y[hit]).any() and np.isfinite(y[~stored]).all(), (l, which)
        x, b, d = (rng.standard_normal(A.shape[0]) for _ in range(3))
        dinv, mag = 1.0 / A.diagonal(), abs(A) @ abs(x)
        bound = (int(np.diff(rp).max()) + 16) * u * (abs(x) + abs(d) + dinv * (abs(b) + mag))
        for mode, c1, c2 in ((0, 0.7, 0.0), (1, 0.3, 0.9)):
            y, dn = s.smoother_step(l, mode, c1, c2, x, b, d)
            r = dinv * (b - A @ x)
            want_d = c1 * d + c2 * r if mode else d
            want = x + want_d if mode else x + c1 * r
            assert np.all(abs(y - want) <= bound) and np.all(abs(dn - want_d) <= bound), (l, mode)
    s.close()
