"""Galerkin products of every level against scipy, over level sizes on both
sides of the sparse products' dispatch (one to sixteen wavefronts per row,
lane groups, rows of the coarsest levels that hold every column)."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n,theta", [(3, 7, 0.0), (3, 12, 0.01), (3, 20, 0.0), (3, 34, 0.01), (3, 61, 0.01),
                                         (2, 40, 0.0), (2, 170, 0.01), (2, 301, 0.0)])
def test_galerkin_products(gpu, fem, dim, n, theta):
    mg = fem.meshgen
    xyz, conn = mg.square_mesh(n, seed=6) if dim == 2 else mg.cube_mesh(n, seed=6)
    kappa = mg.lognormal_kappa(6, conn.shape[0], 0.5)
    s = fem.FEMSolver.from_arrays(dim, xyz, conn, kappa=kappa, mass_coeff=1.0)
    s.set_params(topSize=4, aggregationRule=1, strengthThreshold=theta, proOmega=0.5, solverType=1)
    s.setup()
    levels = s.num_levels()
    assert levels >= 2
    for l in range(levels - 1):
        rp, ci, v, _ = s.level_matrix(l)
        A = sp.csr_matrix((v, ci, rp))
        prp, pci, pv = s.level_prolongator(l)
        crp, cci, cv, _ = s.level_matrix(l + 1)
        nc = crp.size - 1
        P = sp.csr_matrix((pv, pci, prp), shape=(A.shape[0], nc))
        C = sp.csr_matrix((cv, cci, crp), shape=(nc, nc))
        mag = (abs(P).T @ (abs(A) @ abs(P))).toarray() if nc <= 2000 else None
        want = P.T @ (A @ P)
        # the pattern: every structural product, columns ascending and distinct
        ones = lambda M: sp.csr_matrix((np.ones_like(M.data), M.indices, M.indptr), shape=M.shape)
        pat = (ones(P).T @ (ones(A) @ ones(P))).tocsr()
        pat.sort_indices()
        assert np.array_equal(pat.indptr, crp) and np.array_equal(pat.indices, cci)
        terms = int(np.diff(P.tocsc().indptr).max()) + int(np.diff(rp).max()) + 4
        if mag is not None:
            assert np.all(abs(C.toarray() - want.toarray()) <= terms * 2.0 ** -52 * mag)
        else:
            d = abs(C - want)
            assert d.max() <= terms * 2.0 ** -52 * (abs(P).T @ (abs(A) @ abs(P))).max()
    s.close()
