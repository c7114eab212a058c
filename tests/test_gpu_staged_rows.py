"""The LDS-staged row sums at the edges of their dispatch: fewer blocks than
CUs, 2D and 3D row lengths over one and several staging blocks, a slice whose
longest row is far beyond the preloaded steps, ragged row counts.  Each
product and smoothing step against scipy in FP64."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

PARAMS = dict(solverType=1, tolerance=1e-9, maxIters=500, smootherType=1, preInnerIters=3, postInnerIters=3,
              topSize=64, aggregationRule=1, strengthThreshold=0.01, proOmega=0.5)


def _mesh(fem, dim, n, hub):
    mg = fem.meshgen
    xyz, conn = mg.square_mesh(n, seed=2) if dim == 2 else mg.cube_mesh(n, seed=2)
    if hub:
        # one vertex joined to `hub` others (overlapping simplices: only the matrix matters here)
        ring = np.arange(1, hub + 2, dtype=np.int32)
        fan = np.stack([np.zeros(hub, dtype=np.int32), ring[:-1], ring[1:]], 1)
        if dim == 3:
            fan = np.concatenate([fan, np.roll(ring, 3)[:-1, None] + hub + 1], 1)
        conn = np.concatenate([conn, fan.astype(np.int32)])
    return xyz, conn


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("dim,n,hub", [(2, 9, 0), (2, 181, 0), (2, 183, 37), (3, 32, 0), (3, 33, 41)])
def test_staged_products(gpu, fem, dim, n, hub, precision):
    xyz, conn = _mesh(fem, dim, n, hub)
    s = fem.FEMSolver.from_arrays(dim, xyz, conn, mass_coeff=0.5)
    s.set_params(precision=precision, **PARAMS)
    s.setup()
    rng = np.random.default_rng(n)
    u = 2.0 ** -53 if precision == 0 else 2.0 ** -24
    rp, ci, v, _ = s.level_matrix(0)
    A = sp.csr_matrix((v, ci, rp))
    m = int(np.diff(rp).max())
    x, b, d = (rng.standard_normal(A.shape[0]) for _ in range(3))
    mag = abs(A) @ abs(x)
    # m products and sums, and the roundings of the matrix and the vectors
    assert np.all(abs(s.apply_level(0, 0, x) - A @ x) <= (m + 6) * u * mag)
    dinv = 1.0 / A.diagonal()
    for mode, c1, c2 in ((0, 0.7, 0.0), (1, 0.3, 0.9)):
        y, dn = s.smoother_step(0, mode, c1, c2, x, b, d)
        r = dinv * (b - A @ x)
        want_d = c1 * d + c2 * r if mode else d
        want = x + want_d if mode else x + c1 * r
        bound = (m + 16) * u * (abs(x) + abs(d) + dinv * (abs(b) + mag))
        assert np.all(abs(y - want) <= bound) and np.all(abs(dn - want_d) <= bound)
    if s.num_levels() > 1:
        prp, pci, pv = s.level_prolongator(0)
        nc = s.level_matrix(1)[0].size - 1
        P = sp.csr_matrix((pv, pci, prp), shape=(A.shape[0], nc))
        xc = rng.standard_normal(nc)
        assert np.all(abs(s.apply_level(0, 1, xc) - P @ xc) <= (np.diff(prp).max() + 6) * u * (abs(P) @ abs(xc)))
    s.close()
