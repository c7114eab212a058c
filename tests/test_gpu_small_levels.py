"""The V-cycle's small levels run in one launch: the preconditioner against
the host statement of the same V-cycle where that launch takes everything
below level 0, several levels, only the coarsest solve, or nothing (too many
smoothing steps, too large a coarsest level), with odd and even step counts on
both sides of the correction."""
import numpy as np
import pytest

from vcycle_host import HostVCycle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("dim,n,top,smoother,pre,post", [
    (3, 9, 64, 1, 3, 3), (3, 12, 4, 1, 2, 2), (3, 17, 8, 0, 1, 1), (3, 17, 300, 1, 3, 3), (2, 60, 4, 1, 4, 3),
    (2, 60, 4, 0, 2, 5), (2, 97, 16, 1, 0, 1), (2, 97, 16, 1, 1, 0), (2, 40, 8, 1, 8, 8), (2, 40, 8, 1, 9, 9),
    (3, 33, 300, 1, 3, 3), (2, 90, 900, 1, 3, 3)])
def test_small_levels(gpu, fem, dim, n, top, smoother, pre, post, precision):
    mg = fem.meshgen
    xyz, conn = mg.square_mesh(n, seed=5) if dim == 2 else mg.cube_mesh(n, seed=5)
    s = fem.FEMSolver.from_arrays(dim, xyz, conn, mass_coeff=1.0)
    s.set_params(precision=precision, smootherType=smoother, preInnerIters=pre, postInnerIters=post, topSize=top,
                 aggregationRule=1, strengthThreshold=0.01, proOmega=0.5, solverType=1)
    s.setup()
    host = HostVCycle(s)
    perm = s.permutation()
    r = np.random.default_rng(n).normal(size=perm.size)
    z = np.empty_like(r)
    want = host.vcycle(0, r[perm])
    z[perm] = want
    got = s.apply_preconditioner(r)
    err = np.linalg.norm(got - z) / np.linalg.norm(z)
    if precision == 0:
        tol = 1e-10
    else:
        # what rounding the input and the stored hierarchy to FP32 changes, and
        # the rounding of some twenty FP32 operations per level on top
        e = [np.linalg.norm(v - want) / np.linalg.norm(want) for v in
             (host.vcycle(0, r[perm].astype(np.float32).astype(np.float64)), host.rounded_to_fp32().vcycle(0, r[perm]))]
        tol = 20 * sum(e) + 1e-6
    assert err <= tol, (err, tol, s.num_levels())
    assert np.array_equal(got, s.apply_preconditioner(r))
    s.close()
