"""A solve whose work vectors do not fit device memory fails with an error,
and the handle then solves as before: one column, and the many columns once
the memory is there."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu



def _fill_device(torch):
    """Allocations that leave less than 256 MB (64 columns at 49^3 take 0.8 GB).
    Freed memory shows late in the device's free bytes, so it is filled until
    an allocation fails."""
    held = []
    for size in (8 << 30, 1 << 30, 128 << 20):
        try:
            while True:
                held.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
        except torch.cuda.OutOfMemoryError:
            pass
    held.pop()
    torch.cuda.empty_cache()
    return held


@pytest.mark.parametrize("precision", [0, 1])
def test_solve_after_failed_growth(gpu, fem, precision):
    import torch
    n, k = 49, 64
    xyz, conn = fem.meshgen.cube_mesh(n, seed=2)
    b = np.random.default_rng(3).standard_normal((n ** 3, k))
    one = np.ascontiguousarray(b[:, 0])
    s = fem.FEMSolver.from_arrays(3, xyz, conn, mass_coeff=1.0)
    s.set_params(precision=precision, solverType=1, tolerance=1e-8, maxIters=200, smootherType=1, preInnerIters=3,
                 postInnerIters=3, topSize=300, aggregationRule=1, strengthThreshold=0.01, proOmega=0.5)
    want, info = s.solve(one)
    assert info["status"] == 0
    fem.release_cached_memory()
    torch.cuda.empty_cache()
    held = _fill_device(torch)
    with pytest.raises(fem.FemError) as e:
        s.solve(b)
    assert e.value.status == 3
    del held
    torch.cuda.empty_cache()
    again, info = s.solve(one)
    assert info["status"] == 0 and np.array_equal(again, want)
    x, info = s.solve(b)
    # two solutions of relative residual 1e-8 at a condition number of 12 (n - 1)^2
    assert info["status"] == 0
    assert np.linalg.norm(x[:, 0] - want) <= 2e-8 * 12 * (n - 1) ** 2 * np.linalg.norm(want)
    s.close()
