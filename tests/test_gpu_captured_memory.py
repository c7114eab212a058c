"""The allocation-free preconditioner in a caller's graph: every replay, on
streams that the library does not know, gives the eager result, and the memory
that the graph's launches may still use is not handed on by the library: it
goes back to the device, which waits for them."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_captured_preconditioner(gpu, fem, precision):
    import torch
    n = 33
    xyz, conn = fem.meshgen.cube_mesh(n, seed=5)
    s = fem.FEMSolver.from_arrays(3, xyz, conn, mass_coeff=0.1)
    s.set_params(precision=precision, solverType=1, smootherType=1, preInnerIters=3, postInnerIters=3, topSize=300,
                 aggregationRule=1, strengthThreshold=0.01, proOmega=0.5)
    s.setup()
    L = fem.lib()
    rng = np.random.default_rng(8)
    rs = [rng.standard_normal(n ** 3) for _ in range(3)]
    want = [s.apply_preconditioner(r) for r in rs]
    r = torch.zeros(n ** 3, dtype=torch.float64, device="cuda")
    z = torch.zeros_like(r)
    side, other = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    assert L.fem_set_stream(s._h, C.c_void_p(side.cuda_stream)) == 0
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        st = L.fem_apply_preconditioner_noalloc(s._h, C.c_void_p(r.data_ptr()), C.c_void_p(z.data_ptr()))
    assert st == 0, L.fem_last_error(s._h).decode()
    with torch.cuda.stream(other):
        for _ in range(2):
            for a, w in zip(rs, want):
                r.copy_(torch.from_numpy(a))
                g.replay()
                assert np.array_equal(z.cpu().numpy(), w)
    fem.release_cached_memory()
    free = torch.cuda.mem_get_info()[0]
    s.close()
    assert torch.cuda.mem_get_info()[0] - free > 4 << 20  # 215,000 elements, 36,000 rows
