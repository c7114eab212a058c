"""update_kappa with a device tensor (no copy through the host) against the
same coefficients from numpy: layouts and types that a tensor can have, side
streams, and a rejected NaN that leaves the operator as it was."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["plain", "strided", "float32", "grad", "stream", "column"])
def test_device_kappa(gpu, fem, form):
    import torch
    xyz, conn = fem.meshgen.cube_mesh(9, seed=4)
    kappa = fem.meshgen.lognormal_kappa(4, conn.shape[0], 1.0)
    if form == "float32":
        kappa = kappa.astype(np.float32).astype(np.float64)
    ref = fem.FEMSolver.from_arrays(3, xyz, conn, mass_coeff=0.1)
    ref.update_kappa(kappa)
    want = ref.get_matrix_csr()[2]
    s = fem.FEMSolver.from_arrays(3, xyz, conn, mass_coeff=0.1)
    t = torch.from_numpy(kappa).cuda()
    if form == "strided":
        t = torch.stack([t, -t], 1)[:, 0]
    elif form == "float32":
        t = t.to(torch.float32)
    elif form == "grad":
        t = t.requires_grad_(True)
    elif form == "column":
        t = t.reshape(-1, 1)
    if form == "stream":
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            t = torch.zeros_like(t)
            t += torch.from_numpy(kappa).cuda()  # queued on the side stream just before the call
            s.update_kappa(t)
    else:
        s.update_kappa(t)
    assert np.array_equal(s.get_matrix_csr()[2], want)
    bad = torch.from_numpy(kappa).cuda()
    bad[-1] = float("nan")
    with pytest.raises(fem.FemError) as e:
        s.update_kappa(bad)
    assert e.value.status == 6
    assert np.array_equal(s.get_matrix_csr()[2], want)
    s.close()
    ref.close()
