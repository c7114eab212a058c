"""What update_kappa refuses and what it has to resolve before the library reads
memory: arrays with fewer entries than elements, tensors whose values are not
the ones stored."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solver(fem):
    xyz, conn = fem.meshgen.cube_mesh(5, seed=4)
    kappa = fem.meshgen.lognormal_kappa(4, conn.shape[0], 1.0)
    return fem.FEMSolver.from_arrays(3, xyz, conn, kappa=kappa, mass_coeff=0.1), kappa


@pytest.mark.parametrize("form", ["numpy", "tensor", "device", "empty", "one"])
def test_short_kappa_is_refused(gpu, fem, form):
    import torch
    s, kappa = _solver(fem)
    before = s.get_matrix_csr()[2]
    short = {"empty": kappa[:0], "one": kappa[:1]}.get(form, kappa[:-1])
    if form != "numpy":
        short = torch.from_numpy(short.copy())
        if form == "device":
            short = short.cuda()
    with pytest.raises(ValueError):
        s.update_kappa(short)
    assert np.array_equal(s.get_matrix_csr()[2], before)
    s.update_kappa(np.concatenate([kappa, kappa[:3]]))  # more entries than elements: the first ones count
    assert np.array_equal(s.get_matrix_csr()[2], before)
    s.close()


@pytest.mark.parametrize("form", ["imaginary", "contiguous"])
def test_negated_view(gpu, fem, form):
    """Tensors that store the negative of their values (the imaginary part of
    a conjugate)."""
    import torch
    s, kappa = _solver(fem)
    want = s.get_matrix_csr()[2]
    t = torch.from_numpy(-kappa).cuda()
    t = torch.complex(torch.zeros_like(t), t).conj().imag if form == "imaginary" else torch._neg_view(t)
    assert t.is_neg() and t.is_contiguous() == (form == "contiguous")
    s.update_kappa(np.ones_like(kappa))
    s.update_kappa(t)
    assert np.array_equal(s.get_matrix_csr()[2], want)
    s.close()
