"""The gradient's runs of functions on one centre with functions of zero norm at
their starts, ends and in between: those contribute nothing, so the gradient is
that of the basis without them (the same sums in another order: 1e-11 of its
size; the int8 form's slices differ, 1e-6)."""
import dataclasses

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("mixed", 1e-6)])
@pytest.mark.parametrize("zero", [[0], [1, 2], [0, 7, 8], [8, 9, 15, 16, 17], list(range(0, 42, 3))])
def test_zero_norm_functions(zero, precision, tol):
    rng = np.random.default_rng(len(zero))
    xyz, Z = np.array([[0.0, 0.1, 0.0], [0.0, 1.9, 1.3]]), np.array([8, 6], np.int32)
    shells = [(1, 0, 5.0), (2, 0, 1.8), (2, 1, 1.9), (2, 1, 1.9), (3, 2, 1.7), (4, 3, 2.0), (2, 0, 1.1)]
    f = [(n, l, m, z, *x) for x in xyz for n, l, z in shells for m in range(-l, l + 1)]
    nbf = len(f)
    basis = nk.make_manual_basis(f)
    norm = np.array(basis.norm, float)
    norm[zero] = 0.0
    keep = np.setdiff1d(np.arange(nbf), zero)
    small = nk.make_manual_basis([f[i] for i in keep])
    C = np.linalg.qr(rng.normal(size=(nbf, 4)))[0]
    P = 2 * C @ C.T
    c = nk.Context(0)
    try:
        c.make_flat_grid(xyz, Z, nrad=25, nang_order=17)
        c.set_basis(dataclasses.replace(basis, norm=norm))
        a = c.xc_grad(torch.tensor(P, device="cuda"), funcs=(101, 130), precision=precision)[1]
        c.set_basis(small)
        b = c.xc_grad(torch.tensor(P[np.ix_(keep, keep)].copy(), device="cuda"),
                      funcs=(101, 130), precision=precision)[1]
    finally:
        c.close()
    assert np.abs(a - b).max() <= tol * max(1.0, np.abs(b).max())
