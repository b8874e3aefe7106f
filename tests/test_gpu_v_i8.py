"""The int8 V contraction on one to five function blocks (diagonal super-pairs of
one and two blocks, off-diagonal ones with one and two J blocks), split counts
around a window and past the batches, closed and open shell, against the FP64
form: the int8 form's own error is below 1e-7 of the largest element."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402
from nukexc_amd import configs  # noqa: E402


@pytest.fixture(scope="module", params=[2, 7, 13, 17, 26])
def case(request):
    rng = np.random.default_rng(50 + request.param)
    xyz, Z = configs.random_walk_molecule(request.param, rng)
    basis = nk.make_manual_basis(configs.sto_functions(Z, xyz, rng))
    c = nk.Context(0)
    c.make_flat_grid(xyz, Z, nrad=16, nang_order=11)
    c.set_basis(basis)
    S = c.overlap().cpu().numpy()
    _, P = configs.loewdin_orbitals(S, min(8, basis.nbf()), rng)
    P = torch.tensor(P, device="cuda")
    yield c, basis.nbf(), P, c.vxc(P, precision="fp64")
    c.close()


@pytest.mark.parametrize("split", [0, 1, 3, 9, 100000])
def test_closed_and_open_shell(case, split):
    c, nbf, P, ref = case
    print(f"nbf {nbf} split {split}", flush=True)
    c.set_launch(split, 0)
    try:
        r = c.vxc(P, precision="mixed")
        u = c.vxc_polarized(0.5 * P, 0.5 * P, precision="mixed")
    finally:
        c.set_launch()
    big = ref.potential.abs().max().item()
    for V in (r.potential, u.potential_alpha, u.potential_beta):
        assert (V - ref.potential).abs().max().item() <= 1e-7 * max(big, 1.0)
        assert torch.equal(V, V.t())
    assert abs(r.energy - ref.energy) <= 1e-6 and abs(r.n_el - ref.n_el) <= 1e-6


@pytest.mark.parametrize("kind", ["zero", "tiny", "rows", "nan"])
def test_slices_of_unusual_matrices(case, kind):
    """Elements that are zero, below the smallest stored exponent, far apart in
    one row, or not a number (which counts as zero, bit for bit)."""
    c, nbf, P, ref = case
    Q = P.clone()
    if kind == "zero":
        Q.zero_()
    elif kind == "tiny":
        Q *= 1e-200
    elif kind == "rows":
        s = torch.pow(2.0, -4.0 * (torch.arange(nbf, device="cuda", dtype=torch.float64) % 9))
        Q = s[:, None] * Q * s[None, :]
    else:
        Q[0, nbf - 1] = Q[nbf - 1, 0] = 0.0
    r = c.vxc(Q, precision="mixed")
    if kind == "nan":
        Q[0, nbf - 1] = Q[nbf - 1, 0] = float("nan")
        n = c.vxc(Q, precision="mixed")
        assert n.energy == r.energy and n.n_el == r.n_el and torch.equal(n.potential, r.potential)
        return
    f = c.vxc(Q, precision="fp64")
    assert torch.isfinite(r.potential).all()
    assert abs(r.energy - f.energy) <= 1e-6 and abs(r.n_el - f.n_el) <= 1e-6
