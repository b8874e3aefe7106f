"""The FP64 density contraction and V contraction on one to five function
blocks (odd and even counts, the last one partly filled), batch groups of 1, 2
and 4 and a grid whose batch count is no multiple of them, against the FP64
oracle; and the per-point density of a P that is not symmetric.  Sums of at
most 3 000 points x 300 functions of magnitude <= 1e2: 1e-10 absolute leaves
room for any order."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from gpu_util import basis_dict  # noqa: E402
import nukexc_amd as nk  # noqa: E402
from nukexc_amd import api, configs  # noqa: E402
from oracle import oracle as O  # noqa: E402


@pytest.fixture(scope="module", params=[2, 7, 13, 17, 26])
def case(request):
    rng = np.random.default_rng(request.param)
    xyz, Z = configs.random_walk_molecule(request.param, rng)
    basis = nk.make_manual_basis(configs.sto_functions(Z, xyz, rng))
    c = nk.Context(0)
    c.set_basis(basis)
    n = 2987
    pts = xyz[rng.integers(0, len(Z), n)] + rng.normal(size=(n, 3)) * 2.0
    w = rng.uniform(0.01, 0.1, n)
    own = torch.zeros(n, dtype=torch.int32, device="cuda")
    g = nk.FlatGrid(torch.tensor(pts, device="cuda"), torch.tensor(w, device="cuda"),
                    torch.tensor(xyz, device="cuda"), Z, own)
    c.set_grid(g)
    C = rng.normal(size=(basis.nbf(), 9)) / basis.nbf() ** 0.5
    phi = O.collocation(basis_dict(basis), pts, grad=True)
    yield c, basis, g, C, phi, w, rng
    c.close()


@pytest.mark.parametrize("group", [0, 1, 2, 4])
@pytest.mark.parametrize("funcs", [(1,), (101, 130)])
def test_closed_shell(case, funcs, group):
    c, basis, g, C, phi, w, _ = case
    P = 2 * C @ C.T
    kw = dict(gx=phi[1], gy=phi[2], gz=phi[3]) if funcs[0] > 100 else {}
    E, N, V = O.vxc_from_collocation(phi[0], w, funcs, P=P, **kw)
    print(f"nbf {basis.nbf()} funcs {funcs} group {group}", flush=True)
    c.set_launch(0, group)
    try:
        r = c.vxc(torch.tensor(P, device="cuda"), funcs=funcs, precision="fp64")
    finally:
        c.set_launch()
    assert abs(r.energy - E) <= 1e-11 * abs(E) and abs(r.n_el - N) <= 1e-11 * N
    assert np.abs(r.potential.cpu().numpy() - V).max() <= 1e-10
    assert torch.equal(r.potential, r.potential.t())


@pytest.mark.parametrize("split", [1, 3, 47])
def test_open_shell_repeats_closed(case, split):
    c, _, _, C, _, _, _ = case
    P = torch.tensor(2 * C @ C.T, device="cuda")
    c.set_launch(split, 0)
    try:
        r = c.vxc(P, funcs=(101, 130), precision="fp64")
        u = c.vxc_polarized(0.5 * P, 0.5 * P, funcs=(101, 130), precision="fp64")
    finally:
        c.set_launch()
    assert abs(r.energy - u.energy) <= 1e-11 * abs(r.energy)
    for V in (u.potential_alpha, u.potential_beta):
        assert (V - r.potential).abs().max().item() <= 1e-10


def test_density_of_an_asymmetric_matrix(case):
    """rho = phi^T P phi, grad rho = 2 sum_mu grad phi_mu sum_nu P(nu, mu) phi_nu."""
    c, basis, g, _, phi, _, rng = case
    P = rng.normal(size=(basis.nbf(), basis.nbf())) / basis.nbf()
    X = P.T @ phi[0]
    out = api._density_points(c, torch.tensor(P, device="cuda"), True)
    ref = [(phi[0] * X).sum(0)] + [2 * (d * X).sum(0) for d in phi[1:4]]
    for a, b in zip(out[:4], ref):
        assert np.abs(a.cpu().numpy() - b).max() <= 1e-10 * max(1.0, np.abs(b).max())


@pytest.mark.parametrize("nbf", [1, 5, 64, 65, 130])
def test_gradients_formed_in_the_kernels(nbf):
    """grad Phi of the column sums and of Z is evaluated where it is used:
    shells up to l = 5 in an order that breaks every run, both spins."""
    rng = np.random.default_rng(nbf)
    ctr = rng.normal(size=(4, 3)) * 2.0
    f = []
    for i in range(nbf):
        l = int(rng.integers(0, 6 if i % 2 else 3))
        f.append((l + 1 + int(rng.integers(0, 2)), l, int(rng.integers(-l, l + 1)),
                  float(rng.choice([0.8, 1.3, 2.1])), *ctr[rng.integers(0, 4)]))
    basis = nk.make_manual_basis(f)
    n = 777
    pts = ctr[rng.integers(0, 4, n)] + rng.normal(size=(n, 3)) * 1.5
    w = rng.uniform(0.01, 0.1, n)
    Ca, Cb = (rng.normal(size=(nbf, 3)) / nbf ** 0.5 for _ in range(2))
    Pa, Pb = Ca @ Ca.T, Cb @ Cb.T
    p, gx, gy, gz = O.collocation(basis_dict(basis), pts, grad=True)
    ref = O.vxc_polarized(p, w, (101, 130), Pa, Pb, gx=gx, gy=gy, gz=gz)
    c = nk.Context(0)
    try:
        c.set_basis(basis)
        c.set_grid(nk.FlatGrid(torch.tensor(pts, device="cuda"), torch.tensor(w, device="cuda"),
                               torch.tensor(ctr, device="cuda"), np.ones(4, np.int32),
                               torch.zeros(n, dtype=torch.int32, device="cuda")))
        dev = lambda a: torch.tensor(a, device="cuda")
        u = c.vxc_polarized(dev(Pa), dev(Pb), funcs=(101, 130), precision="fp64")
    finally:
        c.close()
    assert abs(u.energy - ref[0]) <= 1e-11 * abs(ref[0])
    for V, R in zip((u.potential_alpha, u.potential_beta), ref[-2:]):
        assert np.abs(V.cpu().numpy() - R).max() <= 1e-10 * max(1.0, np.abs(R).max())
