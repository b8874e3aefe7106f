"""Calls whose kernels need 2^32 work items and more in one launch (more than a
launch takes in one dimension): large bases and many points in the reference-
shaped form.  Each against a small call that has the same sums: a basis of 64
functions repeated, whose orbitals use the first copy only, so that V is the
small V repeated."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402
from nukexc_amd import api  # noqa: E402


@pytest.fixture
def ctx():
    c = nk.Context(0)
    yield c
    c.close()
    torch.cuda.empty_cache()


def _rand(*shape, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand(*shape, dtype=torch.float64, device="cuda", generator=g)


def _same_blocks(V, v):
    """V is v repeated, to the order of a few hundred sums."""
    k, r = v.shape[0], V.shape[0] // v.shape[0]
    d = V.view(r, k, r, k) - v[None, :, None, :]
    assert d.abs_().max().item() <= 1e-12 * v.abs().max().item()


@pytest.mark.parametrize("spins,nbf", [(1, 23296), (2, 16384)])
def test_reference_shaped_basis(ctx, spins, nbf):
    """The sum of the split partials: 8 work items per element of V and spin."""
    n, k = 64, 64
    small = _rand(n, k)
    phi = small.repeat(1, nbf // k).t()
    w = _rand(n, seed=1)
    out = []
    for m, f in ((phi, nbf), (small.t(), k)):
        C = torch.zeros(3, f, dtype=torch.float64, device="cuda")
        C[:, :k] = _rand(3, k, seed=2)
        occ = np.array([2.0, 1.5, 0.5])
        print(f"{f} functions, {spins} spins", flush=True)
        r = (api.compute_lda(ctx, m, w, C.t(), occ, (1,)) if spins == 1 else
             api.compute_lsda(ctx, m, w, C.t(), occ, C[:2].t(), occ[:2], (1,)))
        out.append((r.energy, [r.potential] if spins == 1 else [r.potential_alpha,
                                                                r.potential_beta]))
    assert abs(out[0][0] - out[1][0]) <= 1e-12 * abs(out[1][0])
    for V, v in zip(out[0][1], out[1][1]):
        _same_blocks(V, v)


def test_reference_shaped_points(ctx):
    """2^30 points of one function: collocation, density and V."""
    n = (1 << 30) + 77
    basis = nk.make_manual_basis([(1, 0, 0, 1.3, 0.1, 0.2, 0.3)])
    pts = _rand(n, 3)
    print("collocation", flush=True)
    phi = nk.fill_collocation(ctx, basis, pts)
    pick = torch.tensor([0, 63, 64, n // 2, n - 78, n - 77, n - 65, n - 1], device="cuda")
    assert torch.equal(phi[:, pick], nk.fill_collocation(ctx, basis, pts[pick]))
    del pts
    torch.cuda.empty_cache()
    C, f = np.array([[0.7]]), np.array([2.0])
    print("density", flush=True)
    rho = api.compute_density(ctx, phi, C, f)
    ref = phi[0] * 0.7
    ref.mul_(ref).mul_(2.0)
    assert ((rho - ref).abs_() <= 1e-15 * ref).all()
    w = torch.ones(n, dtype=torch.float64, device="cuda")
    exc, vr, _ = api.functional_eval(ctx, (1,), rho)
    E = torch.dot(exc, rho).item()
    del exc, ref
    V = (torch.dot(phi[0] * vr, phi[0])).item()
    del vr, rho
    torch.cuda.empty_cache()
    # 2^30 terms of one sign: any order of the sums to 1e-10
    print("lda", flush=True)
    r = api.compute_lda(ctx, phi, w, C, f, (1,))
    assert abs(r.energy - E) <= 1e-10 * abs(E) and abs(r.potential.item() - V) <= 1e-10 * abs(V)
    print("lsda", flush=True)
    r = api.compute_lsda(ctx, phi, w, C, f / 2, C, f / 2, (1,))
    assert abs(r.energy - E) <= 1e-10 * abs(E)
    for x in (r.potential_alpha, r.potential_beta):
        assert abs(x.item() - V) <= 1e-10 * abs(V)
