"""Calls whose kernels need 2^32 work items and more in one launch (the most that a
launch takes in one dimension): large bases in the reference-shaped and the
batched form, many points, many batches beside a large basis.  Each against a
small call that has the same sums: bases of 64 (or fewer) functions repeated,
whose orbitals or density matrix use the first copy only, so that V is the
small V repeated."""
import dataclasses

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402
from nukexc_amd import api  # noqa: E402


@pytest.fixture
def ctx():
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 240 << 30:
        pytest.skip("needs up to 240 GB of device memory")
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
    d = torch.sub(V.view(r, k, r, k), v[None, :, None, :], out=V.view(r, k, r, k))  # in place
    assert max(d.max().item(), -d.min().item()) <= 1e-12 * v.abs().max().item()


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


def _small_basis():
    shells = [(1, 0, 4.0), (2, 0, 3.5), (2, 1, 3.7), (3, 2, 4.1)]
    f = [(a, l, m, z * s, 0.0, 0.0, 0.0) for s in (1.0, 1.1, 1.2, 1.3, 1.4, 1.5, 1.6)
         for a, l, z in shells for m in range(-l, l + 1)][:64]
    return nk.make_manual_basis(f)


def _repeated(b, centers):
    """b copied to each centre."""
    r = len(centers)
    t = lambda a: np.tile(a, r)
    O = np.repeat(centers, b.nbf(), axis=0)
    return dataclasses.replace(b, n=t(b.n), l=t(b.l), m=t(b.m), norm=t(b.norm), zeta=t(b.zeta),
                               O=O, cutoff_radii=t(b.cutoff_radii))


def _set_points(ctx, pts, centers):
    n = pts.shape[0]
    ctx.set_grid(nk.FlatGrid(pts, torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda"),
                             torch.tensor(centers, device="cuda"),
                             np.ones(len(centers), np.int32),
                             torch.zeros(n, dtype=torch.int32, device="cuda")))


def _spd(k, nbf, seed):
    C = np.linalg.qr(np.random.default_rng(seed).normal(size=(k, 4)))[0]
    P = torch.zeros(nbf, nbf, dtype=torch.float64, device="cuda")
    P[:k, :k] = torch.tensor(C @ C.T, device="cuda")
    return P


@pytest.mark.parametrize("spins,blocks", [(2, 512), (1, 1024)])
def test_batched_basis(ctx, spins, blocks):
    """The end of a build of many function blocks, 64 workgroups per block pair
    and spin, and (1024 blocks) the gathering of P."""
    b = _small_basis()
    k = b.nbf()
    out = []
    for r in (blocks, 1):
        centers = np.zeros((r, 3))
        _set_points(ctx, _rand(64, 3) - 0.5, centers[:1])
        ctx.set_basis(_repeated(b, centers))
        print(f"{r * k} functions", flush=True)
        if spins == 2:
            x = ctx.vxc_polarized(_spd(k, r * k, 1), _spd(k, r * k, 2), funcs=(1,))
            out.append((x.energy, [x.potential_alpha, x.potential_beta]))
        else:
            x = ctx.vxc(_spd(k, r * k, 1), funcs=(1,))
            out.append((x.energy, [x.potential]))
        del x
    (Ea, Va), (Ec, Vc) = out
    assert abs(Ea - Ec) <= 1e-12 * abs(Ec)
    for V, v in zip(Va, Vc):
        _same_blocks(V, v)


@pytest.mark.parametrize("precision,shape,tol", [("fp64", 0, 1e-11), ("mixed", 65, 1e-8),
                                                 ("mixed", 71, 1e-8)])
def test_batches_beside_a_large_basis(ctx, precision, shape, tol):
    """512 function blocks on centres far apart, 2^23 points around the first: the
    density and gradient kernels deal a workgroup to every (batch, pair of list
    blocks) that the basis allows.  The other centres see nothing.  (FP64: 8 M
    terms a sum, 1e-11 for any order; int8: the blocks are shared with the next
    centres' functions, which have row exponents of their own.)"""
    ctx.set_launch(0, shape)
    b = _small_basis()
    k, n = b.nbf(), (1 << 23) + 129
    pts = (_rand(n, 3) - 0.5) * 3.0
    out = []
    for r in (512, 1):
        centers = np.zeros((r, 3))
        centers[:, 0] = 200.0 * np.arange(r)
        _set_points(ctx, pts, centers)
        ctx.set_basis(_repeated(b, centers))
        P = _spd(k, r * k, 1)
        print(f"{r * k} functions, {n} points", flush=True)
        v = ctx.vxc(P, funcs=(101, 130), precision=precision)
        g = (ctx.xc_grad(P, funcs=(101, 130), partition="fixed")[1] if precision == "fp64" else
             np.zeros((r, 3)))
        out.append((v, g))
    (a, ga), (c, gc) = out
    assert abs(a.energy - c.energy) <= tol * abs(c.energy)
    assert abs(a.n_el - c.n_el) <= tol * c.n_el
    d = (a.potential[:k, :k] - c.potential).abs().max().item()
    assert d <= tol * c.potential.abs().max().item()
    a.potential[:k, :k] = 0.0
    assert a.potential.abs().max() <= 1e-100  # the same block, centres 200 bohr apart
    assert np.abs(ga[:1] - gc).max() <= tol and np.abs(ga[1:]).max() <= 1e-100
