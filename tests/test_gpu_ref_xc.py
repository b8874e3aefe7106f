"""compute_density[_and_sigma], compute_lda / compute_gga and their open-shell
forms on held collocation matrices at the edges of the MFMA tiles (16 orbitals,
16 functions, tiles of 32, 64 and 128 functions, 64 points), the matrices at
8-byte alignment inside a buffer of NaN, against plain FP64 sums.  The sums
have at most 1 500 terms of order one, so 1e-11 of the largest element leaves
room for any order."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402
from nukexc_amd import api  # noqa: E402

SHAPES = [(1, 1, 1), (5, 15, 2), (15, 63, 15), (16, 64, 16), (17, 65, 17), (25, 1000, 5),
          (31, 129, 33), (32, 700, 8), (33, 130, 40), (64, 1500, 49), (65, 200, 65), (80, 333, 14),
          (120, 1111, 21), (128, 64, 64), (129, 257, 3), (200, 500, 80), (257, 130, 9)]


@pytest.fixture(scope="module")
def ctx():
    c = nk.Context(0)
    yield c
    c.close()


def _matrix(a):
    """LayoutLeft view of a (N_bf, N_pts) array, one double into a NaN buffer."""
    nbf, n = a.shape
    buf = torch.full((nbf * n + 40,), float("nan"), dtype=torch.float64, device="cuda")
    v = buf[1:1 + nbf * n].view(n, nbf)
    v.copy_(torch.tensor(np.ascontiguousarray(a.T)))
    return v.t()


def _data(nbf, n, nocc, seed):
    rng = np.random.default_rng(seed)
    m = [rng.normal(size=(nbf, n)) for _ in range(4)]
    C = [rng.normal(size=(nbf, k)) / nbf ** 0.5 for k in (nocc, max(1, nocc - 1))]
    f = [rng.uniform(0.5, 2.0, size=c.shape[1]) for c in C]
    w = rng.uniform(0.1, 1.0, size=n)
    rho, gr = [], []
    for c, o in zip(C, f):
        psi = [c.T @ x for x in m]
        rho.append((o[:, None] * psi[0] ** 2).sum(0))
        gr.append([2 * (o[:, None] * psi[0] * p).sum(0) for p in psi[1:]])
    return m, [_matrix(x) for x in m], C, f, w, rho, gr


def _near(got, ref):
    got = got.cpu().numpy()
    assert np.abs(got - ref).max() <= 1e-11 * max(np.abs(ref).max(), 1e-3), np.abs(got - ref).max()


def _v(m, w, a, b):
    z = w * (0.5 * a * m[0] + sum(x * y for x, y in zip(b, m[1:])))
    A = m[0] @ z.T
    return A + A.T


@pytest.mark.parametrize("nbf,n,nocc", SHAPES)
def test_closed_shell(ctx, nbf, n, nocc):
    m, d, C, f, w, rho, gr = _data(nbf, n, nocc, nbf)
    print(f"closed {nbf} {n} {nocc}", flush=True)
    _near(api.compute_density(ctx, d[0], C[0], f[0]), rho[0])
    r, g, s = api.compute_density_and_sigma(ctx, *d, C[0], f[0])
    sig = sum(x * x for x in gr[0])
    _near(r, rho[0])
    _near(s, sig)
    for x, y in zip(g, gr[0]):
        _near(x, y)
    wd, t = torch.tensor(w, device="cuda"), lambda a: torch.tensor(a, device="cuda")
    for fn in ((1, 12), (101, 130)):
        gga = fn[0] > 100
        e, vr, vs = [None if x is None else x.cpu().numpy() for x in
                     api.functional_eval(ctx, fn, t(rho[0]), t(sig) if gga else None)]
        res = (api.compute_gga(ctx, *d, wd, C[0], f[0], fn) if gga else
               api.compute_lda(ctx, d[0], wd, C[0], f[0], fn))
        assert abs(res.energy - (w * rho[0] * e).sum()) <= 1e-11 * abs((w * rho[0] * e).sum())
        _near(res.potential, _v(m, w, vr, [2 * vs * x for x in gr[0]] if gga else []))
        assert torch.equal(res.potential, res.potential.t())


@pytest.mark.parametrize("nbf,n,nocc", SHAPES)
def test_open_shell(ctx, nbf, n, nocc):
    m, d, C, f, w, rho, gr = _data(nbf, n, nocc, 7 + nbf)
    print(f"open {nbf} {n} {nocc}", flush=True)
    wd, t = torch.tensor(w, device="cuda"), lambda a: torch.tensor(a, device="cuda")
    sg = [sum(x * y for x, y in zip(gr[i], gr[j])) for i, j in ((0, 0), (0, 1), (1, 1))]
    for fn in ((1,), (101, 130)):
        gga = fn[0] > 100
        e, vr, vs = [None if x is None else x.cpu().numpy() for x in
                     api.functional_eval_polarized(ctx, fn, t(np.stack(rho, 1)),
                                                   t(np.stack(sg, 1)) if gga else None)]
        args = (wd, C[0], f[0], C[1], f[1], fn)
        res = (api.compute_gga_lsda(ctx, *d, *args) if gga else
               api.compute_lsda(ctx, d[0], *args))
        E = (w * (rho[0] + rho[1]) * e).sum()
        assert abs(res.energy - E) <= 1e-11 * abs(E)
        for s, V in enumerate((res.potential_alpha, res.potential_beta)):
            b = [2 * vs[:, 2 * s] * x + vs[:, 1] * y for x, y in zip(gr[s], gr[1 - s])] if gga else []
            _near(V, _v(m, w, vr[:, s], b))


@pytest.mark.parametrize("na,nb", [(1, 15), (8, 8), (16, 1), (5, 12), (21, 20), (33, 31), (30, 35),
                                   (2, 62)])
def test_spins_sharing_a_tile_of_orbitals(ctx, na, nb):
    """Alpha and beta orbitals in one row of tiles of 16: the border inside a
    tile, at its edges, in a later pass."""
    m, d, _, _, w, _, _ = _data(70, 300, 5, 3)
    rng = np.random.default_rng(100 * na + nb)
    C = [rng.normal(size=(70, k)) / 70 ** 0.5 for k in (na, nb)]
    f = [rng.uniform(0.2, 1.0, k) for k in (na, nb)]
    psi = [[c.T @ x for x in m] for c in C]
    rho = [(k[:, None] * p[0] ** 2).sum(0) for k, p in zip(f, psi)]
    gr = [[2 * (k[:, None] * p[0] * q).sum(0) for q in p[1:]] for k, p in zip(f, psi)]
    t = lambda a: torch.tensor(a, device="cuda")
    sg = [sum(x * y for x, y in zip(gr[i], gr[j])) for i, j in ((0, 0), (0, 1), (1, 1))]
    e, vr, vs = [x.cpu().numpy() for x in
                 api.functional_eval_polarized(ctx, (101, 130), t(np.stack(rho, 1)),
                                               t(np.stack(sg, 1)))]
    res = api.compute_gga_lsda(ctx, *d, t(w), C[0], f[0], C[1], f[1], (101, 130))
    E = (w * (rho[0] + rho[1]) * e).sum()
    assert abs(res.energy - E) <= 1e-11 * abs(E)
    for s, V in enumerate((res.potential_alpha, res.potential_beta)):
        _near(V, _v(m, w, vr[:, s], [2 * vs[:, 2 * s] * x + vs[:, 1] * y
                                     for x, y in zip(gr[s], gr[1 - s])]))
