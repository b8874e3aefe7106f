"""STO evaluation by runs of functions: the reference-shaped collocation at the
edges of its tiles (32 functions, 64 points), over shells up to l = 7 in an
order that breaks the runs, with points at a nucleus and far away, against the
oracle; and the nuclear gradient with f functions (beyond the closed forms)
against fourth-order differences of the FP64 energy.  Values and gradients
carry a few roundings of terms of their own size (1e-13 of the largest one);
differences at h = 2e-3 bohr carry h^4 and 1e-12 / h, below 1e-7."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from gpu_util import basis_dict  # noqa: E402
import nukexc_amd as nk  # noqa: E402
from nukexc_amd import api  # noqa: E402
from oracle import oracle as O  # noqa: E402


def _basis(nbf, rng):
    ctr = rng.normal(size=(4, 3)) * 2.0
    out = []
    for i in range(nbf):
        l = int(rng.integers(0, 8 if i % 3 == 0 else 3))
        out.append((l + 1 + int(rng.integers(0, 3)), l, int(rng.integers(-l, l + 1)),
                    float(rng.choice([0.7, 1.3, 2.1])), *ctr[rng.integers(0, 4)]))
    return nk.make_manual_basis(out), ctr


@pytest.mark.parametrize("npts", [1, 63, 64, 65, 200])
@pytest.mark.parametrize("nbf", [1, 8, 9, 31, 32, 33, 70])
def test_collocation(nbf, npts):
    rng = np.random.default_rng(100 * nbf + npts)
    basis, ctr = _basis(nbf, rng)
    pts = ctr[rng.integers(0, 4, npts)] + rng.normal(size=(npts, 3)) * 1.5
    if npts > 3:
        pts[1], pts[2] = ctr[0], 300.0  # at a nucleus; far from all
    print(f"{nbf} functions, {npts} points", flush=True)
    c = nk.Context(0)
    try:
        p = torch.tensor(pts, device="cuda")
        got = [api.fill_collocation(c, basis, p), *api.fill_grad_collocation(c, basis, p)]
        ref = O.collocation(basis_dict(basis), pts, grad=True)
        for k, (a, b) in enumerate(zip(got, ref)):
            a = a.cpu().numpy()
            ok = np.isfinite(b) if k else np.ones_like(b, bool)  # no gradient at a nucleus
            assert np.abs(a - b)[ok].max() <= 1e-13 * max(np.abs(b[ok]).max(), 1e-30)
    finally:
        c.close()


@pytest.mark.parametrize("nbf,npts", [(1, 16321), (15, 16385), (16, 16384), (17, 16447),
                                      (33, 130001), (70, 130001)])
def test_collocation_tile_widths(nbf, npts):
    """Tiles of 16 functions (from 256 blocks of points) and 32 (above 64 MB)."""
    test_collocation(nbf, npts)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-7), ("mixed", 5e-7)])
def test_gradient_with_f_functions(precision, tol):
    rng = np.random.default_rng(8)
    xyz, Z = np.array([[0.0, 0.1, 0.0], [0.0, 1.5, 1.1]]), np.array([8, 1], np.int32)
    shells = [(0, n, l, z) for n, l, z in ((1, 0, 7.0), (2, 0, 2.0), (2, 1, 2.2), (3, 2, 1.8),
                                           (4, 3, 2.0), (5, 3, 1.7))] + [(1, 1, 0, 1.1), (1, 2, 1, 1.3)]
    fn = lambda x: nk.make_manual_basis([(n, l, m, z, *x[a]) for a, n, l, z in shells
                                         for m in range(-l, l + 1)])
    nbf = fn(xyz).nbf()
    C = np.linalg.qr(rng.normal(size=(nbf, 5)))[0]
    P = torch.tensor(2 * C @ C.T, device="cuda")
    c = nk.Context(0)

    def energy(x):
        c.make_flat_grid(x, Z, nrad=40, nang_order=21)
        c.set_basis(fn(x))
        return c.vxc(P, funcs=(101, 130)).energy

    try:
        h = 2e-3
        E = {}
        for k in (0, 4, 5):
            d = np.zeros(6)
            d[k] = h
            d = d.reshape(2, 3)
            E[k] = (8 * (energy(xyz + d) - energy(xyz - d)) -
                    (energy(xyz + 2 * d) - energy(xyz - 2 * d))) / (12 * h)
        energy(xyz)
        _, g = c.xc_grad(P, funcs=(101, 130), precision=precision)
        for k, v in E.items():
            assert abs(g.reshape(-1)[k] - v) <= tol, (k, g.reshape(-1)[k], v)
    finally:
        c.close()
