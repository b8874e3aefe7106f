"""Derivative of the Becke weights around the number of cell functions taken
together (4) and kept (16): clusters where every atom is near every point and
chains longer than the 5 bohr cap, both partitions, a directional derivative
against fourth-order differences of the FP64 energy with the oracle's weights.
Differences at h = 5e-4 bohr carry h^4 / 30 of a fifth derivative and 1e-12 / h,
below 1e-7 of the gradient's size."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402
from oracle import oracle as O  # noqa: E402


@pytest.mark.parametrize("shape", ["cluster", "chain"])
@pytest.mark.parametrize("capped", [True, False])
@pytest.mark.parametrize("n", [1, 2, 4, 5, 16, 17, 22])
def test_directional(n, capped, shape):
    rng = np.random.default_rng(10 * n + capped)
    if shape == "cluster":
        q = np.stack(np.meshgrid(*[np.arange(3.0)] * 3), -1).reshape(-1, 3)[:n]
        xyz = 1.5 * q + rng.uniform(-0.15, 0.15, (n, 3))
    else:
        xyz = np.outer(np.arange(n), [1.9, 0.4, 0.0]) + rng.uniform(-0.2, 0.2, (n, 3))
    own = np.repeat(np.arange(n), 90).astype(np.int32)
    off = rng.normal(size=(len(own), 3))
    off *= (rng.uniform(0.05, 4.0, len(own)) / np.linalg.norm(off, axis=1))[:, None]
    w0 = rng.uniform(0.5, 1.5, len(own)) / 90
    A = rng.normal(size=(n, n))
    P = torch.tensor(A @ A.T / n + np.eye(n), device="cuda")
    v = rng.normal(size=(n, 3))

    def energy(c, t, grad=False):
        X = xyz + t * v
        pts = X[own] + off
        g = nk.FlatGrid(torch.tensor(pts, device="cuda"),
                        torch.tensor(O.becke(X, pts, own, w0, capped), device="cuda"),
                        torch.tensor(X, device="cuda"), np.ones(n, np.int32),
                        torch.tensor(own, device="cuda"))
        c.set_grid(g)
        c.set_basis(nk.make_manual_basis([(1, 0, 0, 1.2, *x) for x in X]))
        if grad:
            return c.xc_grad(P, funcs=(101, 130),
                             partition="becke_capped" if capped else "becke")[1]
        return c.vxc(P, funcs=(101, 130), precision="fp64").energy

    print(f"{n} atoms, {shape}, capped {capped}", flush=True)
    c = nk.Context(0)
    try:
        g = energy(c, 0.0, grad=True)
        h = 5e-4
        e = [energy(c, t * h) for t in (2, 1, -1, -2)]
    finally:
        c.close()
    fd = (-e[0] + 8 * e[1] - 8 * e[2] + e[3]) / (12 * h)
    an = float((g * v).sum())
    assert abs(an - fd) <= 1e-7 * max(1.0, np.abs(g).max() * np.sqrt(3 * n)), (an, fd)
    assert np.abs(g.sum(0)).max() <= 1e-10 * max(1.0, np.abs(g).max())
