"""Points and functions that do not meet: no live batch (E, N, V and the gradient
are zero, the density too), and live batches of one, two and three blocks of five
beside others without (against the reference-shaped path)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402
from nukexc_amd import api  # noqa: E402

FN = (101, 130)


def _setup(c, centers, where, n):
    """63 functions of one radius class a centre (one block a centre, about), n
    points around each of the places."""
    rng = np.random.default_rng(n)
    f = [(3, l, m, 1.5 + 0.01 * k, *x) for x in centers for k in range(7) for l in range(3)
         for m in range(-l, l + 1)]
    pts = np.concatenate([x + rng.normal(size=(n, 3)) for x in where])
    w = torch.tensor(rng.uniform(0.1, 1.0, len(pts)), device="cuda")
    pts = torch.tensor(pts, device="cuda")
    b = nk.make_manual_basis(f)
    c.set_grid(nk.FlatGrid(pts, w, torch.tensor(centers, device="cuda"),
                           np.full(len(centers), 8, np.int32),
                           torch.zeros(len(pts), dtype=torch.int32, device="cuda")))
    c.set_basis(b)
    C = np.linalg.qr(rng.normal(size=(b.nbf(), 4)))[0]
    return b, pts, w, C, torch.tensor(C @ C.T, device="cuda")


@pytest.fixture
def ctx():
    c = nk.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_nothing_live(ctx, precision):
    centers = np.array([[0.0, 0.0, 0.0], [3.0, 0.0, 0.0]])
    _, _, _, _, P = _setup(ctx, centers, [np.full(3, 5000.0)], 300)
    assert ctx.plan_stats()["pairs_kept"] == 0
    for fn in ((1,), FN):
        r = ctx.vxc(P, funcs=fn, precision=precision)
        assert r.energy == 0.0 and r.n_el == 0.0 and not r.potential.any()
        r = ctx.vxc_polarized(P, P, funcs=fn, precision=precision)
        assert r.energy == 0.0 and not r.potential_alpha.any() and not r.potential_beta.any()
        E, g = ctx.xc_grad(P, funcs=fn, partition="fixed", precision=precision)
        assert E == 0.0 and not g.any()
    assert not ctx.overlap().any()


@pytest.mark.parametrize("apart", [300.0, 12.0])
@pytest.mark.parametrize("places", [1, 3, 5])
def test_some_live(ctx, places, apart):
    centers = np.zeros((5, 3))
    centers[:, 0] = apart * np.arange(5)
    far = [np.full(3, -4000.0)]
    b, pts, w, C, P = _setup(ctx, centers, far + list(centers[:places]), 500)
    print(ctx.plan_stats(), flush=True)
    M = [nk.fill_collocation(ctx, b, pts), *nk.fill_grad_collocation(ctx, b, pts)]
    ref = api.compute_gga(ctx, *M, w, C, np.ones(4), FN)
    r = ctx.vxc(P, funcs=FN)
    # 2 500 terms a sum and the screening tolerance of 1e-12
    assert abs(r.energy - ref.energy) <= 1e-10 * abs(ref.energy)
    assert (r.potential - ref.potential).abs().max() <= 1e-10 * ref.potential.abs().max()
