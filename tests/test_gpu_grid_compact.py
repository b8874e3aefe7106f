"""The grid build's compaction from one point to more blocks of 1024 points than
one pass of its scan takes (1024) and than its scratch is kept for (4 M points),
on one context, large ones before small ones, against the oracle's order."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402
from oracle import oracle as O  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    c = nk.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("natoms,nrad,order", [(9, 80, 131), (1, 1, 3), (4, 220, 59),
                                               (12, 110, 53), (2, 11, 11), (3, 40, 17)])
def test_order_and_weights(ctx, natoms, nrad, order):
    rng = np.random.default_rng(natoms)
    xyz = rng.normal(size=(natoms, 3)) * 3.0 * natoms ** (1 / 3)
    Z = rng.choice([1, 6, 8], natoms).astype(np.int32)
    print(f"{natoms} atoms, {nrad} shells, order {order}", flush=True)
    g = ctx.make_flat_grid(xyz, Z, nrad=nrad, nang_order=order)
    P, W, own = O.make_flat_grid(xyz, Z, nrad, nk.lebedev_rule(order))
    assert g.weights.shape[0] == len(W)
    assert np.array_equal(g.point_owner.cpu().numpy(), own)
    assert np.abs(g.quad_points.cpu().numpy() - P).max() <= 1e-11 * np.abs(P).max()
    assert np.abs(g.weights.cpu().numpy() - W).max() <= 1e-11 * np.abs(W).max()
