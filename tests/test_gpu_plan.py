"""The launch plan built on the device against the same plan in numpy: batches of
64 points along the Morton curve, live (function block, batch) pairs of the
screening radii, and the algorithmic work, all exact; point counts around a
batch, one point, coincident points, one to three function blocks."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402
from nukexc_amd import api, configs  # noqa: E402


def _spread(v):
    v = v.astype(np.uint64) & np.uint64(0x1FFFFF)
    for s, m in ((32, 0x1F00000000FFFF), (16, 0x1F0000FF0000FF), (8, 0x100F00F00F00F00F),
                 (4, 0x10C30C30C30C30C3), (2, 0x1249249249249249)):
        v = (v | (v << np.uint64(s))) & np.uint64(m)
    return v


def _codes(p, lo, hi):
    t = np.clip((p - lo) / np.maximum(hi - lo, 1e-12), 0.0, 1.0)
    q = (t * 2097151.0).astype(np.uint64)
    return _spread(q[:, 0]) | (_spread(q[:, 1]) << np.uint64(1)) | (_spread(q[:, 2]) << np.uint64(2))


def _plan(pts, basis, tol):
    order = np.argsort(_codes(pts, pts.min(0), pts.max(0)), kind="stable")
    nb = -(-len(pts) // 64)
    order = np.concatenate([order, np.full(nb * 64 - len(pts), order[-1])])
    box = pts[order].reshape(nb, 64, 3)
    lo, hi = box.min(1), box.max(1)
    rad = np.array([api.sto_norm_cutoff(n, z, tol)[1] for n, z in zip(basis.n, basis.zeta)])
    O = np.asarray(basis.O)
    cls = np.floor(2 * np.log2(np.maximum(rad, 0.25))).astype(int)
    key = sorted(zip(cls, _codes(O, O.min(0), O.max(0)).tolist(), range(len(rad))))
    perm = np.array([k[2] for k in key])
    e = np.maximum(np.maximum(lo[:, None] - O[perm], O[perm] - hi[:, None]), 0.0)
    d2 = (e[..., 0] * e[..., 0] + e[..., 1] * e[..., 1]) + e[..., 2] * e[..., 2]
    hit = d2 < rad[perm] ** 2
    nf = -(-len(rad) // 64)
    live = np.stack([hit[:, 64 * f:64 * f + 64].any(1) for f in range(nf)], 1)
    size = np.array([min(len(rad), 64 * f + 64) - 64 * f for f in range(nf)])
    g = np.minimum(64, len(pts) - 64 * np.arange(nb))
    nfun = (live * size).sum(1)
    return nb, int(live.sum()), nb * nf, float((nfun * g).sum()), float((nfun ** 2 * g).sum())


@pytest.mark.parametrize("natoms,spread", [(2, 1.0), (9, 4.0), (20, 12.0)])
@pytest.mark.parametrize("npts", [1, 63, 64, 65, 1000, 20011])
def test_plan_matches_host(npts, natoms, spread):
    rng = np.random.default_rng(npts + natoms)
    xyz, Z = configs.random_walk_molecule(natoms, rng)
    basis = nk.make_manual_basis(configs.sto_functions(Z, xyz, rng))
    pts = xyz[rng.integers(0, natoms, npts)] + rng.normal(size=(npts, 3)) * spread
    if npts > 500:
        pts[200:300] = pts[199]  # coincident points, whose order is the grid's
    c = nk.Context(0)
    try:
        c.set_grid(nk.FlatGrid(torch.tensor(pts, device="cuda"),
                               torch.full((npts,), 0.01, dtype=torch.float64, device="cuda"),
                               torch.tensor(xyz, device="cuda"), Z,
                               torch.zeros(npts, dtype=torch.int32, device="cuda")))
        c.set_basis(basis)
        for tol in (1e-12, 1e-4):
            print(f"{npts} points, {basis.nbf()} functions, tol {tol}", flush=True)
            c.set_screening(tol)
            nb, kept, total, nbg, nb2g = _plan(pts, basis, tol)
            st, wk = c.plan_stats(), c.plan_work()
            assert st == dict(npts=npts, npts_padded=64 * nb, nbatches=nb, pairs_kept=kept,
                              pairs_total=total)
            assert wk["colloc_elems"] == nbg and wk["flops_v"] == 2 * nb2g
    finally:
        c.close()
