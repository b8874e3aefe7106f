"""Builds in several chunks (a small tile-store budget) against the same build in
one: every form, closed and open shell, one molecule and a set whose chunks hold
some of its molecules only, split counts given and automatic.  The numbers are
the same and only the order of the sums over batches differs: 1e-12 (the split-
bf16 form sums in FP32 inside a chunk: 1e-6)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402
from nukexc_amd import configs  # noqa: E402

FN = (101, 130)


def _molecule(n, seed):
    rng = np.random.default_rng(seed)
    xyz, Z = configs.random_walk_molecule(n, rng)
    basis = nk.make_manual_basis(configs.sto_functions(Z, xyz, rng))
    P = []
    for _ in range(2):
        C = np.linalg.qr(rng.normal(size=(basis.nbf(), 6)))[0]
        P.append(torch.tensor(C @ C.T, device="cuda"))
    return dict(xyz=xyz, Z=Z, basis=basis), P


def _near(a, b, tol):
    assert abs(a.energy - b.energy) <= tol * abs(b.energy)
    for k in ("potential", "potential_alpha", "potential_beta"):
        if hasattr(b, k):
            assert (getattr(a, k) - getattr(b, k)).abs().max() <= tol * getattr(b, k).abs().max()


@pytest.mark.parametrize("split", [0, 1, 5, 16])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-12), ("mixed_bf16", 1e-6)])
@pytest.mark.parametrize("natoms", [6, 24])
def test_one_molecule(natoms, precision, tol, split):
    m, P = _molecule(natoms, natoms)
    c = nk.Context(0)
    try:
        c.make_flat_grid(m["xyz"], m["Z"], nrad=60, nang_order=17)
        c.set_basis(m["basis"])
        c.set_launch(split, 0)
        res = []
        for budget in (0, 64 << 20):
            print(f"{natoms} atoms {precision} split {split} budget {budget}", flush=True)
            c.set_memory_budget(budget)
            res.append([c.vxc(P[0], funcs=FN, precision=precision)])
            if precision != "mixed_bf16":
                res[-1].append(c.vxc_polarized(*P, funcs=FN, precision=precision))
        for a, b in zip(res[1], res[0]):
            _near(a, b, tol)
    finally:
        c.close()


@pytest.mark.parametrize("split", [0, 3])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_molecule_set(precision, split):
    mols, Ps = zip(*[_molecule(n, n) for n in (2, 14, 3, 9, 20)])
    Ps = [p[0] for p in Ps]
    c = nk.Context(0)
    try:
        c.molset_create(list(mols), nrad=40, nang_order=17)
        c.set_launch(split, 0)
        res = []
        for budget in (0, 64 << 20):
            print(f"set {precision} split {split} budget {budget}", flush=True)
            c.set_memory_budget(budget)
            res.append(c.molset_vxc(Ps, funcs=FN, precision=precision))
        for a, b in zip(res[1], res[0]):
            _near(a, b, 1e-12)
    finally:
        c.close()
