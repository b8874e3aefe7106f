"""The FP64 V contraction by super-pairs (blocks live together) and by single pairs
(centres apart: few super-pairs are whole), over split counts below, at and
between multiples of eight, closed and open shell, in one chunk and in several,
against the reference-shaped path on the same points.  Sums of 40 000 terms in
another order: 1e-11 of the largest element."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402
from nukexc_amd import api  # noqa: E402

FN = (101, 130)


@pytest.fixture(scope="module", params=[(7, 200.0), (7, 6.0), (2, 200.0), (3, 200.0), (5, 1.5)],
                ids=lambda p: f"{p[0]}x{p[1]}")
def case(request):
    natoms, apart = request.param
    rng = np.random.default_rng(natoms)
    xyz = np.zeros((natoms, 3))
    xyz[:, 0] = apart * np.arange(natoms)
    # 60 functions of one radius class a centre: blocks of neighbouring centres
    f = [(3, l, m, 1.5 + 0.01 * k, *x) for x in xyz for k in range(7) for l in range(3)
         for m in range(-l, l + 1)][:]
    f = [g for i, g in enumerate(f) if i % 63 < 60]
    c = nk.Context(0)
    grid = c.make_flat_grid(xyz, np.full(natoms, 8, np.int32), nrad=60, nang_order=17)
    b = nk.make_manual_basis(f)
    c.set_basis(b)
    c.set_screening(1e-18)
    pts, w = grid.quad_points, grid.weights
    M = [nk.fill_collocation(c, b, pts), *nk.fill_grad_collocation(c, b, pts)]
    C = [np.linalg.qr(rng.normal(size=(b.nbf(), k)))[0] for k in (4, 3)]
    o = [rng.uniform(0.5, 1.0, k) for k in (4, 3)]
    closed = api.compute_gga(c, *M, w, C[0], o[0], FN)
    opened = api.compute_gga_lsda(c, *M, w, C[0], o[0], C[1], o[1], FN)
    P = [torch.tensor(x @ np.diag(y) @ x.T, device="cuda") for x, y in zip(C, o)]
    yield c, P, closed, opened
    c.close()


def _near(V, ref):
    assert (V - ref).abs().max().item() <= 1e-11 * ref.abs().max().item()


@pytest.mark.parametrize("budget", [0, 64 << 20])
@pytest.mark.parametrize("split", [0, 1, 3, 8, 13, 25, 64])
def test_split_counts(case, split, budget):
    c, P, closed, opened = case
    print(f"split {split}, budget {budget}, {c.plan_stats()}", flush=True)
    c.set_launch(split, 0)
    c.set_memory_budget(budget)
    r = c.vxc(P[0], funcs=FN)
    assert abs(r.energy - closed.energy) <= 1e-11 * abs(closed.energy)
    _near(r.potential, closed.potential)
    r = c.vxc_polarized(*P, funcs=FN)
    assert abs(r.energy - opened.energy) <= 1e-11 * abs(opened.energy)
    _near(r.potential_alpha, opened.potential_alpha)
    _near(r.potential_beta, opened.potential_beta)
