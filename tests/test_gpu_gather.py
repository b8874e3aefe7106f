"""Density matrices of a molecule set gathered together: counts around the 32 of
one launch, molecules of different sizes in one launch, against the molecules
built one at a time (same arithmetic: 1e-12)."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402
from nukexc_amd import configs  # noqa: E402

GRID = dict(nrad=12, nang_order=7)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 50])
def test_set_against_single_builds(n, precision):
    c = nk.Context(0)
    try:
        mols, rng = configs.molset(64, 3)
        mols = [m for m in mols if len(m["Z"]) <= 14][:4] * 13
        mols = mols[:n]
        Ps = []
        for m in mols:
            a = torch.tensor(rng.normal(size=(m["basis"].nbf(), 3)), device="cuda") * 0.1
            Ps.append(a @ a.t())
        c.molset_create(mols, **GRID)
        res = c.molset_vxc(Ps, funcs=(101, 130), precision=precision)
        print(f"{n} molecules, {precision}", flush=True)
        for k in sorted({0, 1 % n, n // 2, n - 1}):
            c.make_flat_grid(mols[k]["xyz"], mols[k]["Z"], **GRID)
            c.set_basis(mols[k]["basis"])
            one = c.vxc(Ps[k], funcs=(101, 130), precision=precision)
            assert abs(res[k].energy - one.energy) <= 1e-11 * max(1.0, abs(one.energy)), k
            assert (res[k].potential - one.potential).abs().max().item() <= 1e-12, k
    finally:
        c.close()
