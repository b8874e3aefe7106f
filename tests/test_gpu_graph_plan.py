"""A captured build is tied to the launch plan that it was captured on: a plan
made in between, with the settings back at the capture's, refuses the replay;
settings that came and went without a plan, and a molecule set that was refused
before its plan was begun, leave the replay as it was."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402
from nukexc_amd import configs  # noqa: E402


@pytest.fixture
def ctx():
    c = nk.Context(0)
    yield c
    c.close()


def _molecule(n, seed):
    rng = np.random.default_rng(seed)
    xyz, Z = configs.random_walk_molecule(n, rng)
    basis = nk.make_manual_basis(configs.sto_functions(Z, xyz, rng))
    C = np.linalg.qr(rng.normal(size=(basis.nbf(), 4)))[0]
    return xyz, Z, basis, torch.tensor(2 * C @ C.T, device="cuda")


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("other", [1e-4, 1e-15])
def test_plan_made_in_between(ctx, precision, other):
    xyz, Z, basis, P = _molecule(9, 5)
    ctx.make_flat_grid(xyz, Z, nrad=25, nang_order=17)
    ctx.set_basis(basis)
    V = torch.empty_like(P)
    kw = dict(funcs=(101, 130), precision=precision)
    for back in (False, True):  # with and without a plan of the first settings again
        ctx.set_screening(1e-10)
        E0 = ctx.vxc(P, **kw).energy
        ctx.graph_capture(P, V, **kw)
        assert abs(ctx.graph_launch()[0] - E0) <= 1e-12 * abs(E0)
        ctx.set_screening(other)  # no plan made: the replay stands
        ctx.set_screening(1e-10)
        assert abs(ctx.graph_launch()[0] - E0) <= 1e-12 * abs(E0)
        ctx.set_screening(other)
        ctx.vxc(P, **kw)
        ctx.set_screening(1e-10)
        if back:
            ctx.vxc(P, **kw)
        with pytest.raises(nk.NukexcError) as ei:
            ctx.graph_launch()
        assert ei.value.status == "NKX_ERR_STATE"


def test_refused_molecule_set(ctx):
    mols = [_molecule(n, 10 + n) for n in (3, 5)]
    Ps = [m[3] for m in mols]
    mols = [dict(zip(("xyz", "Z", "basis"), m)) for m in mols]
    Vs = [torch.empty_like(p) for p in Ps]
    ctx.molset_create(mols, nrad=20, nang_order=17)
    r = ctx.molset_vxc(Ps, funcs=(101, 130), precision="mixed")
    ctx.molset_graph_capture(Ps, Vs, funcs=(101, 130), precision="mixed")
    with pytest.raises(nk.NukexcError):  # no point is heavy enough
        ctx.molset_create(mols[::-1], nrad=20, nang_order=17,
                          weight_threshold=1e30)
    E = ctx.molset_graph_launch()[0]
    for e, v, x in zip(E, Vs, r):
        assert abs(e - x.energy) <= 1e-12 * abs(x.energy)
        assert (v - x.potential).abs().max() <= 1e-13
