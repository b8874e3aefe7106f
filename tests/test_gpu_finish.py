"""The end of a build (sum of the split partials, un-permutation, mirror, E
and N) over split counts around its load groups and segments, with one and
two function blocks, against the FP64 oracle.  V sums 13 180 or more points of
magnitude <= 1e2 in FP64, so 1e-11 leaves room for any order of the sums."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from gpu_util import basis_dict, orbitals_on_grid  # noqa: E402
import nukexc_amd as nk  # noqa: E402
from nukexc_amd import configs  # noqa: E402
from oracle import oracle as O  # noqa: E402


@pytest.fixture(scope="module", params=["water", "benzene"])
def case(request):
    w = configs.workload(request.param)
    c = nk.Context(0)
    grid = c.make_flat_grid(w["xyz"], w["Z"], nrad=30, nang_order=17)
    c.set_basis(w["basis"])
    pts, wts = grid.quad_points.cpu().numpy(), grid.weights.cpu().numpy()
    _, _, P = orbitals_on_grid(w, pts, wts)
    phi, gx, gy, gz = O.collocation(basis_dict(w["basis"]), pts, grad=True)
    ref = O.vxc_from_collocation(phi, wts, (101, 130), P=P, gx=gx, gy=gy, gz=gz)
    yield c, torch.tensor(P, device="cuda"), ref
    c.close()


@pytest.mark.parametrize("split", [1, 2, 3, 4, 5, 15, 63, 64, 65, 67, 100000])
def test_split_counts(case, split):
    c, P, (E0, N0, V0) = case
    print(f"split {split}", flush=True)
    c.set_launch(vgemm_split=split)
    try:
        r = c.vxc(P, funcs=(101, 130), precision="fp64")
    finally:
        c.set_launch()
    assert abs(r.energy - E0) <= 1e-11 * abs(E0) and abs(r.n_el - N0) <= 1e-11 * N0
    assert np.abs(r.potential.cpu().numpy() - V0).max() <= 1e-11
