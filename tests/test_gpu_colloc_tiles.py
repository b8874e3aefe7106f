"""Reference-shaped collocation on both sides of the borders between its tile
shapes (64 MB of output, 256 groups of 64 points) and between numbers of
workgroups to a group (2048 over the groups), values and gradients, against the
same points in pieces of 4 000, which take the narrowest tiles: the same bits."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402


@pytest.mark.parametrize("nbf,npts", [(3100, 4100), (1037, 10000), (1037, 8000), (120, 65536),
                                      (120, 65537), (120, 131072), (120, 131073), (61, 150000),
                                      (45, 200001)])
def test_pieces(nbf, npts):
    rng = np.random.default_rng(nbf)
    f = []
    while len(f) < nbf:
        x, z = rng.normal(size=3) * 3, rng.uniform(0.5, 2.0)
        f += [(l + 1, l, m, z, *x) for l in range(4) for m in range(-l, l + 1)]
    b = nk.make_manual_basis(f[:nbf])
    pts = torch.tensor(rng.normal(size=(npts, 3)) * 4, device="cuda")
    c = nk.Context(0)
    try:
        print(f"{nbf} functions, {npts} points", flush=True)
        whole = [nk.fill_collocation(c, b, pts), *nk.fill_grad_collocation(c, b, pts)]
        for i in range(0, npts, 4000):
            p = pts[i:i + 4000]
            part = [nk.fill_collocation(c, b, p), *nk.fill_grad_collocation(c, b, p)]
            for w, x in zip(whole, part):
                assert torch.equal(w[:, i:i + 4000], x)
    finally:
        c.close()
