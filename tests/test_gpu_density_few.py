"""compute_density[_and_sigma] of one to nine functions (up to eight have a kernel of
their own, a point per thread), around its workgroups of 256 points, the matrices
at 8-byte alignment inside a buffer of NaN, against plain FP64 sums of at most 9
functions and 33 orbitals: 1e-13 of the largest element."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402
from nukexc_amd import api  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    c = nk.Context(0)
    yield c
    c.close()


def _matrix(a):
    nbf, n = a.shape
    buf = torch.full((nbf * n + 40,), float("nan"), dtype=torch.float64, device="cuda")
    v = buf[1:1 + nbf * n].view(n, nbf)
    v.copy_(torch.tensor(np.ascontiguousarray(a.T)))
    return v.t()


@pytest.mark.parametrize("nocc", [1, 3, 33])
@pytest.mark.parametrize("n", [1, 255, 256, 257, 5000])
@pytest.mark.parametrize("nbf", range(1, 10))
def test_few_functions(ctx, nbf, n, nocc):
    rng = np.random.default_rng(100 * nbf + nocc)
    m = [rng.normal(size=(nbf, n)) for _ in range(4)]
    C, f = rng.normal(size=(nbf, nocc)) / nbf ** 0.5, rng.uniform(0.5, 2.0, nocc)
    psi = [C.T @ x for x in m]
    rho = (f[:, None] * psi[0] ** 2).sum(0)
    gr = [2 * (f[:, None] * psi[0] * p).sum(0) for p in psi[1:]]
    d = [_matrix(x) for x in m]

    def near(got, ref):
        got = got.cpu().numpy()
        assert np.abs(got - ref).max() <= 1e-13 * np.abs(ref).max()

    near(api.compute_density(ctx, d[0], C, f), rho)
    r, g, s = api.compute_density_and_sigma(ctx, *d, C, f)
    near(r, rho)
    near(s, sum(x * x for x in gr))
    for x, y in zip(g, gr):
        near(x, y)
