"""The reference-shaped XC calls through the C ABI with nothing to sum: no points,
or no orbitals (a negative count of the closed-shell call is none).  E is zero
and V is all zeros, for each width of the V tiles (32, 64, 128 functions).  A
spin without orbitals beside one that has some gives the other what it gets
beside a spin of zero occupation."""
import ctypes

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402
from nukexc_amd import _capi  # noqa: E402
from nukexc_amd.api import _ids, _ptr  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    c = nk.Context(0)
    yield c
    c.close()


def _call(ctx, nbf, npts, nocc, funcs):
    """E and V per spin; nocc: orbitals per spin (one entry: closed shell).  Every
    pointer is valid, whatever the counts."""
    gga = funcs[0] > 100
    rng = torch.Generator(device="cuda").manual_seed(nbf)
    new = lambda n: torch.rand(max(1, n), dtype=torch.float64, device="cuda", generator=rng)
    m = [new(nbf * npts) for _ in range(4 if gga else 1)] + [None] * (0 if gga else 3)
    w, orb = new(npts), []
    keep = []
    for k in nocc:
        C, f = new(nbf * abs(k)), new(abs(k))
        keep += [C, f]
        orb += [k, _ptr(C), _ptr(f)]
    V = [torch.full((nbf, nbf), float("nan"), dtype=torch.float64, device="cuda") for _ in nocc]
    E = ctypes.c_double(float("nan"))
    ids, nf = _ids(funcs)
    L = _capi.lib()
    call = L.nkx_xc_from_collocation if len(nocc) == 1 else L.nkx_xc_from_collocation_polarized
    _capi.check(call(ctx.h, nbf, npts, *[_ptr(x) for x in m], _ptr(w), *orb, nf, ids,
                     _capi.FAMILY_GGA if gga else _capi.FAMILY_LDA, ctypes.byref(E),
                     *[_ptr(v) for v in V]), ctx.h)
    return E.value, V


@pytest.mark.parametrize("funcs", [(1, 12), (101, 130)])
@pytest.mark.parametrize("nocc", [(3,), (3, 2)])
@pytest.mark.parametrize("nbf", [5, 40, 70, 130])
def test_no_points(ctx, nbf, nocc, funcs):
    print(f"{nbf} functions, no points, {nocc}, {funcs}", flush=True)
    E, V = _call(ctx, nbf, 0, nocc, funcs)
    assert E == 0.0 and all(not v.any() for v in V)


@pytest.mark.parametrize("funcs", [(1, 12), (101, 130)])
@pytest.mark.parametrize("nocc", [(0,), (-1,), (-16,), (-31,), (-1000,), (0, 0)])
@pytest.mark.parametrize("nbf", [5, 40, 70, 130])
def test_no_orbitals(ctx, nbf, nocc, funcs):
    print(f"{nbf} functions, {nocc} orbitals, {funcs}", flush=True)
    E, V = _call(ctx, nbf, 200, nocc, funcs)
    assert E == 0.0 and all(not v.any() for v in V)


@pytest.mark.parametrize("nbf", [5, 40, 70])
@pytest.mark.parametrize("empty", [0, 1])
@pytest.mark.parametrize("other", [3, 18])
def test_one_spin_without_orbitals(ctx, nbf, empty, other):
    """Against one orbital of zero occupation, which reads and sums the same
    numbers: equal to the order of the sums, at most 18 orbitals of 70 functions
    (1e-13 of the largest element)."""
    print(f"{nbf} functions, spin {empty} empty, {other} orbitals", flush=True)
    n = 300
    rng = torch.Generator(device="cuda").manual_seed(nbf)
    new = lambda *s: torch.randn(*s, dtype=torch.float64, device="cuda", generator=rng)
    m, w = [new(n, nbf) for _ in range(4)], new(n).abs()
    C, f = new(other, nbf) / nbf ** 0.5, new(other).abs()
    zC, zf = new(1, nbf), torch.zeros(1, dtype=torch.float64, device="cuda")
    res = []
    for k in (0, 1):
        none = [k, _ptr(zC if k else None), _ptr(zf if k else None)]
        orb = [none, [other, _ptr(C), _ptr(f)]]
        V = [torch.empty(nbf, nbf, dtype=torch.float64, device="cuda") for _ in range(2)]
        E = ctypes.c_double()
        ids, nf = _ids((101, 130))
        torch.cuda.synchronize()
        _capi.check(_capi.lib().nkx_xc_from_collocation_polarized(
            ctx.h, nbf, n, *[_ptr(x) for x in m], _ptr(w), *orb[empty], *orb[1 - empty], nf, ids,
            _capi.FAMILY_GGA, ctypes.byref(E), *[_ptr(v) for v in V]), ctx.h)
        res.append((E.value, V))
    (E0, V0), (E1, V1) = res
    assert abs(E0 - E1) <= 1e-13 * abs(E1)
    for a, b in zip(V0, V1):
        assert torch.isfinite(a).all()
        assert (a - b).abs().max() <= 1e-13 * max(1.0, b.abs().max().item())
