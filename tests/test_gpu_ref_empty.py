"""The reference-shaped XC calls through the C ABI with nothing to sum: no points.
E is zero and V is all zeros, for each width of the V tiles (32, 64, 128
functions)."""
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
        C, f = new(nbf * k), new(k)
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
