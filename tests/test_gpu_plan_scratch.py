"""Scratch of a plan's construction: given back after a large plan (what stays is
the plan itself, 36 bytes a point and 12 a batch), while small plans after it and
a second large one come out right."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import nukexc_amd as nk  # noqa: E402


def test_large_plan_gives_scratch_back():
    n = 8_000_000
    b = nk.make_manual_basis([(1, 0, 0, 1.0, 0.0, 0.0, 0.0), (2, 1, 0, 1.2, 0.0, 0.0, 0.0)])
    c = nk.Context(0)

    def grid(m):
        g = torch.Generator(device="cuda").manual_seed(m)
        pts = torch.randn(m, 3, dtype=torch.float64, device="cuda", generator=g)
        c.set_grid(nk.FlatGrid(pts, torch.full((m,), 1.0 / m, dtype=torch.float64, device="cuda"),
                               torch.zeros(1, 3, dtype=torch.float64, device="cuda"),
                               np.ones(1, np.int32),
                               torch.zeros(m, dtype=torch.int32, device="cuda")))
        return pts

    try:
        c.set_basis(b)
        pts = grid(1000)
        P = torch.eye(2, dtype=torch.float64, device="cuda")
        small = c.vxc(P).energy
        pts = grid(n)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        st = c.plan_stats()
        held = free - torch.cuda.mem_get_info()[0]
        print(f"{held / n:.1f} bytes a point")
        assert st["nbatches"] == n // 64 and st["pairs_kept"] == n // 64
        assert held <= 40 * n + (32 << 20)
        phi = nk.fill_collocation(c, b, pts)
        ref = (phi * phi).sum().item() / n
        for tol in (1e-12, 1e-10):  # the second plan allocates the scratch again
            c.set_screening(tol)
            assert abs(c.vxc(P).n_el - ref) <= 1e-10 * ref
        grid(1000)
        c.set_screening(1e-12)
        assert abs(c.vxc(P).energy - small) <= 1e-13 * abs(small)
    finally:
        c.close()
