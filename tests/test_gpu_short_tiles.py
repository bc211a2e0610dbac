"""Four-row tiles of the scalar RK4 kernels, and the multi-step kernel on grids whose last strip or band is
narrower than the 4-cell halo, where a tile also waits for the tile behind its neighbour.

Bar: bitwise equal to 16-row tiles launched step by step (the arithmetic does not depend on the tile)."""
import numpy as np
import pytest

from test_gpu_flow import solver

pytestmark = pytest.mark.gpu

# 56 k + 1 .. 3 columns and ty k + 1 .. 3 rows: narrow last tiles; 58 x 10: two strips, and at 8 rows two bands
SHAPES = [(58, 10, 8), (58, 18, 16), (114, 62, 4), (170, 41 * 2, 10), (226, 130, 16), (60, 6, 4), (112, 64, 4)]


def run(monkeypatch, prec, shape, bc, pot, flow, ty, steps=41):
    monkeypatch.setenv("PHX_RK4_FLOW", flow)
    monkeypatch.setenv("PHX_RK4_TY", str(ty))
    s = solver(prec, shape[0], shape[1], bc, pot, 23)
    assert s.step(steps) == steps
    out = s.get("psi_plus"), s.get("n_plus"), s.info["multi_step_steps"]
    s.close()
    return out


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("bc,pot", [("periodic", False), ("zero", True)])
@pytest.mark.parametrize("N_c,N_r,ty", SHAPES)
def test_narrow_last_tiles(monkeypatch, N_c, N_r, ty, bc, pot, prec):
    print(f"[short tiles] {N_c}x{N_r} ty={ty} {bc} {prec}", flush=True)
    psi, n, _ = run(monkeypatch, prec, (N_c, N_r), bc, pot, "0", 16)
    p1, n1, multi = run(monkeypatch, prec, (N_c, N_r), bc, pot, "1", ty)
    assert multi == 40
    assert np.array_equal(p1, psi) and np.array_equal(n1, n)
    p4, n4, _ = run(monkeypatch, prec, (N_c, N_r), bc, pot, "0", 4)
    assert np.array_equal(p4, psi) and np.array_equal(n4, n)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("N_c,N_r", [(1, 1), (3, 5), (57, 9), (200, 150), (511, 300)])
def test_device_steps_do_not_depend_on_the_tile(monkeypatch, N_c, N_r, prec):
    """rk4_scalar_device picks its tile height by the size of the grid (odd sizes included)"""
    import torch
    from phoenix_amd import _lib
    print(f"[short tiles, device] {N_c}x{N_r} {prec}", flush=True)
    g = torch.Generator().manual_seed(N_c + N_r)
    real, cplx = (torch.float32, torch.complex64) if prec == "fp32" else (torch.float64, torch.complex128)
    psi0 = (0.1 * torch.randn(N_r, N_c, generator=g, dtype=cplx)).cuda()
    n0, P, V = (torch.rand(N_r, N_c, generator=g, dtype=real).cuda() for _ in range(3))
    V *= 1e-3
    ph, _ = _lib.physics_defaults(max(N_c, 2), max(N_r, 2), 0.5 * max(N_c - 1, 1), 0.5 * max(N_r - 1, 1))
    out = []
    for ty in (None, 4, 16):
        if ty:
            monkeypatch.setenv("PHX_RK4_TY", str(ty))
        psi, n = psi0.clone(), n0.clone()
        b, nb = torch.empty_like(psi), torch.empty_like(n)
        _lib.rk4_scalar_device(0 if prec == "fp32" else 1, ph, N_c, N_r, (True, False), psi.data_ptr(), n.data_ptr(), b.data_ptr(),
                               nb.data_ptr(), P.data_ptr(), V.data_ptr(), 0.04, 3, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        out.append((psi, n))
    for psi, n in out[1:]:
        assert torch.equal(psi, out[0][0]) and torch.equal(n, out[0][1])
