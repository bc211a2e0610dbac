"""Grids of one row, of fewer rows than a halo, and of more than 37837 rows (where a 32-bit reciprocal rounded up is
no longer an exact quotient): scalar RK4 on device buffers, ensembles and the adjoint against plain RK4 in 64 bits
(torch on the CPU, gradients by autograd).

Tolerance: the same expressions in another order, at most about 8 operations a stage on each value, so
3 steps x 4 stages x 8 u = 96 u, doubled, in relative L2; gradients: the repository's bar of 1e-10 for FP64."""
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (5, 1), (70, 1), (3, 2), (9, 5), (2, 46349), (3, 65535)]
DX, DT, STEPS = 0.5, 0.02, 3


def physics():
    from phoenix_amd import _lib
    return _lib.physics_defaults(64, 64, DX * 63, DX * 63)[0]


def rk4(ph, psi, n, P, V, steps, periodic):
    """`steps` RK4 steps in 64 bits; outside a zero boundary the state starts at zero and evolves within a step"""
    import torch
    h, (px, py) = 4, periodic

    def pad(f):
        w = (0 if px else h,) * 2 + (0 if py else h,) * 2
        if f.is_complex():
            return torch.complex(torch.nn.functional.pad(f.real, w), torch.nn.functional.pad(f.imag, w))
        return torch.nn.functional.pad(f, w)

    def cut(f):
        return f[..., slice(None) if py else slice(h, -h), slice(None) if px else slice(h, -h)]

    P, V = pad(P), pad(V)

    def rhs(p, m):
        lap = sum(torch.roll(p, s, d) for d in (-1, -2) for s in (1, -1)) - 4 * p
        nrm = p.real ** 2 + p.imag ** 2
        H = ph.m_eff_scaled * lap / DX ** 2 + (ph.g_c * nrm + ph.g_r * m + V) * p
        return -1j * ph.one_over_h_bar_s * H + 0.5 * (ph.R * m - ph.gamma_c) * p, -(ph.gamma_r + ph.R * nrm) * m + P

    for _ in range(steps):
        x, y = pad(psi), pad(n)
        k1 = rhs(x, y)
        k2 = rhs(x + DT / 2 * k1[0], y + DT / 2 * k1[1])
        k3 = rhs(x + DT / 2 * k2[0], y + DT / 2 * k2[1])
        k4 = rhs(x + DT * k3[0], y + DT * k3[1])
        psi = cut(x + DT / 6 * (k1[0] + 2 * k2[0] + 2 * k3[0] + k4[0]))
        n = cut(y + DT / 6 * (k1[1] + 2 * k2[1] + 2 * k3[1] + k4[1]))
    return psi, n


def inputs(N_c, N_r, real):
    """fields rounded to `real`, in 64 bits"""
    import torch
    g = torch.Generator().manual_seed(7 * N_c + N_r)
    f = [torch.rand(N_r, N_c, generator=g, dtype=torch.float64) for _ in range(5)]
    f = [v.to(real).double() for v in (0.3 * f[0] - 0.1, 0.3 * f[1] - 0.1, f[2], 2 * f[3], 1e-3 * f[4])]
    return torch.complex(f[0], f[1]), f[2], f[3], f[4]


def rel(a, b):
    return float((a - b).abs().pow(2).sum().sqrt() / b.abs().pow(2).sum().sqrt())


def types(prec):
    import torch
    return (torch.float32, torch.complex64, 2.0 ** -24) if prec == "fp32" else (torch.float64, torch.complex128, 2.0 ** -53)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("periodic", [(True, True), (False, True), (True, False)])
@pytest.mark.parametrize("N_c,N_r", SHAPES)
def test_forward(N_c, N_r, periodic, prec):
    import torch
    from phoenix_amd import _lib
    print(f"[row wrap] {N_c}x{N_r} periodic={periodic} {prec}", flush=True)
    real, cplx, u = types(prec)
    psi0, n0, P, V = inputs(N_c, N_r, real)
    want = rk4(physics(), psi0, n0, P, V, STEPS, periodic)
    psi, n, p, v = psi0.to(cplx).cuda(), n0.to(real).cuda(), P.to(real).cuda(), V.to(real).cuda()
    b, nb = torch.empty_like(psi), torch.empty_like(n)
    _lib.rk4_scalar_device(0 if prec == "fp32" else 1, physics(), N_c, N_r, periodic, psi.data_ptr(), n.data_ptr(), b.data_ptr(),
                           nb.data_ptr(), p.data_ptr(), v.data_ptr(), DT, STEPS, torch.cuda.current_stream().cuda_stream)
    e = _lib.Ensemble(prec, physics(), [(N_c, N_r)] * 2, [(DX, DX)] * 2, periodic, potential=True)
    for i in range(2):
        for name, f in (("psi_plus", psi0.to(cplx)), ("n_plus", n0.to(real)), ("pump_plus", P.to(real)), ("potential_plus", V.to(real))):
            e.set(i, name, f.numpy())
    e.step(DT, STEPS)
    got = [(psi.cpu(), n.cpu())] + [(torch.from_numpy(e.get(i, "psi_plus")), torch.from_numpy(e.get(i, "n_plus"))) for i in range(2)]
    e.close()
    for a, m in got:
        errs = rel(a.to(torch.complex128), want[0]), rel(m.double(), want[1])
        print(f"  psi {errs[0]:.2e} n {errs[1]:.2e}", flush=True)
        assert max(errs) <= 192 * u


# one periodic cell: V turns the phase only, so dJ/dV is what the steps' own error leaves (7e-9) of terms near 1
# that cancel, which neither side knows to 1e-10
UNIFORM = pytest.mark.xfail(reason="dJ/dV of a uniform state is rounding and step error alone")


@pytest.mark.parametrize("N_c,N_r,periodic", [pytest.param(c, r, p, marks=[UNIFORM] if c == r == 1 and all(p) else [])
                                              for c, r in SHAPES for p in ((True, True), (True, False))])
def test_adjoint(N_c, N_r, periodic):
    import torch
    from phoenix_amd.adjoint import rk4_evolve
    print(f"[row wrap, adjoint] {N_c}x{N_r} periodic={periodic}", flush=True)
    psi0, n0, P, V = inputs(N_c, N_r, torch.float64)
    w = torch.arange(1, N_c * N_r + 1, dtype=torch.float64).view(N_r, N_c) / (N_c * N_r)
    grads = []
    for dev in ("cpu", "cuda"):
        leaf = [f.to(dev).clone().requires_grad_(True) for f in (P, V, psi0[None], n0[None])]
        if dev == "cpu":
            a, m = rk4(physics(), leaf[2][0], leaf[3][0], leaf[0], leaf[1], STEPS, periodic)
        else:
            a, m = rk4_evolve(*leaf, physics=physics(), dt=DT, steps=STEPS, checkpoint_every=2, periodic=periodic)
        J = ((a.real ** 2 + a.imag ** 2) * w.to(dev)).sum() + 0.3 * (m * w.to(dev)).sum()
        grads.append([g.cpu() for g in torch.autograd.grad(J, leaf)])
    for name, g, want in zip(("P", "V", "psi", "n"), grads[1], grads[0]):
        print(f"  d{name} {rel(g, want):.2e}", flush=True)
        assert rel(g, want) <= 1e-10, name
