"""Tile heights that the size rules and the autotuners choose, forced by their environment values on small grids: the
generic RK4 kernels (TE-TM, noise) and the chain kernels at 4, 8 and 16 rows, the adaptive Dormand-Prince kernels at 8,
16, 28, 32 and 42, and the scalar RK4 kernels at 2 and 4 (multi-step: 4) with every prefetch depth.

Bars: those of the tests that run the heights of small grids (oracle: FP64 relative L2 <= 1e-12, FP32 <= 1e-5; staged
path; spinor trajectories of the 16-row kernel to 1e-6; scalar RK4 bitwise)."""
import numpy as np
import pytest

import test_gpu_chain as chain
import test_gpu_dp45_tetm as dp45
import test_gpu_instantiations as inst
import test_gpu_tile_shapes as shapes

pytestmark = pytest.mark.gpu
PRECS = ["fp64", "fp32"]


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("tetm,res,noise", [f for f in inst.FLAGS if f[0] or f[2]], ids=lambda v: str(int(v)))
@pytest.mark.parametrize("ty", [4, 8, 16])
def test_generic_rk4(monkeypatch, ty, tetm, res, noise, prec):
    monkeypatch.setenv("PHX_RK4G_TY", str(ty))
    inst.test_instantiation_matches_oracle("RK4", False, tetm, res, noise, prec)


@pytest.mark.parametrize("tetm,res,noise,prec,ty",
                         [(*f, p, ty) for f in inst.FLAGS for p in PRECS for ty in (8, 16, 28, 32, 42)
                          if ty <= 16 or (f[0] and p == "fp32")], ids=lambda v: v if isinstance(v, str) else str(int(v)))
def test_adaptive_dp45(monkeypatch, tetm, res, noise, prec, ty):
    monkeypatch.setenv("PHX_GEN_TY", str(ty))
    inst.test_instantiation_matches_oracle("DP45", True, tetm, res, noise, prec)


@pytest.mark.parametrize("noise", [False, True])
@pytest.mark.parametrize("pot", [False, True])
def test_spinor_dp45_trajectories(monkeypatch, pot, noise):
    """several tiles in each direction, the last ones ragged; with and without the potential compiled in"""
    N, L, dt0, tmax, seed = 150, 74.5, 0.04, 0.6, 9
    psi, n, Pp, psim, nm, Pm = dp45.inputs(N, L, 41, tetm=True)
    fields = {"psi_plus": psi, "n_plus": n, "pump_plus": Pp, "psi_minus": psim, "n_minus": nm, "pump_minus": Pm}
    args = ["-tetm", "--iterator", "DP45", "-adaptive", "--tol", 1e-6, "--rkvdt", 1e-4, 0.1, "--tstep", dt0, "--tmax", tmax]
    if noise:
        args += ["--dw", 0.05, "--initRandom", 0.0, seed]
    if pot:
        x = -L / 2 + L / (N - 1) * np.arange(N)
        V = 2e-3 * np.exp(-0.5 * ((x[None, :] - 3) ** 2 + (x[:, None] + 2) ** 2) / 6.0 ** 2)
        fields.update(potential_plus=V, potential_minus=V[::-1].copy())
        args += ["--potential", 1.0, "add", 10, 10, 0, 0, "both", 1, "none", "gauss+noDivide"]
    want = None
    for ty in (16, 8, 28, 32, 42):
        monkeypatch.setenv("PHX_GEN_TY", str(ty))
        print(f"[heights] spinor DP45 {ty} rows, potential {pot}, noise {noise}", flush=True)
        out, done, info = dp45.gpu("fp32", N, L, args, fields, 100000)
        if want is None:
            want = out, done, info["rejected"]
            continue
        assert (done, info["rejected"]) == want[1:]
        for k in ("psi_plus", "psi_minus", "n_plus", "n_minus"):
            assert dp45.rel_l2(out[k], want[0][k]) <= 1e-6, (ty, k)


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("tetm", [False, True])
@pytest.mark.parametrize("form", list(chain.FORMS))
@pytest.mark.parametrize("ty", [8, 16])
def test_chain(monkeypatch, ty, form, tetm, prec):
    monkeypatch.setenv("PHX_RK4G_TY", str(ty))
    print(f"[heights] chain {ty} rows, {form}, tetm={tetm} {prec}", flush=True)
    chain.check(prec, (62, 54), ("periodic", "zero"), chain.FORMS[form] + (["-tetm"] if tetm else []))


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("name,N_c,N_r,bc,pot", shapes.GRIDS, ids=["zero_pot_200x136", "periodic_256"])
@pytest.mark.parametrize("flow,tys", [("0", (2, 4)), ("1", (4,))], ids=["one_step", "multi_step"])
def test_scalar_rk4(monkeypatch, flow, tys, name, N_c, N_r, bc, pot, prec):
    steps = 31
    monkeypatch.setenv("PHX_RK4_FLOW", "0")
    monkeypatch.setenv("PHX_RK4_TY", "16")
    psi, n, _ = shapes.run(prec, N_c, N_r, bc, pot, steps)
    monkeypatch.setenv("PHX_RK4_FLOW", flow)
    for ty in tys:
        for pf in shapes.PFS:
            monkeypatch.setenv("PHX_RK4_TY", str(ty))
            monkeypatch.setenv("PHX_RK4_PF", str(pf))
            print(f"[heights] scalar RK4 {prec} {name} {ty} rows, {pf} ahead, multi-step {flow}", flush=True)
            p, m, i = shapes.run(prec, N_c, N_r, bc, pot, steps)
            assert i["tile_rows"] == ty and i["prefetch_rows"] == pf and (i["multi_step_steps"] > 0) == (flow == "1")
            assert np.array_equal(p, psi) and np.array_equal(m, n), (ty, pf)
