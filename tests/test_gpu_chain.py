"""The chain kernel (phx_rk_chain.hip: RK4 under sources of at most two temporal groups, one launch per
step) against the staged path (phx_staged.hip), which a third pulse group of amplitude 0 selects.

Tolerance: both evaluate the same expressions with other roundings, at most about 8 operations' worth per
stage on each value: 4 stages x 6 steps x 8 u = 192 u of the unit roundoff u, relative L2."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CW = ["--pump", 6.0, "add", 8, 8, 0, 0, "both", 1, "none", "gauss+noDivide"]
TIMED_PUMP = ["--pump", 3.0, "add", 5, 5, 2, -3, "plus", 1, "none", "gauss+noDivide", "time", "cos", 0.1, 0.4, 9.0]
POT = ["--potential", 2e-3, "add", 6, 6, -3, 1, "both", 1, "none", "gauss+noDivide"]
TIMED_POT = ["--potential", 1e-3, "add", 5, 5, 1, 1, "both", 1, "none", "gauss+noDivide", "time", "iexp", 0.1, 0.5, 5.0]
PULSE = ["--pulse", 2e-4, "add", 5, 5, 2, -1, "both", 1, 1, "gauss+noDivide", "time", "iexp", 0.1, 0.3, 7.0]
PULSE2 = ["--pulse", 1e-4, "add", 7, 7, -2, 0, "minus", 1, "none", "gauss+noDivide", "time", "gauss", 0.05, 0.2, 1.0]
# one group: the constant one cannot be told from a timed one by its field, so it has an envelope of its own
NOTHING = [t for k in (1, 2, 3) for t in
           ("--pulse", 0.0, "add", 5, 5, 0, 0, "both", 1, "none", "gauss+noDivide", "time", "gauss", 0.1 * k, 0.7, 1.0)]


def run(prec, shape, boundary, args, steps=6):
    from phoenix_amd._lib import Solver
    Nc, Nr = shape
    base = ["--N", Nc, Nr, "--L", 0.5 * (Nc - 1), 0.6 * (Nr - 1), "--boundary", *boundary, "--outEvery", 1e9, "--fftEvery", 1e9,
            "--tstep", 0.04, "--tmax", 10]
    s = Solver([str(a) for a in base + args], prec)
    rng = np.random.default_rng(Nc + 3 * Nr)
    tetm, res = "-tetm" in args, s.info["use_reservoir"]
    out = {}
    for k in ("plus", "minus") if tetm else ("plus",):
        s.set("psi_" + k, 0.3 * (rng.standard_normal((Nr, Nc)) + 1j * rng.standard_normal((Nr, Nc))))
        if res:
            s.set("n_" + k, rng.random((Nr, Nc)))
    assert s.step(steps) == steps
    for k in ("plus", "minus") if tetm else ("plus",):
        out["psi_" + k] = s.get("psi_" + k).astype(np.complex128)
        if res:
            out["n_" + k] = s.get("n_" + k).astype(np.float64)
    s.close()
    return out


FORMS = {
    "pulse": CW + PULSE,
    "pulse without reservoir": PULSE + POT,
    "pump and potential chains": CW + TIMED_PUMP + POT + TIMED_POT + PULSE,
    "two pulses, no potential": CW + PULSE + PULSE2,
    "complex potential": CW + TIMED_POT,
    "noise": CW + PULSE + POT + ["--dw", 0.5, "--initRandom", 0.0, 7],
    "noise without reservoir": PULSE + ["--dw", 0.5, "--initRandom", 0.0, 7],
    "imaginary time": PULSE + PULSE2 + POT + ["--imagTime", 2.0],
}


def check(prec, shape, boundary, args):
    a, b = run(prec, shape, boundary, args), run(prec, shape, boundary, args + NOTHING)
    u = 2.0 ** -24 if prec == "fp32" else 2.0 ** -53
    for k in a:
        e = float(np.linalg.norm(a[k] - b[k]) / np.linalg.norm(b[k]))
        print(f"  {k} {e:.2e}", flush=True)
        assert e <= 192 * u, k


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("tetm", [False, True])
@pytest.mark.parametrize("form", list(FORMS))
def test_forms(form, tetm, prec):
    print(f"[chain] {form} tetm={tetm} {prec}", flush=True)
    check(prec, (62, 54), ("periodic", "zero"), FORMS[form] + (["-tetm"] if tetm else []))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("boundary", [("periodic", "periodic"), ("zero", "periodic"), ("zero", "zero")])
@pytest.mark.parametrize("shape", [(8, 6), (56, 16), (58, 18), (642, 482), (1026, 514)])
def test_shapes(shape, boundary, prec):
    """grids smaller than a tile's halo, whole and ragged tiles, and sizes that take tiles of 4, 8 and 16 rows"""
    print(f"[chain] {shape} {boundary} {prec}", flush=True)
    check(prec, shape, boundary, CW + POT + PULSE + (PULSE2 + ["-tetm"] if shape[0] == 58 else []))
