"""Runs of the split-step iterator (column passes with both half steps, rows and pointwise step in one
kernel, phx_ssfm_rows.hip) against the same steps taken one by one, which the oracle tests cover, and
against a split-step in numpy.

Tolerance: a propagation is one transform each way on both axes, at most 16 u (log2 4 N_c + log2 4 N_r)
relative L2 (test_gpu_fft_mixed.py); a step has two, and five steps are taken.  The pointwise factors add
a few u each."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# row lengths: several rows a workgroup and one, powers of two, 5-smooth, 13-smooth, Bluestein (34: several
# rows a workgroup, 1030: a length 2^a 3^b 5^c)
SHAPES = [(16, 10), (64, 34), (34, 16), (1030, 8), (22, 6), (60, 26), (512, 20), (2048, 6)]
PUMP = ["--pump", 6.0, "add", 8, 8, 0, 0, "both", 1, "none", "gauss+noDivide"]
TIMED = ["--pump", 2.0, "add", 5, 5, 1, 0, "both", 1, "none", "gauss+noDivide", "time", "cos", 0.05, 0.2, 7.0]
POT = ["--potential", 2e-3, "add", 6, 6, -1, 1, "both", 1, "none", "gauss+noDivide", "time", "iexp", 0.1, 0.5, 5.0]
PULSE = ["--pulse", 2e-4, "add", 5, 5, 1, -1, "both", 1, 1, "gauss+noDivide", "time", "iexp", 0.1, 0.3, 7.0]
FORMS = {"plain": PUMP, "no reservoir": POT, "chains": PUMP + TIMED + POT, "pulse": PUMP + PULSE, "pulse alone": PULSE}


def run(prec, shape, args, calls, tmax=10.0, extra=()):
    from phoenix_amd._lib import Solver
    Nc, Nr = shape
    base = ["--N", Nc, Nr, "--L", 0.5 * (Nc - 1), 0.5 * (Nr - 1), "--boundary", "periodic", "periodic", "--outEvery", 0.13, "--fftEvery", 1e9,
            "--tstep", 0.04, "--tmax", tmax, "--iterator", "SSFM"]
    s = Solver([str(a) for a in base + args + list(extra)], prec)
    rng = np.random.default_rng(Nc + 3 * Nr)
    s.set("psi_plus", 0.3 * (rng.standard_normal((Nr, Nc)) + 1j * rng.standard_normal((Nr, Nc))))
    res = s.info["use_reservoir"]
    if res:
        s.set("n_plus", rng.random((Nr, Nc)))
    for n in calls:
        if n == "interval":
            s.run_interval()
        else:
            assert s.step(n) == n
    out = [s.get("psi_plus").astype(np.complex128)] + ([s.get("n_plus").astype(np.float64)] if res else [])
    t = s.time()[0]
    s.close()
    return out, t


def tolerance(prec, shape):
    u = 2.0 ** -24 if prec == "fp32" else 2.0 ** -53
    return 5 * 2 * 16 * u * (np.log2(4 * shape[0]) + np.log2(4 * shape[1]))


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("form", list(FORMS))
def test_run_equals_single_steps(form, shape, prec):
    print(f"[ssfm runs] {form} {shape} {prec}", flush=True)
    (a, ta), (b, tb) = run(prec, shape, FORMS[form], [5]), run(prec, shape, FORMS[form], [1] * 5)
    assert ta == tb
    for x, y in zip(a, b):
        print(f"  {rel(x, y):.2e} (<= {tolerance(prec, shape):.2e})", flush=True)
        assert rel(x, y) <= tolerance(prec, shape)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_interval_lands_with_a_shortened_step(prec):
    """0.13 is three whole steps and a shorter one, whose factors are other ones"""
    a, ta = run(prec, (60, 26), FORMS["plain"], ["interval"])
    b, tb = run(prec, (60, 26), FORMS["plain"], [1, 1, 1, "interval"])
    assert ta == tb and abs(ta - 0.13) < 1e-6
    for x, y in zip(a, b):
        assert rel(x, y) <= tolerance(prec, (60, 26))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", [(34, 16), (60, 26), (64, 34)])
def test_linear_run_matches_numpy(prec, shape):
    """without sources five steps are the exact propagator of the time they cover, damped by gamma_c"""
    Nc, Nr = shape
    (out,), t = run(prec, shape, ["-noReservoir", "--gc", 0.0], [5])
    rng = np.random.default_rng(Nc + 3 * Nr)
    psi0 = 0.3 * (rng.standard_normal((Nr, Nc)) + 1j * rng.standard_normal((Nr, Nc)))
    hs, m = 1.0545718e-34 / 1.60217662e-19 * 1e12, 9.10938356e-31 / 1.60217662e-19 * 1e8
    k = [2 * 3.1415926535 * np.where(np.arange(n) <= n // 2, np.arange(n), np.arange(n) - n) / (0.5 * (n - 1)) for n in (Nr, Nc)]
    ref = np.fft.ifft2(np.fft.fft2(psi0) * np.exp(-0.5j * hs / m * (k[0][:, None] ** 2 + k[1][None, :] ** 2) * t)) * np.exp(-0.075 * t)
    # FP32: the inputs and the factors of the propagator are rounded too (phases of up to about 10 rad)
    assert rel(out, ref) <= (tolerance(prec, shape) if prec == "fp64" else 2e-5)
