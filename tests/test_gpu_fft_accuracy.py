"""Accuracy of the k-space filter at lengths with a large prime factor (Bluestein's convolution): FP64 against FP32, each in
units of its own roundoff, the reference in extended precision (numpy, long double).

Tolerance: both precisions do the same operations on tables rounded once from more digits, so in units of the roundoff
their relative L2 errors agree but for chance, a few per cent over 10^4 values; 1.5 leaves room.  Tables that carry
errors of their own, as those of a transform in double do in FP64, show as a larger ratio."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def units(prec, N_c, N_r):
    from phoenix_amd._lib import Solver
    real, cplx, u = (np.float32, np.complex64, 2.0 ** -24) if prec == "fp32" else (np.float64, np.complex128, 2.0 ** -53)
    args = ["--N", N_c, N_r, "--L", 0.5 * (N_c - 1), 0.5 * (N_r - 1), "--boundary", "periodic", "periodic", "--tstep", 0.04, "--tmax", 1e9,
            "--outEvery", 1e12, "--fftEvery", 1e12, "--fftMask", 1.0, "add", 10, 10, 0, 0, "both", 1, "none", "gauss+noDivide"]
    s = Solver([str(a) for a in args], prec)
    rng = np.random.default_rng([N_c, N_r])
    psi = (rng.standard_normal((N_r, N_c)) + 1j * rng.standard_normal((N_r, N_c))).astype(cplx)
    mask = rng.random((N_r, N_c)).astype(real)
    s.set("psi_plus", psi)
    s.set("fft_mask_plus", mask)
    s.apply_fft_filter()
    got = s.get("psi_plus").astype(np.clongdouble)
    s.close()
    f = psi.astype(np.clongdouble)
    f = np.fft.fft(np.fft.fft(f, axis=0), axis=1) * np.fft.ifftshift(mask.astype(np.longdouble))
    f = np.fft.ifft(np.fft.ifft(f, axis=0), axis=1)
    assert f.dtype == np.clongdouble
    return float(np.linalg.norm((got - f).astype(complex)) / np.linalg.norm(f.astype(complex))) / u


@pytest.mark.parametrize("N_c,N_r", [(102, 102), (122, 122), (118, 134), (138, 158), (302, 302), (646, 122)])
def test_fp64_errors_are_fp32_errors_in_units_of_roundoff(N_c, N_r):
    e32, e64 = units("fp32", N_c, N_r), units("fp64", N_c, N_r)
    print(f"[fft accuracy] {N_c}x{N_r}: FP32 {e32:.2f} u, FP64 {e64:.2f} u", flush=True)
    assert e64 <= 1.5 * e32


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("N_c,N_r", [(34, 34), (76, 76), (106, 106), (514, 106), (100, 100), (150, 34)])
def test_split_step_runs_keep_their_amplitude(N_c, N_r, prec):
    """200 linear steps against the exact propagator: what the rounded constants of the transforms do to the amplitude
    of everything alike adds up over the steps.

    Tolerance, in units of roundoff a step: four one-dimensional transforms whose mean gain is made up for to 0.2 each
    (the estimate, and the rounding of the table that holds it), and 0.5 for the damping factor exp(-gamma_c dt / 2), the
    same in every step: 1.3, and 0.2 for everything random."""
    from phoenix_amd._lib import Solver
    real, cplx, u = (np.float32, np.complex64, 2.0 ** -24) if prec == "fp32" else (np.float64, np.complex128, 2.0 ** -53)
    ld, steps, dt = np.longdouble, 200, np.longdouble(real(0.04))
    args = ["--N", N_c, N_r, "--L", 0.5 * (N_c - 1), 0.5 * (N_r - 1), "--boundary", "periodic", "periodic", "--outEvery", 1e9, "--fftEvery", 1e9,
            "--tstep", 0.04, "--tmax", 1e9, "--iterator", "SSFM", "-noReservoir", "--gc", 0.0]
    s = Solver([str(a) for a in args], prec)
    rng = np.random.default_rng([N_c, N_r, 1])
    psi = (rng.standard_normal((N_r, N_c)) + 1j * rng.standard_normal((N_r, N_c))).astype(cplx)
    s.set("psi_plus", psi)
    assert s.step(steps) == steps
    got = s.get("psi_plus").astype(np.clongdouble)
    s.close()
    hs, m = ld("1.0545718e-34") / ld("1.60217662e-19") * ld("1e12"), ld("9.10938356e-31") / ld("1.60217662e-19") * ld("1e8")
    k2 = [(2 * ld("3.1415926535") * np.where(np.arange(n) <= n // 2, np.arange(n), np.arange(n) - n) / (ld("0.5") * (n - 1))) ** 2 for n in (N_r, N_c)]
    f = np.fft.fft(np.fft.fft(psi.astype(np.clongdouble), axis=0), axis=1)
    f = f * np.exp(np.clongdouble(-0.5j) * (hs / m * dt * steps * (k2[0][:, None] + k2[1][None, :])))
    f = np.fft.ifft(np.fft.ifft(f, axis=0), axis=1) * np.exp(-ld(real(0.15)) / 2 * dt * steps)
    gain = abs(np.vdot(f.ravel(), got.ravel()) / np.vdot(f.ravel(), f.ravel()))
    drift = float((gain - 1) / u) / steps
    print(f"[fft accuracy] {N_c}x{N_r} {prec}: {drift:.2f} u of amplitude a step", flush=True)
    assert abs(drift) <= 1.5
