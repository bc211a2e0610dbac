"""GPU parity of the mixed-radix transforms (phx_fft_mixed.hip) against numpy: the k-space filter, the
stored spectrum and the plain forward transform of lengths that are not powers of two.

Tolerance: a transform of L points by radix passes has a relative L2 error of at most about
4 u log2 L (u the unit roundoff: products with rounded twiddles and sums, per radix-2 level); the
filter runs two transforms on each axis, and a Bluestein length is itself two transforms of fewer than
4 L points with chirp products, so 16 u (log2 4 N_c + log2 4 N_r) bounds every case."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# row length x column length.  2 x 4: one pass; 16 x 18: one pass and two; 6, 22: ragged column blocks;
# 26 = 2 13 and 34 = 2 17 on either side of the Bluestein rule; 352, 2002 = 2 7 11 13, 1458 = 2 3^6: every
# radix; 400: the default grid; 512 / 1024 next to other lengths: two kernels in one transform
SHAPES = [(2, 4), (16, 18), (6, 22), (26, 34), (34, 26), (62, 6), (400, 400), (352, 250), (512, 300), (300, 512), (1024, 22),
          (2002, 8), (8, 2002), (1458, 10), (2038, 4), (4, 2038)]


def solver(prec, Nc, Nr, mask=True):
    from phoenix_amd._lib import Solver
    args = ["--N", Nc, Nr, "--L", 0.5 * (Nc - 1), 0.5 * (Nr - 1), "--boundary", "periodic", "periodic", "--tstep", 0.04, "--tmax", 10,
            "--outEvery", 1e9, "--fftEvery", 0.02, "--pump", 1.0, "add", 10, 10, 0, 0, "both", 1, "none", "gauss+noDivide"]
    if mask:
        args += ["--fftMask", 1.0, "add", 0.5, 0.5, 0, 0, "both", 6, "none", "gauss+noDivide+local"]
    return Solver([str(a) for a in args], prec)


def tolerance(prec, Nc, Nr):
    u = 2.0 ** -24 if prec == "fp32" else 2.0 ** -53
    return 16 * u * (np.log2(4 * Nc) + np.log2(4 * Nr))


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def check(prec, Nc, Nr):
    rng = np.random.default_rng(Nc * 11 + Nr)
    psi = (rng.standard_normal((Nr, Nc)) + 1j * rng.standard_normal((Nr, Nc))).astype(np.complex64 if prec == "fp32" else np.complex128)
    mask = rng.random((Nr, Nc)).astype(np.float32 if prec == "fp32" else np.float64)
    print(f"[mixed fft] {prec} {Nc}x{Nr}", flush=True)
    s = solver(prec, Nc, Nr)
    s.set("psi_plus", psi)
    s.set("fft_mask_plus", mask)
    s.apply_fft_filter()
    out, spec = s.get("psi_plus").astype(np.complex128), s.get("fft_plus").astype(np.complex128)
    s.close()
    F = np.fft.fft2(psi.astype(np.complex128)) / (Nc * Nr) * np.fft.ifftshift(mask.astype(np.float64))
    want = np.fft.ifft2(F) * (Nc * Nr)
    tol = tolerance(prec, Nc, Nr)
    print(f"  filter {rel(out, want):.2e}, spectrum {rel(spec, F):.2e} (<= {tol:.2e})", flush=True)
    assert rel(out, want) <= tol
    assert rel(spec, F) <= tol


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", SHAPES)
def test_filter_and_spectrum(prec, shape):
    check(prec, *shape)


@pytest.mark.parametrize("shape", [(4094, 6), (6, 4094), (3430, 6), (6, 4050)])
def test_longest_fp32_lengths(shape):
    """Bluestein of 8192 points (128 KiB of LDS) and long smooth lengths"""
    check("fp32", *shape)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", [(90, 34), (46, 60)])
def test_forward_spectrum_without_mask(prec, shape):
    """without a mask the spectrum is the unnormalised transform of psi at the last FFT time"""
    Nc, Nr = shape
    s = solver(prec, Nc, Nr, mask=False)
    rng = np.random.default_rng(3)
    s.set("psi_plus", rng.standard_normal((Nr, Nc)) + 1j * rng.standard_normal((Nr, Nc)))
    assert s.step(1) == 1
    psi, spec = s.get("psi_plus").astype(np.complex128), s.get("fft_plus").astype(np.complex128)
    s.close()
    assert rel(spec, np.fft.fft2(psi)) <= tolerance(prec, Nc, Nr)
