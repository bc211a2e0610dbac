"""phx_apply_fft_filter where the transforms exist but no mask does (split-step iterator, spectra for output): an error,
as in a configuration without transforms, and the state stays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("extra", [["--iterator", "SSFM"], ["--fftEvery", 0.1, "--output", "fft"], []], ids=["ssfm", "spectra", "neither"])
def test_refused(extra, prec):
    from phoenix_amd._lib import PhxError, Solver
    print(f"[filter without mask] {extra} {prec}", flush=True)
    args = ["--N", 32, 32, "--L", 15.5, 15.5, "--tstep", 0.02, "--tmax", 1, "--outEvery", 1, *extra]
    s = Solver([str(a) for a in args], prec)
    psi = np.random.default_rng(1).standard_normal((32, 32)) + 0j
    s.set("psi_plus", psi)
    before = s.get("psi_plus")
    with pytest.raises(PhxError, match="no FFT mask"):
        s.apply_fft_filter()
    assert np.array_equal(s.get("psi_plus"), before)
    s.close()
