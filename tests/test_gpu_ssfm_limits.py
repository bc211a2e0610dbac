"""The split-step iterator's row kernel at the longest rows that it takes, which fill its LDS: powers of two, and
Bluestein lengths whose convolution has the longest length.  Bars: those of test_gpu_ssfm_runs."""
import numpy as np
import pytest

import test_gpu_ssfm_runs as runs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,shape", [("fp32", (8192, 4)), ("fp64", (4096, 4)), ("fp32", (4094, 6)), ("fp64", (2046, 6)), ("fp32", (4096, 10)),
                                        ("fp32", (4090, 4)), ("fp64", (2048, 34))])
@pytest.mark.parametrize("form", ["plain", "pulse"])
def test_longest_rows(form, prec, shape):
    print(f"[ssfm limits] {form} {shape} {prec}", flush=True)
    (a, ta), (b, tb) = runs.run(prec, shape, runs.FORMS[form], [5]), runs.run(prec, shape, runs.FORMS[form], [1] * 5)
    assert ta == tb
    for x, y in zip(a, b):
        assert np.isfinite(x).all() and runs.rel(x, y) <= runs.tolerance(prec, shape)


@pytest.mark.parametrize("prec,shape", [("fp64", (4096, 4)), ("fp64", (2046, 6))])
def test_longest_rows_match_numpy(prec, shape):
    runs.test_linear_run_matches_numpy(prec, shape)
