"""First steps of many handles on several threads at once: each tunes its launch shape and shares it with the process.
Bitwise against the same handles stepped one after the other."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from test_gpu_flow import solver

pytestmark = pytest.mark.gpu


def test_handles_tune_on_several_threads():
    sizes = [(96 + 2 * k, 64 + 4 * (k % 5)) for k in range(24)]

    def one(k):
        s = solver("fp32" if k % 2 else "fp64", *sizes[k], "periodic", k % 3 == 0, k)
        assert s.step(13) == 13
        out = s.get("psi_plus"), s.get("n_plus")
        s.close()
        return out

    print("[threads] 24 handles on 6 threads", flush=True)
    with ThreadPoolExecutor(6) as ex:
        got = list(ex.map(one, range(len(sizes))))
    for k, (psi, n) in enumerate(got):
        want = one(k)
        assert np.array_equal(psi, want[0]) and np.array_equal(n, want[1]), sizes[k]
