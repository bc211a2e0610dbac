"""A captured run of an ensemble holds the addresses of its tables: a change of the tile height, which rebuilds them,
ends it, also where the height that was captured comes back.  Bitwise against stepping launch by launch."""
import numpy as np
import pytest

from test_gpu_ensemble import SIZES, make_ensemble

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("between", [0, 4])  # steps at the other height: launched one by one, fewer than a graph's
@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_tile_height_there_and_back(prec, between):
    print(f"[ensemble graph] {prec} 8, 10 and 8 rows, {between} steps between", flush=True)
    dt = 0.02
    a, *_ = make_ensemble(prec)
    b, *_ = make_ensemble(prec)
    a.set_tile_rows(12)
    for rows, steps in ((8, 12), (10, between), (8, 12), (20, 2), (8, 6)):
        b.set_tile_rows(rows)
        b.step(dt, steps, graph_steps=6)
        a.step(dt, steps)
    for i in range(len(SIZES)):
        assert np.array_equal(a.get(i, "psi_plus"), b.get(i, "psi_plus"))
        assert np.array_equal(a.get(i, "n_plus"), b.get(i, "n_plus"))
    a.close()
    b.close()
