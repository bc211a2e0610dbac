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


def test_capture_by_the_caller():
    """a caller captures Ensemble.step on its own stream while the ensemble holds a graph for that call"""
    import torch
    print("[ensemble graph] captured by the caller", flush=True)
    dt, stream = 0.02, torch.cuda.Stream()
    a, *_ = make_ensemble("fp32")
    b, *_ = make_ensemble("fp32")
    a.set_stream(stream.cuda_stream)
    for e in (a, b):
        e.step(dt, 12, graph_steps=6)
    a.sync()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        a.step(dt, 6, graph_steps=6)
    for k in range(4):
        print(f"  replay {k}", flush=True)
        with torch.cuda.stream(stream):
            g.replay()
        stream.synchronize()
        b.step(dt, 6)
        for i in range(len(SIZES)):
            assert np.array_equal(a.get(i, "psi_plus"), b.get(i, "psi_plus"))
            assert np.array_equal(a.get(i, "n_plus"), b.get(i, "n_plus"))
    a.step(dt, 12, graph_steps=6)
    b.step(dt, 12)
    assert np.array_equal(a.get(0, "psi_plus"), b.get(0, "psi_plus"))
    a.close()
    b.close()
