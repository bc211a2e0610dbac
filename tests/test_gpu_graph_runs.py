"""Runs of single-step launches replayed from a captured graph (phx_step on grids below the multi-step kernel's): which
runs are replayed, from which graph, and what is left over of them.

Bar: bitwise equal to stepping one at a time, with the same time; PhxInfo.graph_replays tells that graphs ran.  A handle
captures once it has launched 400 steps one by one."""
import numpy as np
import pytest

from test_gpu_flow import solver

pytestmark = pytest.mark.gpu
N = 128


def start(prec):
    return solver(prec, N, N, "periodic", False, 47)


def state(s):
    return s.get("psi_plus"), s.get("n_plus"), s.time()[0], s.info["iteration"]


def single(s, steps):
    for _ in range(steps):
        assert s.step(1) == 1


def check(a, b):
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    assert a[2:] == b[2:]


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("runs", [[10] * 45 + [12, 7, 10, 61, 33, 2, 100, 1, 50, 11, 50], [51] * 20, [60] * 9 + [1] + [60] * 9],
                         ids=["mixed", "odd", "other_buffer"])
def test_runs_equal_single_steps(runs, prec):
    print(f"[graph runs] {prec} {runs}", flush=True)
    a, b = start(prec), start(prec)
    for r in runs:
        assert a.step(r) == r
    single(b, sum(runs))
    assert a.info["graph_replays"] > 0 and b.info["graph_replays"] == 0
    check(state(a), state(b))
    a.close()
    b.close()


def test_longer_runs_get_a_longer_graph():
    """after runs of 10 steps a run of 500 is first served by their graph, and by one of 50 once it repeats"""
    s = start("fp32")
    for _ in range(50):
        s.step(10)
    for _ in range(2):
        s.step(500)
    before = s.info["graph_replays"]
    s.step(500)
    print(f"[graph runs] {s.info['graph_replays'] - before} replays for 500 steps", flush=True)
    assert s.info["graph_replays"] - before == 10
    # and shorter runs, now and then, leave it
    s.step(10)
    before = s.info["graph_replays"]
    s.step(500)
    assert s.info["graph_replays"] - before == 10
    s.close()


def test_runs_from_the_other_buffer_get_a_graph():
    """one odd run, and every later run starts in the buffer that the captured one does not"""
    s = start("fp32")
    for _ in range(10):
        s.step(60)
    assert s.info["graph_replays"] > 0
    s.step(1)
    for _ in range(10):
        s.step(60)
    before = s.info["graph_replays"]
    s.step(60)
    assert s.info["graph_replays"] - before == 1
    s.close()


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_runs_cut_by_the_filter(prec):
    from phoenix_amd._lib import Solver
    print(f"[graph runs] {prec} filter every 25 steps", flush=True)
    L, dt = 0.5 * (N - 1), 0.04
    args = ["--N", N, N, "--L", L, L, "--boundary", "periodic", "periodic", "--tstep", dt, "--tmax", 1e9, "--outEvery", 1e12, "--fftEvery",
            24.5 * dt, "--pump", 20.0, "add", 10, 10, 0, 0, "both", 1, "none", "gauss+noDivide", "--fftMask", "1.0", "add",
            "0.565685", "0.565685", "0", "0", "both", "6", "none", "gauss+noDivide+local"]
    rng = np.random.default_rng(3)
    psi = 0.1 * (rng.standard_normal((N, N)) + 1j * rng.standard_normal((N, N)))
    a, b = (Solver([str(v) for v in args], prec) for _ in range(2))
    for s in (a, b):
        s.set("psi_plus", psi)
    runs = [60] * 10 + [37, 100, 24]
    for r in runs:
        assert a.step(r) == r
    single(b, sum(runs))
    assert a.info["graph_replays"] > 0
    check(state(a), state(b))
    a.close()
    b.close()


def test_capture_by_the_caller():
    """a caller captures phx_step on its own stream while the handle holds a graph: the launches are recorded"""
    import torch
    stream = torch.cuda.Stream()
    a, b = start("fp32"), start("fp32")
    a.set_stream(stream.cuda_stream)
    for s in (a, b):
        for _ in range(50):
            s.step(10)
    a.sync()
    assert a.info["graph_replays"] > 0
    replays = a.info["graph_replays"]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        assert a.step(20) == 20
    assert a.info["graph_replays"] == replays
    for k in range(4):
        print(f"[graph runs] replay {k}", flush=True)
        with torch.cuda.stream(stream):
            g.replay()
        stream.synchronize()
        b.step(20)
        assert np.array_equal(a.get("psi_plus"), b.get("psi_plus")) and np.array_equal(a.get("n_plus"), b.get("n_plus"))
    a.step(3)
    b.step(3)
    assert np.array_equal(a.get("psi_plus"), b.get("psi_plus"))
    a.close()
    b.close()
