"""GPU tests of the multi-step RK4 kernel (rk4_scalar_flow) where its blocks take ticket after ticket instead of
keeping one chunk of tiles: from the start (PHX_FLOW_GATE_LIMIT=-1), or after a gate that some blocks find closed
(0: the first block that has done its first chunk closes it, unless all were resident by then).

Bar: bitwise equal to the same steps launched one by one, whichever way a launch went; several handles at once too.
Runs of several lengths follow each other, so that the words which a launch puts back are used by the next.
"""
import numpy as np
import pytest

from test_gpu_flow import say, solver

pytestmark = pytest.mark.gpu
RUNS = (1, 2, 11, 40, 3)  # the first step tunes the tile shape


def fields(s):
    return s.get("psi_plus"), s.get("n_plus")


@pytest.mark.parametrize("gate", [-1, 0])
@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("N_c,N_r,bc,pot", [(1024, 1024, "periodic", False), (174, 134, "zero", True), (58, 46, "periodic", False),
                                            (56, 20, "zero", False), (618, 334, "periodic", True)])
def test_tickets_equal_step_by_step(monkeypatch, prec, N_c, N_r, bc, pot, gate):
    say(f"[tickets] {prec} {N_c}x{N_r} {bc} potential={pot} gate limit {gate}")
    out = []
    for flow in ("0", "1"):
        monkeypatch.setenv("PHX_RK4_FLOW", flow)
        monkeypatch.setenv("PHX_FLOW_GATE_LIMIT", str(gate))
        s = solver(prec, N_c, N_r, bc, pot, 29)
        for n in RUNS:
            assert s.step(n) == n
        out.append(fields(s))
        assert s.info["multi_step_steps"] == (0 if flow == "0" else sum(RUNS[1:]))
        s.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_handles_at_once_equal_one_alone(monkeypatch, prec):
    say(f"[tickets] {prec} three handles of 1024x1024 at once")
    monkeypatch.setenv("PHX_RK4_FLOW", "1")
    alone = solver(prec, 1024, 1024, "periodic", False, 31)
    for n in RUNS:
        alone.step(n)
    want = fields(alone)
    alone.close()
    three = [solver(prec, 1024, 1024, "periodic", False, 31) for _ in range(3)]
    for n in RUNS:
        for s in three:
            s.step(n)
    for s in three:
        got = fields(s)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        s.close()
