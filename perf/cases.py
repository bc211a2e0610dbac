"""Performance cases: what a user of phoenix_amd has it do, through its public entry points.

Each case is one call sequence of a user's program on inputs made from a seed:

  device     fixed RK4 steps on torch-owned buffers (rk4_scalar_device), as a loop that looks at
             the state after every few steps makes them: the smallest calls
  rk4        Solver.step on the scalar model, optionally with the k-space filter every few steps
  spinor     Solver.step on the TE-TM model: adaptive Dormand-Prince (with or without noise) or RK4
  ssfm       Solver.step of the split-step Fourier iterator
  pulse      Solver.step of RK4 under a resonant pulse with a temporal envelope
  ensemble   Ensemble.step: grids of different sizes stepped together
  adjoint    rk4_evolve: objective and gradients with respect to pump, potential and initial state

listed() holds one or more of each at a size in ordinary use; draw() makes others of the same
ranges.  Passes continue from the state that the previous one left, as a simulation does.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from phoenix_amd import _lib
from phoenix_amd.adjoint import rk4_evolve

# model defaults of the framework's configuration surface
H_BAR, M_E, E_E = 1.0545718e-34, 9.10938356e-31, 1.60217662e-19
H_BAR_S = H_BAR / E_E * 1e12
M_EFF = M_E / E_E * 1e8
GAMMA_C, GAMMA_R, G_C, G_R, RR = 0.15, 0.225, 3e-6, 6e-6, 0.01
G_PM, DELTA_LT = -3e-6 / 5, 0.025e-3
P_TH = GAMMA_C * GAMMA_R / RR
DX, DT = 0.5, 0.04  # um, ps
CW = 5.0  # amplitude of the continuous pump of the command line
PULSE = (6.0, 4.0, 1.2)  # t0, sigma, frequency of the pulse's temporal envelope
PUMP_T = (10.0, 8.0, 0.3)  # ... and of the second, time-dependent pump
ENSEMBLE_SIDES = (128, 192, 256, 384, 512)


def listed():
    return [
        # an interactive loop: a few steps at a time on a small grid held in torch tensors
        {"name": "device_200x150_fp32", "kind": "device", "nc": 200, "nr": 150, "prec": "fp32", "px": False, "py": False,
         "pot": True, "steps": 2},
        # the plain scalar run in double precision: Gaussian pump, 256^2, periodic
        {"name": "rk4_256_fp64", "kind": "rk4", "nc": 256, "nr": 256, "prec": "fp64", "px": True, "py": True, "pot": False,
         "pump": "gauss", "every": 0, "steps": 100},
        # the ring-pump run with the k-space low-pass filter every 50 steps, both precisions
        {"name": "rk4_1024_fp32_filter", "kind": "rk4", "nc": 1024, "nr": 1024, "prec": "fp32", "px": True, "py": True,
         "pot": False, "pump": "ring", "every": 50, "steps": 50},
        {"name": "rk4_1024_fp64_filter", "kind": "rk4", "nc": 1024, "nr": 1024, "prec": "fp64", "px": True, "py": True,
         "pot": False, "pump": "ring", "every": 50, "steps": 50},
        # the default grid (400 x 400, zero boundaries) with a potential and a frequent filter
        {"name": "rk4_400_fp64_filter5", "kind": "rk4", "nc": 400, "nr": 400, "prec": "fp64", "px": False, "py": False,
         "pot": True, "pump": "gauss", "every": 5, "steps": 20},
        # a large domain whose state does not fit the last-level cache
        {"name": "rk4_3600x3200_fp32", "kind": "rk4", "nc": 3600, "nr": 3200, "prec": "fp32", "px": True, "py": True,
         "pot": False, "pump": "ring", "every": 0, "steps": 10},
        # stochastic spinor model under an elliptically polarised pump, adaptive steps
        {"name": "spinor_2048_fp32_dp45_noise", "kind": "spinor", "nc": 2048, "nr": 2048, "prec": "fp32", "px": True,
         "py": True, "pot": False, "iterator": "DP45", "noise": True, "steps": 2},
        # deterministic spinor model in a potential, fixed RK4 steps in double precision
        {"name": "spinor_480x640_fp64_rk4", "kind": "spinor", "nc": 480, "nr": 640, "prec": "fp64", "px": False, "py": True,
         "pot": True, "iterator": "RK4", "noise": False, "steps": 10},
        # split-step Fourier run
        {"name": "ssfm_1024x512_fp32", "kind": "ssfm", "nc": 1024, "nr": 512, "prec": "fp32", "px": True, "py": True,
         "pot": True, "steps": 10},
        # resonant pulse on top of a continuous pump, in a potential
        {"name": "pulse_512x384_fp32", "kind": "pulse", "nc": 512, "nr": 384, "prec": "fp32", "px": True, "py": True,
         "pot": True, "tetm": False, "npulse": 1, "timed_pump": False, "steps": 10},
        # a parameter sweep: 32 grids of uneven sizes, one pump amplitude and noise seed each
        {"name": "ensemble_32_fp32", "kind": "ensemble", "count": 32, "sizes_seed": 99, "prec": "fp32", "px": True, "py": True,
         "pot": False, "steps": 50},
        # inverse design: gradient of an objective over 16 noise seeds
        {"name": "adjoint_16x512_fp32", "kind": "adjoint", "nc": 512, "nr": 512, "batch": 16, "prec": "fp32", "px": True,
         "py": True, "steps": 100, "checkpoint": 50},
    ]


def _log_int(rng, lo, hi, even=False):
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(hi, max(lo, v + (v & 1 if even else 0)))


def draw(rng):
    kind = rng.choice(["device", "rk4", "rk4", "rk4", "spinor", "spinor", "ssfm", "pulse", "ensemble", "adjoint"])
    c = {"kind": kind, "prec": rng.choice(["fp32", "fp64"])}
    c["px"], c["py"] = rng.choice([(True, True), (True, True), (False, False), (True, False), (False, True)])
    if kind == "ensemble":
        c.update(count=rng.randint(4, 32), sizes_seed=rng.randint(1, 10 ** 6), pot=rng.random() < 0.3, steps=2 * rng.randint(2, 25))
        return c
    lo, hi = {"device": (64, 768), "rk4": (96, 2048), "spinor": (128, 1536), "ssfm": (128, 1024), "pulse": (128, 1024),
              "adjoint": (96, 512)}[kind]
    even = kind not in ("device", "adjoint")  # the configuration surface takes even grids only
    c["nc"] = _log_int(rng, lo, hi, even)
    # most grids are square or nearly so
    c["nr"] = c["nc"] if rng.random() < 0.4 else min(hi, max(lo, _log_int(rng, max(lo, c["nc"] // 2), min(hi, 2 * c["nc"]), even)))
    if rng.random() < 0.35:  # powers of two stay common
        c["nc"] = c["nr"] = 1 << rng.randint((lo - 1).bit_length(), hi.bit_length() - 1)
    cells = c["nc"] * c["nr"]
    most = lambda budget, top: max(1, min(top, int(budget / cells)))  # noqa: E731
    if kind == "device":
        c.update(pot=rng.random() < 0.5, steps=rng.randint(1, 12))
    elif kind == "rk4":
        c.update(pot=rng.random() < 0.4, pump=rng.choice(["gauss", "ring"]), every=0, steps=rng.randint(1, most(1e8, 100)))
        if rng.random() < 0.5:
            c["every"] = rng.choice([1, 2, 5, 10, 25, 50])
            # at most four applications of the filter on the largest grids
            c["steps"] = c["every"] * max(1, min(c["steps"] // c["every"], most(8e6, 8)))
    elif kind == "spinor":
        it = rng.choice(["DP45", "RK4"])
        c.update(pot=rng.random() < 0.5, iterator=it, noise=rng.random() < 0.4, steps=rng.randint(1, most(4e6, 10)))
    elif kind == "ssfm":
        c.update(pot=rng.random() < 0.5, steps=rng.randint(1, most(3e6, 10)))
    elif kind == "pulse":
        c.update(pot=rng.random() < 0.5, tetm=rng.random() < 0.4, npulse=rng.choice([1, 1, 2]), timed_pump=rng.random() < 0.4,
                 steps=rng.randint(1, most(5e6, 12)))
    else:
        c["prec"] = rng.choice(["fp32", "fp32", "fp64"])
        b = max(1, min(16, int(2e6 / cells)))
        c.update(batch=rng.randint(1, b), checkpoint=rng.choice([10, 20, 25, 50]), steps=rng.randint(20, 100))
    return c


# ------------------------------------------------------------------------------------- inputs

def _two(case):
    return case["kind"] == "spinor" or bool(case.get("tetm"))


def _real(case):
    return np.float32 if case["prec"] == "fp32" else np.float64


def _cplx(case):
    return np.complex64 if case["prec"] == "fp32" else np.complex128


def _axes(nc, nr):
    return -0.5 * DX * (nc - 1) + DX * np.arange(nc), -0.5 * DX * (nr - 1) + DX * np.arange(nr)


def _gauss(nc, nr, amp, width, x0=0.0, y0=0.0):
    x, y = _axes(nc, nr)
    return amp * np.exp(-0.5 * ((y - y0) / width) ** 2)[:, None] * np.exp(-0.5 * ((x - x0) / width) ** 2)[None, :]


def _ring(nc, nr, amp, radius, width):
    x, y = _axes(nc, nr)
    r = np.sqrt(y[:, None] ** 2 + x[None, :] ** 2)
    return amp * np.exp(-((r - radius) ** 2) / (2 * width * width))


def _disk(nc, nr, x0, radius):
    x, y = _axes(nc, nr)
    return y[:, None] ** 2 + (x[None, :] - x0) ** 2 <= radius * radius


def _noise(rng, nc, nr, amp, dtype):
    f = rng.standard_normal((nr, nc, 2), dtype=np.float32 if dtype == np.complex64 else np.float64)
    f *= amp
    return f.view(dtype)[..., 0]


def _bumps(rng, nc, nr, count, amp, width):
    f = np.zeros((nr, nc))
    for _ in range(count):
        f += _gauss(nc, nr, rng.uniform(*amp), rng.uniform(*width), rng.uniform(-0.4, 0.4) * DX * nc, rng.uniform(-0.4, 0.4) * DX * nr)
    return f


def _mask(nc, nr):
    """radial super-Gaussian low-pass of exponent 6 with its 1/e radius at 0.8 k_max (k = 0 in the middle)"""
    kx, ky = (np.arange(nc) - nc // 2) / (nc // 2), (np.arange(nr) - nr // 2) / (nr // 2)
    return np.exp(-((ky[:, None] ** 2 + kx[None, :] ** 2) / 0.8 ** 2) ** 6)


def _host_inputs(case, seed):
    """The fields of one case as host arrays in its precision (what a user loads or computes)."""
    rng = np.random.default_rng([seed, 17])
    rd, cd, kind = _real(case), _cplx(case), case["kind"]
    if kind == "ensemble":
        sides = _sides(case)
        out = []
        for N in sides:
            amp = rng.uniform(0.8, 3.0)
            out.append({"psi_plus": _noise(rng, N, N, 0.01, cd), "n_plus": np.zeros((N, N), rd),
                        "pump_plus": _gauss(N, N, amp * P_TH, 10.0).astype(rd)})
            if case["pot"]:
                out[-1]["potential_plus"] = _bumps(rng, N, N, 2, (-5e-4, 5e-4), (5.0, 15.0)).astype(rd)
        return out
    nc, nr = case["nc"], case["nr"]
    span = DX * min(nc, nr)
    if kind == "adjoint":
        P = _bumps(rng, nc, nr, 32, (0.0, 1.0), (5.0, 20.0))
        return {"psi": np.stack([_noise(rng, nc, nr, 0.01, cd) for _ in range(case["batch"])]),
                "n": np.zeros((case["batch"], nr, nc), rd), "pump": (1.5 * P_TH / P.max() * P).astype(rd),
                "pot": _bumps(rng, nc, nr, 32, (-5e-4, 5e-4), (5.0, 20.0)).astype(rd),
                "target": _disk(nc, nr, 0.12 * DX * nc, 0.08 * span).astype(rd)}
    f = {}
    amp = rng.uniform(1.3, 1.7) * P_TH
    ring = case.get("pump") == "ring"
    pump = _ring(nc, nr, amp, min(40.0, 0.25 * span), 5.0) if ring else _gauss(nc, nr, amp, 10.0)
    chi = math.sin(math.pi / 4)  # an elliptically polarised pump splits unevenly over the components
    for k, share in (("plus", 0.5 * (1 + chi)), ("minus", 0.5 * (1 - chi))) if _two(case) else (("plus", 1.0),):
        f["psi_" + k] = _noise(rng, nc, nr, 0.05, cd)
        f["n_" + k] = (0.1 * rng.random((nr, nc))).astype(rd)
        f["pump_" + k] = (share * pump).astype(rd)
        if case["pot"]:
            f["potential_" + k] = _bumps(rng, nc, nr, 3, (-2e-3, 2e-3), (4.0, 12.0)).astype(rd)
    if case.get("every"):
        f["fft_mask_plus"] = _mask(nc, nr).astype(rd)
    return f


def _sides(case):
    r = np.random.default_rng(case["sizes_seed"])
    return [int(n) for n in r.choice(ENSEMBLE_SIDES, size=case["count"])]


def _env(amp, width=10.0, pol="both", time=None):
    a = [amp, "add", width, width, 0, 0, pol, 1, "none", "gauss+noDivide"]
    return a + (["time", *time] if time else [])


def _solver(case, seed):
    nc, nr, kind = case["nc"], case["nr"], case["kind"]
    lx, ly = DX * (nc - 1), DX * (nr - 1)
    b = lambda p: "periodic" if p else "zero"  # noqa: E731
    a = ["--N", nc, nr, "--L", lx, ly, "--boundary", b(case["px"]), b(case["py"]), "--tstep", DT, "--tmax", 1e9, "--outEvery", 1e12,
         "--fftEvery", (case["every"] - 0.5) * DT if case.get("every") else 1e12, "--pump", *_env(CW)]
    if case["pot"]:
        a += ["--potential", *_env(1e-3)]
    if case.get("every"):
        a += ["--fftMask", *_env(1.0)]
    if _two(case):
        a += ["-tetm"]
    if kind == "spinor":
        a += ["--iterator", case["iterator"]]
        if case["iterator"] == "DP45":
            a += ["-adaptive", "--tol", 1e-6, "--rkvdt", 1e-4, 0.1]
        if case["noise"]:
            a += ["--dw", 1, "--initRandom", 0.0, seed % 2 ** 31]
    elif kind == "ssfm":
        a += ["--iterator", "SSFM"]
    elif kind == "pulse":
        if case["timed_pump"]:
            a += ["--pump", *_env(2.0, 8.0, time=("cos", *PUMP_T))]
        a += ["--pulse", *_env(1e-5, 6.0, time=("iexp", *PULSE))]
        if case["npulse"] > 1:
            a += ["--pulse", *_env(2e-5, 9.0, time=("gauss", PULSE[0], PULSE[1], 1.0))]
    return _lib.Solver([str(v) for v in a], case["prec"])


class _DeviceField:
    """A device array of a handle as a zero-copy torch tensor; keeps the handle alive."""

    def __init__(self, ptr, shape, dtype, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": np.dtype(dtype).str, "data": (ptr, False), "version": 3}


def _fields(state):
    """psi and n of a Solver as tensors over its current buffers."""
    s, views = state["solver"], state["views"]
    out = {}
    for name, dtype in state["out"]:
        p = s.device_ptr(name)
        t = views.get(p)
        if t is None:
            t = views[p] = torch.as_tensor(_DeviceField(p, state["shape"], dtype, s), device="cuda")
        out[name] = t
    return out


def prepare(case, seed):
    kind = case["kind"]
    h = _host_inputs(case, seed)
    if kind == "ensemble":
        sides = _sides(case)
        ph, _ = _lib.physics_defaults(512, 512, DX * 511, DX * 511)
        e = _lib.Ensemble(case["prec"], ph, [(N, N) for N in sides], [(DX, DX)] * len(sides), (case["px"], case["py"]),
                          potential=case["pot"])
        for i, f in enumerate(h):
            for name, v in f.items():
                e.set(i, name, v)
        out = []  # an even number of steps leaves every instance in the buffer it started in
        for i, N in enumerate(sides):
            for name, dtype in (("psi_plus", _cplx(case)), ("n_plus", _real(case))):
                out.append(torch.as_tensor(_DeviceField(e.device_ptr(i, name), (N, N), dtype, e), device="cuda"))
        return {"kind": kind, "ensemble": e, "out": out, "steps": case["steps"]}
    if kind in ("device", "adjoint"):
        nc, nr = case["nc"], case["nr"]
        ph, _ = _lib.physics_defaults(nc, nr, DX * (nc - 1), DX * (nr - 1))
        d = {k: torch.from_numpy(v).cuda() for k, v in h.items()}
        st = {"kind": kind, "physics": ph, "steps": case["steps"], "periodic": (case["px"], case["py"])}
        if kind == "adjoint":
            for k in ("pump", "pot", "psi"):
                d[k].requires_grad_(True)
            st.update(d, checkpoint=case["checkpoint"])
        else:
            st.update(prec=_lib.PHX_FP32 if case["prec"] == "fp32" else _lib.PHX_FP64, nc=nc, nr=nr, psi=d["psi_plus"],
                      n=d["n_plus"], psi_b=torch.empty_like(d["psi_plus"]), n_b=torch.empty_like(d["n_plus"]),
                      pump=d["pump_plus"], pot=d.get("potential_plus"))
        return st
    s = _solver(case, seed)
    for name, v in h.items():
        if kind == "pulse" and name.startswith("pump"):
            continue  # the pulse runs take their pumps from the command line
        s.set(name, v)
    comps = ("plus", "minus") if _two(case) else ("plus",)
    out = [(f + k, t) for k in comps for f, t in (("psi_", _cplx(case)), ("n_", _real(case)))]
    return {"kind": kind, "solver": s, "steps": case["steps"], "out": out, "shape": (case["nr"], case["nc"]), "views": {},
            "adaptive": case.get("iterator") == "DP45"}


def run(state):
    kind = state["kind"]
    if kind == "ensemble":
        state["ensemble"].step(DT, state["steps"], graph_steps=state["steps"])
        return state["out"]
    if kind == "device":
        a, pot = state, state["pot"]
        _lib.rk4_scalar_device(a["prec"], a["physics"], a["nc"], a["nr"], a["periodic"], a["psi"].data_ptr(), a["n"].data_ptr(),
                               a["psi_b"].data_ptr(), a["n_b"].data_ptr(), a["pump"].data_ptr(),
                               pot.data_ptr() if pot is not None else None, DT, a["steps"], torch.cuda.current_stream().cuda_stream)
        return a["psi"], a["n"]
    if kind == "adjoint":
        a = state
        psi_T, n_T = rk4_evolve(a["pump"], a["pot"], a["psi"], a["n"], physics=a["physics"], dt=DT, steps=a["steps"],
                                checkpoint_every=a["checkpoint"], periodic=a["periodic"])
        J = (psi_T.abs() ** 2 * a["target"]).sum() * DX * DX
        gP, gV, gpsi = torch.autograd.grad(J, (a["pump"], a["pot"], a["psi"]))
        return {"J": J.detach(), "psi_T": psi_T.detach(), "n_T": n_T.detach(), "g_pump": gP, "g_pot": gV, "g_psi": gpsi}
    s = state["solver"]
    s.step(state["steps"])
    out = _fields(state)
    if state["adaptive"]:
        out["t"] = s.time()[0]
    return out


def work(case):
    kind, r = case["kind"], 4 if case["prec"] == "fp32" else 8
    if kind == "ensemble":
        cells = sum(N * N for N in _sides(case))
    else:
        cells = case["nc"] * case["nr"]
    steps, pot = case["steps"], 1 if case.get("pot") else 0
    # scalar RK4 step: read psi, n, P (, V), write psi, n; four right-hand sides of about 46 operations
    b, fl = (7 + pot) * r, 4 * 46
    if _two(case):
        b, fl = 2 * (7 + pot) * r, (7 if case.get("iterator") == "DP45" else 4) * 2 * 85
        b += 2 * r if case.get("noise") else 0
    if kind == "pulse":
        n = 2 if case["tetm"] else 1
        b += n * (2 * case["npulse"] + (1 if case["timed_pump"] else 0)) * r
    bytes_, flops = float(b) * cells * steps, float(fl) * cells * steps
    fft = 5 * 2 * math.log2(max(2, cells))  # forward and inverse transform, per cell
    if kind == "ssfm":
        # the propagator twice (read and write psi) and the nonlinear step between them on what it left
        bytes_, flops = (2 * 4 + 3 + pot) * r * cells * steps, (2 * fft + 60) * cells * steps
    if case.get("every"):
        k = steps // case["every"]
        bytes_ += 5 * r * cells * k
        flops += fft * cells * k
    if kind == "adjoint":
        # forward, and the adjoint of every step: read state, cotangent, P, V and their gradients, write the latter
        B = case["batch"]
        bytes_ = float(cells) * B * steps * r * (8 + 3 + 3 + 2 + 3 + 4)
        flops = float(cells) * B * steps * (4 * 46 * 2 + 4 * 70)
    return {"bytes": bytes_, "flops": flops}


# ------------------------------------------------------------------------ the same in 64 bits

RK4 = {"c": (0, 0.5, 0.5, 1), "a": ((), (0.5,), (0, 0.5), (0, 0, 1)), "b": (1 / 6, 1 / 3, 1 / 3, 1 / 6), "e": None}
# Dormand, Prince 1980
DP45 = {"c": (0, 1 / 5, 3 / 10, 4 / 5, 8 / 9, 1, 1),
        "a": ((), (1 / 5,), (3 / 40, 9 / 40), (44 / 45, -56 / 15, 32 / 9),
              (19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729),
              (9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656),
              (35 / 384, 0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84)),
        "b": (35 / 384, 0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84, 0),
        "e": (71 / 57600, 0, -71 / 16695, 71 / 1920, -17253 / 339200, 22 / 525, -1 / 40)}


def _pad(f, h, px, py):
    if h == 0 or (px and py):
        return f
    w = (0 if px else h, 0 if px else h, 0 if py else h, 0 if py else h)
    if f.is_complex():
        return torch.complex(torch.nn.functional.pad(f.real, w), torch.nn.functional.pad(f.imag, w))
    return torch.nn.functional.pad(f, w)


def _crop(f, h, px, py):
    return f[..., slice(None) if py else slice(h, -h), slice(None) if px else slice(h, -h)]


def _rhs(psi, n, P, V, F, dx, dy):
    """k_psi and k_n of every component: psi, n, P, V, F are lists (one or two components)."""
    m = -0.5 * H_BAR_S * H_BAR_S / M_EFF
    kp, kn = [], []
    two = len(psi) == 2
    for k, p in enumerate(psi):
        S, N = torch.roll(p, -1, -2), torch.roll(p, 1, -2)
        E, W = torch.roll(p, -1, -1), torch.roll(p, 1, -1)
        lap = (E + W - 2 * p) / dx ** 2 + (N + S - 2 * p) / dy ** 2
        nrm = p.real ** 2 + p.imag ** 2
        h = m * lap + (G_C * nrm + G_R * n[k]) * p
        if V is not None:
            h = h + V[k] * p
        if two:
            o = psi[1 - k]
            So, No = torch.roll(o, -1, -2), torch.roll(o, 1, -2)
            D = torch.roll(So - No, -1, -1) - torch.roll(So - No, 1, -1)
            cross = (torch.roll(o, -1, -1) + torch.roll(o, 1, -1)) / dx ** 2 - (No + So) / dy ** 2
            cross = cross + (0.5j if k == 0 else -0.5j) / (dx * dy) * D
            h = h + G_PM * (o.real ** 2 + o.imag ** 2) * p + DELTA_LT * cross
        q = -1j / H_BAR_S * h + 0.5 * (RR * n[k] - GAMMA_C) * p
        if F is not None:
            q = q + F / H_BAR_S
        kp.append(q)
        kn.append(-(GAMMA_R + RR * nrm) * n[k] + P[k])
    return kp, kn


def _step(tab, psi, n, sources, t, t1, dt, dx, dy, px, py):
    """One explicit Runge-Kutta step; sources(t) -> (P list, V list or None, F or None) at one time.  Outside a
    zero boundary the state starts at zero and evolves within the step.  Returns psi, n and the error sum."""
    S = len(tab["c"])
    h = S + 1
    cut = lambda f: _crop(f, h, px, py) if not (px and py) else f  # noqa: E731
    X = [_pad(p, h, px, py) for p in psi]
    XN = [_pad(v, h, px, py) for v in n]

    def padded(src):
        P, V, F = src
        return ([_pad(p, h, px, py) for p in P], None if V is None else [_pad(v, h, px, py) for v in V],
                None if F is None else _pad(F, h, px, py))

    s0, s1 = padded(sources(t)), padded(sources(t1))
    mix = lambda a, b, w: a if a is b else a * (1 - w) + w * b  # noqa: E731
    Kp, Kn = [], []

    def combine(base, K, w, k):
        for wj, Kj in zip(w, K):
            if wj:
                base = base + dt * wj * Kj[k]
        return base

    for s in range(S):
        w = tab["c"][s]
        Y = [combine(X[k], Kp, tab["a"][s], k) for k in range(len(X))]
        YN = [combine(XN[k], Kn, tab["a"][s], k) for k in range(len(X))]
        P = [mix(a, b, w) for a, b in zip(s0[0], s1[0])]
        V = None if s0[1] is None else [mix(a, b, w) for a, b in zip(s0[1], s1[1])]
        F = None if s0[2] is None else mix(s0[2], s1[2], w)
        kp, kn = _rhs(Y, YN, P, V, F, dx, dy)
        Kp.append(kp)
        Kn.append(kn)
    out = [cut(combine(X[k], Kp, tab["b"], k)) for k in range(len(X))]
    outn = [cut(combine(XN[k], Kn, tab["b"], k)) for k in range(len(X))]
    err = 0.0
    if tab["e"] is not None:
        e = cut(dt * sum(wj * Kj[0] for wj, Kj in zip(tab["e"], Kp) if wj))
        err = len(X) * float((e.real ** 2 + e.imag ** 2).sum())
    return out, outn, err


def _up(v):
    t = torch.from_numpy(np.ascontiguousarray(v)).cuda()
    return t.to(torch.complex128 if t.is_complex() else torch.float64)


def _fft2(f, inverse=False):
    f = f.cpu()  # rows and columns on the host: no transform library on the device is needed
    return (torch.fft.ifft2(f) if inverse else torch.fft.fft2(f)).cuda()


def _time(kind, p, t):
    t0, sigma, fr = p
    if kind == "iexp":
        return complex(np.exp(-complex((t - t0) ** 2 / (2 * sigma * sigma), fr * (t - t0))))
    if kind == "cos":
        return math.exp(-0.5 * ((t - t0) / sigma) ** 2) * (1 + math.cos(fr * (t - t0))) / 2
    return math.exp(-0.5 * (((t - t0) / sigma) ** 2) ** fr)


def exact(case, seed):
    """What run() returns for these inputs in 64 bits; None where a random stream of the framework enters."""
    kind = case["kind"]
    if case.get("noise"):
        return None
    rnd = (lambda v: float(np.float32(v))) if case["prec"] == "fp32" else float  # numbers are read in the case's precision
    px, py, dt, steps = case["px"], case["py"], rnd(DT), case["steps"]
    with torch.no_grad():
        h = _host_inputs(case, seed)
        if kind == "ensemble":
            out = []
            for f in h:
                psi, n, P = [_up(f["psi_plus"])], [_up(f["n_plus"])], [_up(f["pump_plus"])]
                src = (P, [_up(f["potential_plus"])] if case["pot"] else None, None)
                for _ in range(steps):
                    psi, n, _ = _step(RK4, psi, n, lambda t: src, 0, 0, dt, DX, DX, px, py)
                out += [psi[0], n[0]]
            return out
    if kind == "adjoint":
        return _exact_adjoint(case, h, dt)
    with torch.no_grad():
        nc, nr = case["nc"], case["nr"]
        comps = ("plus", "minus") if _two(case) else ("plus",)
        psi, n = [_up(h["psi_" + k]) for k in comps], [_up(h["n_" + k]) for k in comps]
        P = [_up(h["pump_" + k]) for k in comps]
        V = [_up(h["potential_" + k]) for k in comps] if case["pot"] else None
        sources = lambda t: (P, V, None)  # noqa: E731
        if kind == "pulse":
            cw = _up(_gauss(nc, nr, CW, 10.0))
            timed, f1, f2 = _up(_gauss(nc, nr, 2.0, 8.0)), _up(_gauss(nc, nr, 1e-5, 6.0)), _up(_gauss(nc, nr, 2e-5, 9.0))

            def sources(t):
                p = cw + timed * _time("cos", PUMP_T, t) if case["timed_pump"] else cw
                F = f1 * _time("iexp", PULSE, t)
                if case["npulse"] > 1:
                    F = F + f2 * _time("gauss", (PULSE[0], PULSE[1], 1.0), t)
                return [p] * len(comps), V, F
        if kind == "ssfm":
            psi, n = _exact_ssfm(case, psi[0], n[0], P[0], V, dt)
            return {"psi_plus": psi, "n_plus": n}
        mask = torch.fft.ifftshift(_up(h["fft_mask_plus"])) if case.get("every") else None
        t, tab = 0.0, DP45 if case.get("iterator") == "DP45" else RK4
        for k in range(steps):
            t1 = rnd(t + dt)
            new, newn, err = _step(tab, psi, n, sources, t, t1, dt, DX, DX, px, py)
            while tab is DP45:  # step-size control: retries from the advanced time
                norm = float((new[0].real ** 2 + new[0].imag ** 2).sum())
                E = abs(err / norm)
                dt = rnd(max(min(dt * (rnd(1e-6) / 2 / max(E, 2.2250738585072014e-308)) ** 0.25, rnd(0.1)), rnd(1e-4)))
                if E < rnd(1e-6):
                    break
                new, newn, err = _step(tab, psi, n, sources, t1, t1 + dt, dt, DX, DX, px, py)
            psi, n, t = new, newn, t1
            if mask is not None and (k + 1) % case["every"] == 0:
                psi = [_fft2(_fft2(p) * mask, True) for p in psi]
        if kind == "device":
            return psi[0], n[0]
        out = {}
        for k, c in enumerate(comps):
            out["psi_" + c], out["n_" + c] = psi[k], n[k]
        if tab is DP45:
            out["t"] = t
        return out


def _exact_ssfm(case, psi, n, P, V, dt):
    nc, nr = case["nc"], case["nr"]
    kx = torch.from_numpy(2 * 3.1415926535 * np.where(np.arange(nc) <= nc // 2, np.arange(nc), np.arange(nc) - nc) / (DX * (nc - 1))).cuda()
    ky = torch.from_numpy(2 * 3.1415926535 * np.where(np.arange(nr) <= nr // 2, np.arange(nr), np.arange(nr) - nr) / (DX * (nr - 1))).cuda()
    half = torch.exp(-1j * (H_BAR_S / 2 / M_EFF) * (ky[:, None] ** 2 + kx[None, :] ** 2) * dt / 2)
    for _ in range(case["steps"]):
        psi = _fft2(_fft2(psi) * half, True)
        nrm = psi.real ** 2 + psi.imag ** 2
        A = G_C * nrm + G_R * n + (V[0] if V is not None else 0.0)
        psi = psi * torch.exp(torch.complex(0.5 * dt * (RR * n - GAMMA_C), -A * dt / H_BAR_S))
        n = n + dt * (-(GAMMA_R + RR * nrm) * n + P)
        psi = _fft2(_fft2(psi) * half, True)
    return psi, n


def _exact_adjoint(case, h, dt):
    from torch.utils.checkpoint import checkpoint
    px, py = case["px"], case["py"]
    P, V, psi0 = (_up(h[k]).requires_grad_(True) for k in ("pump", "pot", "psi"))
    target = _up(h["target"])

    def one(p, v, psi, n):
        a, b, _ = _step(RK4, [psi], [n], lambda t: ([p], [v], None), 0, 0, dt, DX, DX, px, py)
        return a[0], b[0]

    def run_steps(p, v, psi, n, k):
        for _ in range(k):
            psi, n = checkpoint(one, p, v, psi, n, use_reentrant=False)
        return psi, n

    psi, n = run_steps(P, V, psi0, _up(h["n"]), case["steps"])
    J = ((psi.real ** 2 + psi.imag ** 2) * target).sum() * DX * DX
    gP, gV, gpsi = torch.autograd.grad(J, (P, V, psi0))
    return {"J": J.detach(), "psi_T": psi.detach(), "n_T": n.detach(), "g_pump": gP, "g_pot": gV, "g_psi": gpsi}
