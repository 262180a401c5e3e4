"""The work that a user of the timestep library has it do, as cases to be timed.

Kinds of case, each through the package's public Python API or C ABI:

  step      some steps of one model, then the output fields of the last one
            (what a run does between two outputs);
  state     a whole state to the device, one operator on it, the whole state
            back (what every per-operator static of the C++ API does, and a
            restart);
  poisson   the isolated elliptic solve on device vectors;
  ensemble  some steps of members of uneven grids, then their output fields;
  forward   inference of the guess network;
  grad      loss and gradient of the guess network on a batch of crops.

`listed` names the cases, `draw` gives others of the same ranges, `prepare`
makes what a program holds before the call, `run` is one pass, `work` what a
pass cannot do without, `exact` the outputs in 64 bits where plain numpy or
torch can give them.
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "2d-vector-vorticity-model_amd"))

import vvm_amd as V  # noqa: E402

# the fields a run writes at an output step
OUTPUT = ("zeta", "th", "qv", "qc", "qr", "u", "w")
MEMBER_OUTPUT = ("zeta", "th", "qv", "u", "w")
LARGEST = 4096 * 256  # at 100 m, 256 levels reach as high as the analytic sounding is meant for
# Columns and rows that cannot be halved leave the multigrid hierarchy with a
# large coarsest level; such grids are drawn no larger than this many points
# on it.
COARSEST = 20000
LAYERS, CH, TAPS = 6, 32, 9
LAYER_PARAMS = CH * CH * TAPS + CH


def listed():
    return [
        # one step at a time on the smallest grid of the operator tests: a
        # program that looks at the fields after every step
        {"name": "step 16x12 fp64", "kind": "step", "nx": 16, "nz": 12, "solver": "fp64", "steps": 1},
        # the warm bubble (128x64, dx 200 m) with the library's defaults
        {"name": "step 128x64 fp64", "kind": "step", "nx": 128, "nz": 64, "solver": "fp64", "steps": 20},
        # the 1024x128 surface-flux run, mixed precision
        {"name": "step 1024x128 mixed", "kind": "step", "nx": 1024, "nz": 128, "solver": "mixed", "steps": 20},
        # the benchmark grid, FP64 from a zero guess
        {"name": "step 2048x256 fp64", "kind": "step", "nx": 2048, "nz": 256, "solver": "fp64", "steps": 20},
        # the benchmark grid with the guess network attached
        {"name": "step 2048x256 learned", "kind": "step", "nx": 2048, "nz": 256, "solver": "learned", "steps": 20},
        # a domain whose columns and rows are no powers of two
        {"name": "step 317x61 mixed", "kind": "step", "nx": 317, "nz": 61, "solver": "mixed", "steps": 3},
        # the largest domain: twice the benchmark grid's columns
        {"name": "step 4096x256 mixed", "kind": "step", "nx": 4096, "nz": 256, "solver": "mixed", "steps": 20},
        # state to the device, one operator, state back
        {"name": "state 1024x128", "kind": "state", "nx": 1024, "nz": 128, "op": "microphysics"},
        # the isolated solve of the benchmark grid on a k^-3 vorticity field
        {"name": "poisson 2048x256 fp64", "kind": "poisson", "nx": 2048, "nz": 256, "solver": "fp64"},
        # an ensemble of uneven grids
        {"name": "ensemble 12 members", "kind": "ensemble", "members": 12, "nxmax": 1024, "nzmax": 128, "steps": 4},
        # the guess network over a whole periodic domain
        {"name": "forward 1024x127", "kind": "forward", "batch": 1, "h": 127, "w": 1024, "periodic": True},
        # one training batch of the guess network
        {"name": "grad 16x64x64", "kind": "grad", "batch": 16, "h": 64, "w": 64, "periodic": False},
    ]


def _log(rng, lo, hi):
    """An integer spread evenly over the logarithm of lo..hi."""
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def _coarsest(nx, nz):
    """Points of the level where halving the columns and rows ends."""
    n, m = nx, nz - 1
    while m >= 3 and m % 2 == 1 and n >= 4 and n % 2 == 0:
        n, m = n // 2, (m - 1) // 2
    return n * m


def _grid(rng):
    """A grid of any size: powers of two, multiples of 16, or anything."""
    while True:
        nx, nz = _log(rng, 16, 4096), _log(rng, 12, 256)
        how = rng.random()
        if how < 0.3:
            nx, nz = 1 << (nx.bit_length() - 1), max(16, 1 << (nz.bit_length() - 1))
        elif how < 0.6:
            nx, nz = max(16, nx // 16 * 16), max(16, nz // 16 * 16)
        if nx * nz <= LARGEST and _coarsest(nx, nz) <= COARSEST:
            return nx, nz


def draw(rng):
    how = rng.random()
    if how < 0.5:
        nx, nz = _grid(rng)
        slow = _coarsest(nx, nz) > 2000
        # the FP64 solver's parity rule needs columns that can be halved (its
        # residual falls too slowly on others to be told from round-off)
        solver = rng.choice(("fp64", "mixed")) if nx % 2 == 0 and not slow else "mixed"
        return {"kind": "step", "nx": nx, "nz": nz, "solver": solver, "steps": rng.randint(1, 3 if slow else 10)}
    if how < 0.7:
        nx, nz = _grid(rng)
        solver = rng.choice(("fp64", "mixed")) if nx % 2 == 0 and _coarsest(nx, nz) <= 2000 else "mixed"
        return {"kind": "poisson", "nx": nx, "nz": nz, "solver": solver}
    if how < 0.78:
        nx, nz = _grid(rng)
        return {"kind": "state", "nx": nx, "nz": nz, "op": rng.choice(("microphysics", "turbulence"))}
    if how < 0.86:
        return {"kind": "ensemble", "members": rng.randint(2, 12), "nxmax": rng.choice((256, 512, 1024)),
                "nzmax": rng.choice((64, 128)), "steps": rng.randint(1, 5)}
    if how < 0.93:
        return {"kind": "forward", "batch": 1, "h": _log(rng, 31, 255), "w": _log(rng, 64, 2048), "periodic": True}
    return {"kind": "grad", "batch": rng.randint(1, 16), "h": rng.randint(16, 64), "w": rng.randint(16, 64),
            "periodic": False}


# ----------------------------------------------------------------- states

def _options(solver):
    """Solver options.  The relative stop rule is tighter than the throughput
    benchmark's 1e-10, so that the fields are settled by the equations and not
    by where the iteration stopped."""
    if solver == "fp64":
        return {}
    guess = V.VVM_GUESS_LEARNED if solver == "learned" else V.VVM_GUESS_EXTRAP2
    return dict(solver_mode=V.VVM_SOLVER_MIXED, guess_mode=guess, stop_mode=V.VVM_STOP_REL, tol_rel=1e-12,
                max_iter=1000)


def _model(nx, nz, solver, seed):
    over = _options(solver)
    if (nx, nz) == (16, 12):
        return V.case("tiny", seed=seed, **over)
    if (nx, nz) == (128, 64):
        return V.case("c0", seed=seed, **over)
    return V.grid_case(nx, nz, seed=seed, **over)


def _download(dev, host, names):
    """The named fields of the device's state into the host state's arrays."""
    v = host.view()
    for n, _ in V.VvmHostView._fields_:
        if n in host.a and n not in names:
            setattr(v, n, None)
    rc = dev.lib.vvm_dev_download(dev.h, V.C.byref(v))
    if rc < 0:
        raise V.VvmError(f"download failed ({rc})")
    return {n: host[n] for n in names}


def _members(case, seed):
    rng = np.random.default_rng(case["members"] * 1000 + case["nxmax"] + case["nzmax"])
    out = []
    for k in range(case["members"]):
        nx = int(rng.choice([n for n in (128, 256, 512, 1024) if n <= case["nxmax"]]))
        nz = int(rng.choice([n for n in (64, 128) if n <= case["nzmax"]]))
        out.append((nx, nz, float(rng.uniform(0.05, 0.2)), float(rng.uniform(50, 200)), seed * 64 + k))
    return out


def _k3_field(nx, nz, rng):
    """A Gaussian random vorticity field with a k^-3 power spectrum, RMS
    1e-2 1/s: rows z, columns x (periodic)."""
    kx, kz = np.fft.rfftfreq(nx)[None, :], np.fft.fftfreq(nz)[:, None]
    kk = np.sqrt(kx * kx + kz * kz)
    kk[0, 0] = np.inf
    z = np.fft.irfft2(np.fft.rfft2(rng.standard_normal((nz, nx))) * kk ** -1.5, s=(nz, nx))
    return z * (1e-2 / np.sqrt(np.mean(z * z)))


def _rhs(c, st, seed):
    """cal_w's right-hand side of such a field, in the reference's row order
    (rows k = 2 .. nz-2 of the model's array)."""
    nx, nz = c.cfg.nx - 2, c.cfg.nz - 2
    z = _k3_field(nx, nz, np.random.default_rng(seed))[1:]
    k = np.arange(2, c.cfg.nz - 1)
    return np.ascontiguousarray(st["rhow"][k, None] ** 2 * (np.roll(z, -1, axis=1) - z) * c.cfg.dx).ravel()


def _network(seed):
    rng = np.random.default_rng(seed)
    p = np.zeros((LAYERS, LAYER_PARAMS), dtype=np.float32)
    w = p[:, :CH * CH * TAPS].reshape(LAYERS, CH, CH, TAPS)
    for l in range(LAYERS):
        ci, co = 3 if l == 0 else CH, 1 if l == LAYERS - 1 else CH
        w[l, :co, :ci] = rng.standard_normal((co, ci, TAPS)) * np.sqrt(2.0 / (ci * TAPS))
        p[l, CH * CH * TAPS:CH * CH * TAPS + co] = 0.1 * rng.standard_normal(co)
    return p.ravel()


def _batch(case, seed):
    rng = np.random.default_rng(seed + 1)
    b, h, w = case["batch"], case["h"], case["w"]
    x = rng.standard_normal((b, 3, h, w)).astype(np.float32)
    target = rng.standard_normal((b, h, w)).astype(np.float32)
    mask = np.zeros((b, h, w), dtype=np.float32)
    mask[:, 6:-6, 6:-6] = 1.0  # the network's receptive field
    return x, target, mask


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("step", "state", "poisson"):
        c = _model(case["nx"], case["nz"], case.get("solver", "fp64"), seed % 100000 + 1)
        host = V.init_state(c)
        dev = V.Device(c.cfg)
        dev.upload(host)
        s = {"kind": kind, "dev": dev, "host": host, "case": case}
        if kind == "step":
            if case["solver"] == "learned":
                s["net"] = V.Net()
                s["net"].init_params(seed % 1000 + 1)
                dev.set_guess_net(s["net"])
        elif kind == "state":
            # rain and cloud water, as a run has them once it convects
            rng = np.random.default_rng(seed)
            for f, top in (("qcp", 2e-3), ("qrp", 1e-3)):
                host[f][1:-1, 1:-1] = np.maximum(0.0, rng.uniform(-top, top, (case["nx"], case["nz"])))
            s["out"] = host.copy()
        else:
            s["b"] = torch.from_numpy(_rhs(c, host, seed)).cuda()
            s["x"] = torch.zeros_like(s["b"])
        return s
    if kind == "ensemble":
        opt = _options("mixed")
        cases = [V.grid_case(nx, nz, seed=sd % 100000 + 1, sigma=sg, heat=hf, **opt)
                 for nx, nz, sg, hf, sd in _members(case, seed)]
        ens = V.Ensemble(cases)
        return {"kind": kind, "ens": ens, "hosts": [V.HostState(c.cfg.nx, c.cfg.nz) for c in cases], "case": case}
    net = V.Net()
    net.set_params(_network(seed))
    return {"kind": kind, "net": net, "batch": _batch(case, seed), "case": case}


def run(state):
    kind, case = state["kind"], state["case"]
    if kind == "step":
        state["dev"].step(case["steps"])
        return _download(state["dev"], state["host"], OUTPUT)
    if kind == "state":
        dev, out = state["dev"], state["out"]
        dev.upload(state["host"])
        dev.op(case["op"])
        dev.download(out)
        return {n: out[n] for n in ("zetap", "thp", "qvp", "qcp", "qrp", "RKM", "RKH", "evaporation", "accretion",
                                    "autoconversion", "condensation", "th", "qv", "u", "w", "dth_advect")}
    if kind == "poisson":
        # the handle works on a stream of its own: the guess has to be there
        state["x"].zero_()
        torch.cuda.current_stream().synchronize()
        state["dev"].poisson_device(state["b"].data_ptr(), state["x"].data_ptr())
        return state["x"]
    if kind == "ensemble":
        ens = state["ens"]
        ens.step(case["steps"])
        return [_download(ens.member(i), h, MEMBER_OUTPUT) for i, h in enumerate(state["hosts"])]
    x, target, mask = state["batch"]
    if kind == "forward":
        return state["net"].forward(x, case["periodic"])
    loss, grad = state["net"].grad(x, target, mask, case["periodic"])
    return {"loss": loss, "grad": grad}


# ------------------------------------------------------------------- work

def _step_work(nx, nz, steps, fields):
    """Per step and point: 5 fields, 7 old tendencies, u and w read; 5 fields,
    7 new tendencies, u, w, two coefficients and four rates written; the
    output fields read once and written to the host.  The operations are the
    advection of five fields, microphysics, turbulence, diffusion and a
    direct solve's two transforms."""
    pts = nx * nz
    return {"bytes": pts * 8.0 * (steps * (14 + 20) + 2 * fields), "flops": float(pts * steps * (600.0 + 10 * np.log2(nx)))}


def work(case):
    kind = case["kind"]
    if kind == "step":
        return _step_work(case["nx"], case["nz"], case["steps"], len(OUTPUT))
    if kind == "state":
        # 24 fields and 7 pairs of tendencies there and back
        return {"bytes": case["nx"] * case["nz"] * 8.0 * 38 * 4, "flops": case["nx"] * case["nz"] * 200.0}
    if kind == "poisson":
        n = case["nx"] * (case["nz"] - 1)
        return {"bytes": n * 8.0 * 2, "flops": float(n * (10 * np.log2(case["nx"]) + 10))}
    if kind == "ensemble":
        parts = [_step_work(nx, nz, case["steps"], len(MEMBER_OUTPUT)) for nx, nz, *_ in _members(case, 0)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    px = case["batch"] * case["h"] * case["w"]
    macs = TAPS * (3 * CH + 4 * CH * CH + CH)
    params = 4.0 * LAYERS * LAYER_PARAMS
    if kind == "forward":
        return {"bytes": px * 4.0 * 4 + params, "flops": 2.0 * macs * px}
    return {"bytes": px * 4.0 * 5 + 2 * params, "flops": 6.0 * macs * px}


# ------------------------------------------------------------------ exact

def _exact_poisson(case, seed):
    """The cal_w system (src/PoissonSolver.cpp:760-796) by a Fourier transform
    along the periodic x and a tridiagonal elimination along z."""
    c = _model(case["nx"], case["nz"], case["solver"], 1)
    host = V.HostState(c.cfg.nx, c.cfg.nz)
    # the density profiles of the host-side initial state; no timestep code
    v = host.view()
    if V.load_lib().vvm_init_case(V.C.byref(c.cfg), V.C.byref(c.params), V.C.byref(v)) != 0:
        return None
    rhou, rhow = host["rhou"], host["rhow"]
    n, m = case["nx"], case["nz"] - 1
    b = _rhs(c, host, seed).reshape(m, n)
    k = np.arange(2, 2 + m)
    # row k of A / rhow: cx (x_{i-1} - 2 x + x_{i+1}) + cu_k (x_{k+1} - x_k) - cu_{k-1} (x_k - x_{k-1})
    f = np.fft.rfft(b / rhow[k, None], axis=1)
    lam = 2.0 - 2.0 * np.cos(2.0 * np.pi * np.arange(n // 2 + 1) / n)
    up, dn = 1.0 / rhou[k], 1.0 / rhou[k - 1]
    diag = -(lam[None, :] / rhow[k, None] + (up + dn)[:, None])
    x = np.empty_like(f)
    cp = np.empty_like(diag)
    cp[0], x[0] = up[0] / diag[0], f[0] / diag[0]
    for j in range(1, m):
        den = diag[j] - dn[j] * cp[j - 1]
        cp[j] = up[j] / den
        x[j] = (f[j] - dn[j] * x[j - 1]) / den
    for j in range(m - 2, -1, -1):
        x[j] -= cp[j] * x[j + 1]
    return np.ascontiguousarray(np.fft.irfft(x, n=n, axis=1)).ravel()


def _net64(params, x, periodic):
    """The network in float64, nothing rounded: 3x3 convolutions, tanh GELU
    between them; rows beyond the input are zero, columns wrap if periodic."""
    a = x
    for l in range(LAYERS):
        w = params[l, :CH * CH * TAPS].reshape(CH, CH, 3, 3)
        co, ci = 1 if l == LAYERS - 1 else CH, a.shape[1]
        a = torch.nn.functional.pad(a, (1, 1, 0, 0), mode="circular" if periodic else "constant")
        a = torch.nn.functional.conv2d(torch.nn.functional.pad(a, (0, 0, 1, 1)), w[:co, :ci],
                                       params[l, CH * CH * TAPS:CH * CH * TAPS + co])
        if l < LAYERS - 1:
            a = torch.nn.functional.gelu(a, approximate="tanh")
    return a[:, 0]


def exact(case, seed):
    kind = case["kind"]
    if kind == "poisson":
        return _exact_poisson(case, seed)
    if kind in ("forward", "grad"):
        params = torch.from_numpy(_network(seed)).double().reshape(LAYERS, LAYER_PARAMS)
        x, target, mask = (torch.from_numpy(a).double() for a in _batch(case, seed))
        if kind == "forward":
            return _net64(params, x, case["periodic"])
        params.requires_grad_()
        loss = (mask * (_net64(params, x, case["periodic"]) - target) ** 2).sum() / mask.sum()
        loss.backward()
        return {"loss": float(loss.detach()), "grad": params.grad.reshape(-1)}
    return None
