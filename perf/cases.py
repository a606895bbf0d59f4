"""The solves that users of this library run, as cases to be timed.

Each case goes through a public entry point: SimulateODE (host arrays in and
out, the drop-in call), device-resident plans (executed, or replayed as a
graph), the request server (one request with host outputs; a batch with device
outputs) and the grouped solve.  Sizes span the benchmark's configurations
(parode_amd/synth.py, bench.py) and the reference's study (m = p = 4, up to
128,000 points), with odd and ragged ones between.
"""
import math

import numpy as np
import torch

from parode_amd import api, synth

DEV = "cuda:0"


# ------------------------------------------------------------------- cases
def _case(kind, method, n, m, p, points, precision, states=False, name=None):
    c = dict(kind=kind, method=method, n=n, m=m, p=p, points=points, precision=precision,
             states=states)
    if name:
        c["name"] = name
    return c


def _many(kind, count, sizes, n_hi, points_hi, name=None):
    c = dict(kind=kind, count=count, sizes=sizes, n_hi=n_hi, points_hi=points_hi)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest drop-in call: one small system, host arrays, a UFunc input
        _case("c_abi", api.RK4, 8, 2, 2, 4096, api.PLAIN32, name="c_abi_rk4_n8"),
        # the reference's study at its longest horizon, through the same call
        _case("c_abi", api.ABM, 64, 4, 4, 128000, api.PLAIN32, name="c_abi_abm_n64"),
        # the small plain configuration on device arrays: launch-bound
        _case("plan", api.RK4, 8, 2, 2, 4096, api.PLAIN32, name="plan_rk4_n8_plain"),
        # a control loop that replays one short solve as a graph
        _case("replay", api.ABM, 12, 3, 3, 3000, api.MIXED, name="replay_abm_n12_mixed"),
        # full precision on an odd shape
        _case("plan", api.RK4, 37, 5, 3, 50001, api.FP64, name="plan_rk4_n37_fp64"),
        # every state as an output (no C, no D)
        _case("plan", api.RK4, 48, 6, 48, 65537, api.MIXED, states=True,
              name="plan_rk4_n48_states"),
        # the wide RK4 configuration
        _case("plan", api.RK4, 128, 16, 16, 1 << 18, api.MIXED, name="plan_rk4_n128_mixed"),
        # the long ABM configuration
        _case("plan", api.ABM, 64, 8, 8, 1 << 20, api.MIXED, name="plan_abm_n64_mixed"),
        # a wide, ragged ABM system on a short horizon: the power table dominates
        _case("plan", api.ABM, 203, 25, 25, 30011, api.MIXED, name="plan_abm_n203_mixed"),
        # one request to an idle server, outputs on the host: the latency a client sees
        _case("serve", api.RK4, 24, 3, 3, 9000, api.MIXED, name="serve_one_rk4_n24"),
        # a batch of small systems from sampled inputs
        _many("group", 64, 1, 64, 1 << 14, name="group_64_small"),
        # the batch the benchmark serves: 512 systems, n up to 256, up to 2^18 points
        _many("batch", 512, 0, 256, 1 << 18, name="served_512"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["c_abi", "plan", "plan", "plan", "replay", "serve", "group", "batch"])
    if kind == "group":
        return _many(kind, rng.randint(8, 96), rng.randrange(1 << 20), _log_int(rng, 16, 96),
                     1 << rng.randint(12, 15))
    if kind == "batch":
        return _many(kind, _log_int(rng, 16, 384), rng.randrange(1 << 20),
                     _log_int(rng, 32, 256), 1 << rng.randint(13, 18))
    method = rng.choice([api.RK4, api.ABM])
    n_hi, pts_hi = {"c_abi": (64, 1 << 17), "plan": (256, 1 << 20), "replay": (64, 1 << 14),
                    "serve": (256, 1 << 18)}[kind]
    n = _log_int(rng, 4, n_hi)
    pts = _log_int(rng, 1 << 10, min(pts_hi, (1 << 26) // (n * (4 if method else 1))))
    m = rng.choice([max(1, n // 8), rng.randint(1, max(1, n // 4))])
    p = rng.choice([max(1, n // 8), rng.randint(1, max(1, n // 4))])
    prec = (api.PLAIN32 if kind == "c_abi" else api.MIXED if kind == "serve"
            else rng.choice([api.PLAIN32, api.MIXED, api.MIXED, api.FP64]))
    if prec == api.FP64:
        pts = max(1 << 10, pts // 4)
    states = kind == "plan" and rng.random() < 0.15
    return _case(kind, method, n, m, n if states else p, pts, prec, states)


def _sizes(case):
    """(method, n, m, p, points, h) of every system of a case, from the case alone."""
    if "count" not in case:
        return [(case["method"], case["n"], case["m"], case["p"], case["points"],
                 5e-4 if case["points"] > 1 << 16 else 1e-3)]
    rng = np.random.default_rng(case["sizes"])
    out = []
    for i in range(case["count"]):
        n = int(round(math.exp(rng.uniform(math.log(4), math.log(case["n_hi"])))))
        pts = int(round(2.0 ** rng.uniform(10, math.log2(case["points_hi"]))))
        m = max(1, n // 8)
        out.append((i % 2, n, m, m, pts, float(rng.uniform(1e-4, 1e-3))))
    return out


def _systems(case, seed):
    return [synth.make_system(meth, n, m, p, -5.0, -0.1, h, pts, seed * 1009 + i)
            for i, (meth, n, m, p, pts, h) in enumerate(_sizes(case))]


def _samples(s, seed, dtype, noise=0.1):
    """u on the h/2 grid on the device: the sinusoids of the system, noisy as measured ones."""
    t = torch.arange(2 * s.steps + 1, dtype=torch.float64, device=DEV) * (s.h / 2)
    c = torch.from_numpy(s.ucoef).to(DEV)
    u = torch.sin(t[:, None] * c[:, 4] + c[:, 5])
    if noise:
        g = torch.Generator(device=DEV)
        g.manual_seed(seed)
        u += noise * torch.randn(u.shape, generator=g, dtype=torch.float64, device=DEV)
    return u.to(dtype).contiguous()


# ----------------------------------------------------------------- prepare
_gpu_ready = False


def _init_c_abi():
    global _gpu_ready
    if not _gpu_ready:   # (initialising again would drop the inputs registered so far)
        ids, e = api.get_available_gpus()
        if e or api.initialize_selected_gpus(ids[:1]):
            raise RuntimeError("no GPU")
        _gpu_ready = True


def _device_arrays(s, states):
    f = lambda a: torch.from_numpy(a).to(DEV)
    return [f(s.A), f(s.B), None if states else f(s.C), None if states else f(s.D), f(s.x0)]


def prepare(case, seed):
    kind = case["kind"]
    systems = _systems(case, seed)
    s = systems[0]
    if kind == "c_abi":
        _init_c_abi()
        idx, e = api.register_input(synth.ufunc_source(s.ucoef))
        if e:
            raise RuntimeError(f"RegisterInput: {e}")
        return dict(kind=kind, s=s, u=idx)
    if kind in ("plan", "replay"):
        states, prec = case["states"], case["precision"]
        dt = torch.float32 if prec == api.PLAIN32 else torch.float64
        arrays = _device_arrays(s, states) + [_samples(s, seed, dt)]
        y = torch.zeros((s.steps, case["p"]), dtype=torch.float32, device=DEV)
        plan = api.Plan(s.method, s.n, s.m, case["p"], states, states, s.steps, s.h, prec,
                        dt == torch.float64)
        ptrs = [0 if a is None else a.data_ptr() for a in arrays] + [y.data_ptr()]
        st = dict(kind=kind, plan=plan, ptrs=ptrs, keep=arrays, y=y)
        if kind == "replay":
            torch.cuda.synchronize()
            stream = torch.cuda.Stream()
            plan.capture(*ptrs, stream.cuda_stream)
            torch.cuda.synchronize()
        return st
    sizes = [x.steps * x.p for x in systems]
    off = np.concatenate([[0], np.cumsum(sizes)])
    if kind == "group":
        y = torch.zeros(int(off[-1]), dtype=torch.float32, device=DEV)
        keep, recs = [], []
        for i, x in enumerate(systems):
            a = _device_arrays(x, False) + [_samples(x, seed + i, torch.float64)]
            keep.append(a)
            recs.append(dict(method=x.method, n=x.n, m=x.m, p=x.p, points=x.steps, h=x.h,
                             **{k: t.data_ptr() for k, t in zip("A B C D x0 U".split(), a)},
                             Y=y.data_ptr() + 4 * int(off[i])))
        return dict(kind=kind, group=api.Group(recs), keep=keep, y=y)
    need = sum(api.Server.footprint(x.method, x.n, x.m, x.p, x.steps) for x in systems)
    srv = api.Server(lanes=8, device_bytes=int(need * 1.1) + (1 << 30),
                     pinned_bytes=1 << 28, precision=api.MIXED)
    if kind == "serve":
        return dict(kind=kind, server=srv, s=s)
    y = torch.zeros(int(off[-1]), dtype=torch.float32, device=DEV)
    items = [(x.method, x.A, x.B, x.C, x.D, x.x0, x.steps, x.h, y.data_ptr() + 4 * int(o),
              x.ucoef) for x, o in zip(systems, off)]
    return dict(kind=kind, server=srv, items=items, y=y)


# --------------------------------------------------------------------- run
def run(state):
    kind = state["kind"]
    if kind == "c_abi":
        s = state["s"]
        tv, xv, e = api.simulate_ode(s.method, s.A, s.B, s.C, s.D, state["u"], s.t0, s.t_end, s.h,
                                     s.x0)
        return dict(t=tv, x=xv, err=e)
    if kind == "plan":
        state["plan"].execute(*state["ptrs"], 0)
        return state["y"]
    if kind == "replay":
        state["plan"].replay(0)
        return state["y"]
    if kind == "group":
        state["group"].execute(0)
        return state["y"]
    if kind == "serve":
        s, srv = state["s"], state["server"]
        ticket, y = srv.submit(s.method, s.A, s.B, s.C, s.D, s.x0, s.steps, s.h, coef=s.ucoef)
        status = srv.wait(ticket)[0]
        return dict(y=y, status=status)
    srv = state["server"]
    status = srv.wait_batch(srv.submit_device_batch(state["items"]))[0]
    return dict(y=state["y"], status=status)


# -------------------------------------------------------------------- work
def work(case):
    """Matrices, samples (or their coefficients) read once, outputs written
    once; per step one product with the step map (ABM: with A, twice), the
    input and the output products."""
    kind = case["kind"]
    b = f = 0.0
    for meth, n, m, p, pts, _ in _sizes(case):
        states = case.get("states", False)
        b += 4.0 * (n * n + n * m + n + pts * p) + (0 if states else 4.0 * p * (n + m))
        if kind in ("plan", "replay", "group"):
            plain = case.get("precision") == api.PLAIN32
            b += (pts if meth else 2 * pts + 1) * m * (4.0 if plain else 8.0)
        else:
            b += 48.0 * m
        f += pts * (2.0 * n * n * (2 if meth else 1) + 2.0 * n * m * (2 if meth else 3) +
                    (0 if states else 2.0 * p * (n + m)))
    return dict(bytes=b, flops=f)


# ------------------------------------------------------------------- exact
def _trajectory(M, V, x0):
    """x_0 = x0, x_{e+1} = M x_e + V_e (rows of V), e < len(V): chunks in step,
    then the chunks' starts, then every state."""
    N, na = V.shape
    lc = 7 if N >= 4096 else 5
    T = 1 << lc
    nc = -(-N // T)
    V = torch.nn.functional.pad(V, (0, 0, 0, nc * T - N)).view(nc, T, na)
    MT = M.T.contiguous()
    a = torch.zeros((nc, na), dtype=torch.float64, device=DEV)
    for t in range(T):
        a = torch.addmm(V[:, t], a, MT)
    P = MT
    for _ in range(lc):
        P = P @ P
    b = torch.cat([x0[None], a])[:nc]
    d = 1
    while d < nc:   # inclusive scan: b_c = sum_{q <= c} P^(c-q) b_q
        b = torch.cat([b[:d], torch.addmm(b[d:], b[:-d], P)])
        P = P @ P
        d *= 2
    X = torch.empty((nc, T, na), dtype=torch.float64, device=DEV)
    for t in range(T):
        X[:, t] = b
        b = torch.addmm(V[:, t], b, MT)
    return X.view(nc * T, na)[:N]


def _solve64(s, U, states):
    """Outputs of one system in 64 bits; U: samples on the h/2 grid."""
    f = lambda a: torch.from_numpy(a).to(DEV).double()
    A, B, C, D, x0, h = f(s.A), f(s.B), f(s.C), f(s.D), f(s.x0), s.h
    U = U.double()
    n, N = s.n, s.steps
    eye = torch.eye(n, dtype=torch.float64, device=DEV)
    if s.method == api.RK4:
        A2 = A @ A
        A3 = A2 @ A
        M = eye + h * A + h**2 / 2 * A2 + h**3 / 6 * A3 + h**4 / 24 * (A2 @ A2)
        B1 = (h * B + h**2 * (A @ B) + h**3 / 2 * (A2 @ B) + h**4 / 4 * (A3 @ B)) / 6
        B2 = (4 * h * B + 2 * h**2 * (A @ B) + h**3 / 2 * (A2 @ B)) / 6
        B3 = h / 6 * B
        V = U[0:2 * N:2] @ B1.T + U[1:2 * N:2] @ B2.T + U[2:2 * N + 1:2] @ B3.T
        X = _trajectory(M, V, x0)
    else:
        xs = [x0]   # three classic RK4 steps
        for k in range(3):
            x, u0, u1, u2 = xs[-1], U[2 * k], U[2 * k + 1], U[2 * k + 2]
            k1 = A @ x + B @ u0
            k2 = A @ (x + h / 2 * k1) + B @ u1
            k3 = A @ (x + h / 2 * k2) + B @ u1
            k4 = A @ (x + h * k3) + B @ u2
            xs.append(x + h / 6 * (k1 + 2 * k2 + 2 * k3 + k4))
        A2, AB, q = A @ A, A @ B, h * h / 576
        a = [(0, -81), (1, 333), (-5, -531), (28, 495)]   # AB4 predictor in the AM4 corrector
        b = [(0, -81), (1, 333), (-5, -531), (19, 495), (9, 0)]
        M = torch.zeros((4 * n, 4 * n), dtype=torch.float64, device=DEV)
        M[:3 * n, n:] = torch.eye(3 * n, dtype=torch.float64, device=DEV)
        for i, (c1, c2) in enumerate(a):
            M[3 * n:, i * n:(i + 1) * n] = c1 * h / 24 * A + q * c2 * A2
        M[3 * n:, 3 * n:] += eye
        ns = N - 3
        E = U[0::2]
        V = torch.zeros((ns, 4 * n), dtype=torch.float64, device=DEV)
        for i, (c1, c2) in enumerate(b):
            V[:, 3 * n:] += E[i:i + ns] @ (c1 * h / 24 * B + q * c2 * AB).T
        X = torch.cat([torch.stack(xs[:3]), _trajectory(M, V, torch.cat(xs))[:, 3 * n:]])
    return X if states else X @ C.T + U[0:2 * N:2] @ D.T


def exact(case, seed):
    kind = case["kind"]
    systems = _systems(case, seed)
    s = systems[0]
    if kind == "c_abi":
        # the call samples its input function on a grid of 32-bit times
        k = torch.arange(2 * s.steps + 1, device=DEV).float()
        t = (k * float(np.float32(s.h / 2))).double()
        c = torch.from_numpy(s.ucoef).to(DEV)
        y = _solve64(s, torch.sin(t[:, None] * c[:, 4] + c[:, 5]), False)
        return dict(t=np.arange(s.steps) * s.h, x=y, err=None)
    if kind in ("plan", "replay"):
        dt = torch.float32 if case["precision"] == api.PLAIN32 else torch.float64
        return _solve64(s, _samples(s, seed, dt), case["states"])
    if kind == "group":
        return torch.cat([_solve64(x, _samples(x, seed + i, torch.float64), False).reshape(-1)
                          for i, x in enumerate(systems)])
    ys = [_solve64(x, _samples(x, 0, torch.float64, 0.0), False).reshape(-1) for x in systems]
    if kind == "serve":
        return dict(y=ys[0].view(s.steps, s.p), status=None)
    return dict(y=torch.cat(ys), status=None)
