"""Performance cases of the explicit update path.

Each case is one call sequence of a program that uses this framework:

- api "grid": the driver loop's body on a host-side program: step the resident
  grid by one increment, read the field totals, download the state
  (MMSP.main.hpp's update() then output()). With "fresh" the increment starts
  from an upload, as for a solve of its own.
- api "device": a torch program that keeps its two state buffers in HBM and
  advances them in place (step_noalloc on the current stream).
- api "batch": many independent grids advanced together, every member read.
- api "server": a burst of solve requests through the continuous-batching
  server, every result fetched.

Sizes are the benchmark configurations' and the tests' (512^2, 256^3, 2048^2 x
32 fields, one-hot grains of 16 nodes) or generic ones, odd ones among them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import mmsp_amd as mx

PARAMS = {
    "ac": [1.0, 1.0, 1.0, 1.0, 0.01],
    "ch": [1.0, 1.0, 1.0, 1.0, 0.01],
    "ch_dw": [1.0, 1.0, 0.005],
    "gg": [0.05],
    "zener": [0.01],
    "ostwald": [0.001, 1.0, 1.0, 0.05, 0.95, 2.0, 1.0, 3.0, 2.0],
    "gg_aniso": [0.01, 8.0, 1.0, 1.0],
    "ac_noise": [1.0, 1.0, 1.0, 1.0, 0.01, math.sqrt(2.0), 20260107],
    "ch_noise": [1.0, 1.0, 1.0, 1.0, 0.01, math.sqrt(2.0), 20260107],
}
# initial fields: uniform in these bounds (gg_aniso starts from one-hot grains)
START = {"ac": (-0.01, 0.01), "ch": (-0.01, 0.01), "ch_dw": (0.45, 0.55), "gg": (0.0, 0.01), "zener": (0.0, 1.0),
         "ostwald": (0.0, 1.0), "ac_noise": (-0.01, 0.01), "ch_noise": (-0.01, 0.01)}
VECTOR = ("gg", "zener", "ostwald", "gg_aniso")
P, N, M = mx.PERIODIC, mx.NEUMANN, mx.MIRROR
BOUNDS = {"periodic": [(P, P)] * 3, "neumann": [(N, N)] * 3, "walls": [(N, M), (P, P), (M, N)]}
MOST_UPDATES = 1.2e9  # node x field x step of the largest drawn case


def listed():
    def c(name, api, model, shape, steps, precision="f64", fields=1, bc="periodic", dx=1.0, fresh=False):
        return dict(name=name, api=api, model=model, shape=shape, steps=steps, precision=precision, fields=fields, bc=bc,
                    dx=dx, fresh=fresh)

    return [
        # an interactive run: ten steps of the reference's 128 x 128 example grid, read back each time
        c("ac2d_128_increment", "grid", "ac", "128x128", 10),
        # the 2-D Allen-Cahn benchmark as one solve: upload, 1000 steps, download
        c("ac2d_512_solve", "grid", "ac", "512x512", 1000, fresh=True),
        # a large 3-D Allen-Cahn state advanced by its owner
        c("ac3d_256", "device", "ac", "256x256x256", 50),
        # 2-D Cahn-Hilliard between two written outputs
        c("ch2d_1024_increment", "grid", "ch_dw", "1024x1024", 500),
        # the reference's chemical potential between walls, odd extents
        c("ch2d_333x517_walls", "grid", "ch", "333x517", 200, bc="walls"),
        # the headline workload: 3-D Cahn-Hilliard in double
        c("ch3d_256", "device", "ch_dw", "256x256x256", 100),
        # a mid-sized 3-D solve in single precision, odd extents
        c("ch3d_150x203x97_f32", "grid", "ch_dw", "150x203x97", 400, precision="f32", fresh=True),
        # 2-D grain growth with 32 order parameters
        c("gg2d_2048_q32_f32", "device", "gg", "2048x2048", 20, precision="f32", fields=32),
        # 3-D grain growth with 8 order parameters
        c("gg3d_256_q8_f32", "device", "gg", "256x256x256", 20, precision="f32", fields=8),
        # multi-phase grain growth from grains of 16 nodes
        c("gga2d_1024_q8", "device", "gg_aniso", "1024x1024", 50, fields=8),
        # a parameter study: 32 Allen-Cahn grids of uneven size
        dict(name="batch_ac_32_f32", api="batch", model="ac", members=32, low=96, high=640, layout=4, steps=200,
             precision="f32"),
        # a burst of Cahn-Hilliard requests, short ones in single and long ones in double precision
        dict(name="serve_ch_16", api="server", model="ch_dw", requests=16, low=64, high=384, layout=6, steps=800),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _fit(nodes_fields, steps):
    return max(2, min(steps, int(MOST_UPDATES / nodes_fields)))


def draw(rng):
    kind = rng.choice(["scalar2d", "scalar2d", "scalar2d", "scalar3d", "scalar3d", "scalar3d", "vector2d", "vector3d",
                       "batch", "server"])
    prec = rng.choice(["f64", "f64", "f32"])
    if kind == "batch":
        low = _log(rng, 64, 160)
        return dict(api="batch", model="ac", members=rng.randint(8, 40), low=low, high=low * rng.randint(2, 4),
                    layout=rng.randint(0, 10**6), steps=_log(rng, 50, 300), precision=prec)
    if kind == "server":
        low = _log(rng, 48, 96)
        return dict(api="server", model="ch_dw", requests=rng.randint(6, 18), low=low, high=low * rng.randint(2, 4),
                    layout=rng.randint(0, 10**6), steps=_log(rng, 200, 900))
    if kind == "scalar2d":
        model, fields = rng.choice(["ac", "ac", "ch", "ch_dw", "ch_dw", "ac_noise", "ch_noise"]), 1
        sides = [_log(rng, 48, 1536) for _ in range(2)]
        steps = _log(rng, 8, 1000)
    elif kind == "scalar3d":
        model, fields = rng.choice(["ac", "ac", "ch", "ch_dw", "ch_dw", "ch_noise"]), 1
        sides = [_log(rng, 24, 256) for _ in range(3)]
        steps = _log(rng, 8, 400)
    elif kind == "vector2d":
        model = rng.choice(["gg", "gg", "zener", "ostwald", "gg_aniso"])
        fields = rng.choice([2, 4, 8] if model == "gg_aniso" else [2, 3, 4] if model == "ostwald" else [2, 4, 8, 16, 32])
        sides = [_log(rng, 64, 1536) for _ in range(2)]
        steps = _log(rng, 8, 200)
    else:
        model = rng.choice(["gg", "gg", "zener", "ostwald", "gg_aniso"])
        fields = rng.choice([2] if model == "ostwald" else [2, 4, 8])
        sides = [_log(rng, 24, 192) for _ in range(3)]
        steps = _log(rng, 8, 100)
    if rng.random() < 0.5:  # every other grid on extents a power of two or a multiple of 16 is common
        sides = [max(16, s // 16 * 16) for s in sides]
    bc = "periodic" if rng.random() < 0.75 else rng.choice(["neumann", "walls"])
    dx = rng.choice([1.0, 1.0, 0.8]) if model in ("ac", "gg", "zener") else 1.0
    steps = _fit(float(np.prod(sides)) * fields, steps)
    api = "grid" if len(sides) == 2 and rng.random() < 0.6 or rng.random() < 0.3 else "device"
    return dict(api=api, model=model, shape="x".join(map(str, sides)), steps=steps, precision=prec, fields=fields, bc=bc,
                dx=dx, fresh=rng.random() < 0.5)


def _shape(case):
    return tuple(int(v) for v in case["shape"].split("x"))


def _np(precision):
    return np.float64 if precision == "f64" else np.float32


def _uniform(seed, shape, lo, hi, dtype=np.float64):
    return (lo + (hi - lo) * np.random.default_rng(seed).random(shape)).astype(dtype)


def _layout(case):
    """The extents (and steps) of a batch's members or a server's requests: the program's own work list."""
    r = np.random.default_rng(case["layout"])
    if case["api"] == "batch":
        side = np.exp(r.uniform(math.log(case["low"]), math.log(case["high"]), case["members"])).round().astype(int)
        kappa = r.uniform(0.5, 2.0, case["members"])
        return [((int(s), int(s)), [1.0, 1.0, float(k), 1.0, 0.01]) for s, k in zip(side, kappa)]
    out = []
    for k in range(case["requests"]):
        side = int(round(math.exp(r.uniform(math.log(case["low"]), math.log(case["high"])))))
        steps = int(round(math.exp(r.uniform(math.log(case["steps"] / 8), math.log(case["steps"])))))
        out.append(((side, side) if k % 2 else (max(16, side // 3),) * 3, steps))
    return out


def _initial(case, seed):
    """The field-major initial state, made on the GPU in the case's precision."""
    shape, q = _shape(case), case["fields"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = torch.float64 if case["precision"] == "f64" else torch.float32
    if case["model"] == "gg_aniso":
        ids = torch.randint(0, q, tuple((n + 15) // 16 for n in shape), generator=g, device="cuda")
        for ax, n in enumerate(shape):
            ids = ids.repeat_interleave(16, dim=ax).narrow(ax, 0, n)
        return torch.stack([(ids == j).to(dtype) for j in range(q)]).contiguous()
    lo, hi = START[case["model"]]
    return torch.empty((q,) + shape, dtype=dtype, device="cuda").uniform_(lo, hi, generator=g)


def prepare(case, seed):
    api = case["api"]
    if api == "batch":
        members = _layout(case)
        b = mx.Batch([s for s, _ in members], "ac", precision=case["precision"])
        b.set_params([p for _, p in members])
        for m, (s, _) in enumerate(members):
            b.upload(m, _uniform(seed * 1000 + m, s, -0.01, 0.01, _np(case["precision"])))
        return dict(api=api, batch=b, count=len(members), steps=case["steps"])
    if api == "server":
        work = _layout(case)
        sv = mx.Server("ch_dw", "f32", hbm_budget=8 << 30, max_slots=64, chunk_steps=100,
                       fp64_above_steps=case["steps"] // 2)
        inits = [_uniform(seed * 1000 + k, s, 0.45, 0.55) for k, (s, _) in enumerate(work)]
        return dict(api=api, server=sv, inits=inits, work=work)
    shape, q, vec = _shape(case), case["fields"], case["model"] in VECTOR
    bc, dx = BOUNDS[case["bc"]], (case["dx"],) * 3
    first = _initial(case, seed)
    if api == "device":
        d = mx.make_desc(shape, q, vec, case["precision"], bc, dx)
        return dict(api=api, desc=d, model=case["model"], params=PARAMS[case["model"]], steps=case["steps"],
                    bufs=[first, torch.zeros_like(first)], done=0)
    host = first.movedim(0, -1).contiguous().cpu().numpy()
    g = mx.Grid(shape, q, vec, case["precision"], bc[:len(shape)], dx[:len(shape)])
    host = host if vec else host.reshape(shape)
    g.upload(host)
    return dict(api=api, grid=g, host=host, fresh=case["fresh"], model=case["model"], params=PARAMS[case["model"]],
                steps=case["steps"])


def run(state):
    api = state["api"]
    if api == "device":
        a, b = state["bufs"]
        which = mx.step_noalloc(state["desc"], a.data_ptr(), b.data_ptr(), state["model"], state["params"], state["steps"],
                                first_step=state["done"], stream=torch.cuda.current_stream().cuda_stream)
        if which:
            state["bufs"] = [b, a]
        state["done"] += state["steps"]
        return state["bufs"][0]
    if api == "grid":
        g = state["grid"]
        if state["fresh"]:
            g.upload(state["host"])
        g.step(state["model"], state["params"], state["steps"])
        return {"mass": g.mass(), "state": g.download()}
    if api == "batch":
        b = state["batch"]
        b.step(state["steps"], graph_steps=min(100, state["steps"]))
        return [b.download(m) for m in range(state["count"])]
    sv = state["server"]
    ids = [sv.submit(a, PARAMS["ch_dw"], steps) for a, (_, steps) in zip(state["inits"], state["work"])]
    for i in ids:
        sv.wait(i)
    return [sv.fetch(i) for i in ids]


# operations one node-field update cannot do without, besides 4 per axis for each Laplacian (two for Cahn-Hilliard)
_OPS = {"ac": 9, "ch": 9, "ch_dw": 9, "gg": 11, "zener": 11, "ostwald": 12, "gg_aniso": 30, "ac_noise": 60, "ch_noise": 60}


def work(case):
    def scalar(model, dim, updates):
        laps = 2 if model in ("ch", "ch_dw", "ch_noise") else 1
        return updates * (4 * dim * laps + _OPS[model])

    if case["api"] == "batch":
        nodes = sum(s[0] * s[1] for s, _ in _layout(case))
        return {"bytes": 2 * nodes * (8 if case["precision"] == "f64" else 4),
                "flops": scalar("ac", 2, nodes * case["steps"])}
    if case["api"] == "server":
        work_list = _layout(case)
        return {"bytes": sum(16 * float(np.prod(s)) for s, _ in work_list),
                "flops": sum(scalar("ch_dw", len(s), float(np.prod(s)) * steps) for s, steps in work_list)}
    shape = _shape(case)
    values = float(np.prod(shape)) * case["fields"]
    return {"bytes": 2 * values * (8 if case["precision"] == "f64" else 4),
            "flops": scalar(case["model"], len(shape), values * case["steps"])}


# ---- the same results in plain torch, 64 bits ---------------------------------


def _ends(n, b0, b1, device):
    """Indices of the nodes each node's upper and lower neighbour maps to (check_boundary)."""
    hi, lo = torch.arange(1, n + 1, device=device), torch.arange(-1, n - 1, device=device)
    lo[0] = {P: n - 1, N: 0, M: min(1, n - 1)}[b0]
    hi[-1] = {P: 0, N: n - 1, M: max(n - 2, 0)}[b1]
    return hi, lo


def _laplacian(x, ends, weight):
    out = 0
    for ax, (hi, lo) in enumerate(ends):
        ax += x.dim() - len(ends)
        out = out + weight * (x.index_select(ax, hi) - 2 * x + x.index_select(ax, lo))
    return out


def _ostwald(x, lap, p):
    dt, L, D, ca, cb, A, delta, eps, kappa = p
    cm = 0.5 * (ca + cb)
    B, gam = A / (cb - cm) ** 2, 2.0 / (cb - ca) ** 2
    d = gam / delta ** 2
    C, ph = x[0], x[1:]
    s = (ph ** 2).sum(0)
    w = (-A * (C - cm) + B * (C - cm) ** 3 + d * (C - ca) ** 3 + d * (C - cb) ** 3 - gam * (C - ca) * s -
         kappa * lap(C))
    new = ph - dt * L * (-gam * (C - ca) ** 2 + delta * ph ** 3 + eps * ph * (s - ph ** 2) - kappa * lap(ph))
    return torch.cat([(C + dt * D * lap(w))[None], new])


def _multiphase(x, ends, lap, p):
    dt, width, gamma, mu = p
    eps2 = (4.0 / math.acos(-1.0)) ** 2 * 0.5 * gamma * width
    w = 4.0 * gamma / width
    on = x > 0
    for ax, (hi, lo) in enumerate(ends):
        on = on | (x.index_select(ax + 1, hi) > 0) | (x.index_select(ax + 1, lo) > 0)
    on = on.double()
    S = on.sum(0)
    e = on * (0.5 * eps2 * lap(x) + w * x)
    ph = on * x
    s1, s2 = ph.sum(0), (ph ** 2).sum(0)
    # sum over pairs j < k of the others: ((s1 - ph)^2 - (s2 - ph^2)) / 2
    dF = on * (e.sum(0) - e + 1.5 * ((s1 - ph) ** 2 - (s2 - ph ** 2)))
    rate = -mu * on * (S * dF - dF.sum(0))
    new = (x + dt * 2.0 / S.clamp(min=1) * rate).clamp(0, 1)
    total = new.sum(0)
    new = torch.where(total > 0, new / total, torch.zeros_like(new))
    return torch.where(S >= 2, new, x)


def _advance(x, model, p, steps, ends, dx):
    """`steps` explicit steps of a (fields, *extents) state."""
    def lap(v):
        return _laplacian(v, ends, 1.0 / (dx * dx))

    for _ in range(steps):
        if model == "ac":
            x = x - p[4] * p[3] * (-p[0] * x + p[1] * x ** 3 - p[2] * lap(x))
        elif model == "ch":
            x = x + p[4] * p[3] * lap(-p[0] * x + p[1] * x ** 3 - p[2] * lap(x))
        elif model == "ch_dw":
            x = x + p[2] * p[1] * lap(2 * x * (1 - x) * (1 - 2 * x) - p[0] * lap(x))
        elif model in ("gg", "zener"):
            new = x - p[0] * (-x - x ** 3 + 2 * (x * (x ** 2).sum(0) - lap(x)))
            if model == "zener":
                new[0] = x[0]
            x = new
        elif model == "ostwald":
            x = _ostwald(x, lap, p)
        else:
            x = _multiphase(x, ends, lap, p)
    return x


def _solve(start, model, p, steps, bc, dx):
    x = start.double()
    ends = [_ends(n, b0, b1, x.device) for n, (b0, b1) in zip(x.shape[1:], bc)]
    return _advance(x, model, p, steps, ends, dx)


def exact(case, seed):
    if case["api"] == "batch":
        out = []
        for m, (s, p) in enumerate(_layout(case)):
            a = torch.from_numpy(_uniform(seed * 1000 + m, s, -0.01, 0.01, _np(case["precision"]))).cuda()
            out.append(_solve(a[None], "ac", p, case["steps"], BOUNDS["periodic"], 1.0)[0].cpu())
        return out
    if case["api"] == "server":
        out = []
        for k, (s, steps) in enumerate(_layout(case)):
            a = torch.from_numpy(_uniform(seed * 1000 + k, s, 0.45, 0.55)).cuda()
            a = a if steps > case["steps"] // 2 else a.float()
            out.append(_solve(a[None], "ch_dw", PARAMS["ch_dw"], steps, BOUNDS["periodic"], 1.0)[0].cpu())
        return out
    if case["model"] in ("ac_noise", "ch_noise"):
        return None  # the noise is this repository's own sequence
    x = _solve(_initial(case, seed), case["model"], PARAMS[case["model"]], case["steps"], BOUNDS[case["bc"]], case["dx"])
    if case["api"] == "device":
        return x
    mass = x.reshape(case["fields"], -1).sum(1).cpu().numpy()
    x = x.movedim(0, -1).cpu().numpy()
    return {"mass": mass, "state": x if case["model"] in VECTOR else x.reshape(_shape(case))}
