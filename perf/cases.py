"""What the framework's speed is measured on.

Each case is one piece of work that a user of libmcb has it do, through the
Python binding of its C ABI: a lattice advanced to its next snapshot, a batch
of uneven cases, a serving round, the reference's kernels on the caller's own
buffers, the diagnostics. listed() names the standing cases, draw() gives
further ones of the same ranges; prepare() makes what a program holds before
the call, run() is one pass, work() what a pass cannot do without, exact() the
same outputs in 64 bits from plain torch.
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "multic-bubble-cuda_amd"))
import mcb  # noqa: E402

STORAGE = {"fp32": mcb.STORE_FP32, "fp16": mcb.STORE_FP16, "bf16": mcb.STORE_BF16}
WIDTH = 3.0
DEVICE = "cuda" if torch.cuda.is_available() else "cpu"


def listed():
    def lattice(name, nx, ny, nz, storage, tau_f, tau_g, steps, fields, bc="periodic", bubbles=1):
        return {"name": name, "kind": "lattice", "nx": nx, "ny": ny, "nz": nz, "storage": storage, "bc": bc,
                "tau_f": tau_f, "tau_g": tau_g, "sigma": 0.1, "bubbles": bubbles, "steps": steps, "fields": fields}

    return [
        # Monitoring: the FP64 sum of phi and kinetic energy of fields that the
        # caller holds, as code under graph capture or a loop that must not
        # allocate calls it. The smallest call; launches and latency.
        {"name": "diagnostics 64^3", "kind": "reduce", "nx": 64, "ny": 64, "nz": 64},
        # A small periodic case (the 'cfg0' preset's lattice) to its next
        # snapshot with velocity: latency and launches count. g as populations.
        lattice("small 64^3 tau_g 0.8", 64, 64, 64, "fp32", 0.55, 0.8, 100, "all"),
        # The reference's own case (the 'reference' preset: ghost-layer
        # boundaries, one centred bubble) to its next phi snapshot.
        lattice("reference 64x64x256", 64, 64, 256, "fp32", 0.505, 1.0, 100, "phi", bc="reference"),
        # A mid-size periodic case with g as populations (the 'cfg1' preset).
        lattice("mid 128^3 tau_g 0.8", 128, 128, 128, "fp32", 0.55, 0.8, 100, "all"),
        # The headline case (the 'cfg2' preset) to its next phi snapshot, in
        # FP32 and with populations stored as FP16.
        lattice("large 256^3 fp32", 256, 256, 256, "fp32", 0.52, 1.0, 100, "phi", bubbles=2),
        lattice("large 256^3 fp16", 256, 256, 256, "fp16", 0.52, 1.0, 100, "phi", bubbles=2),
        # The largest serving side, stored as BF16.
        lattice("serving side 192^3 bf16", 192, 192, 192, "bf16", 0.6, 1.0, 100, "phi"),
        # Sides that no tile or layout was made for, one of them odd: a channel
        # someone cuts to their own experiment, in FP32 and in FP16.
        lattice("ragged 150x105x77 fp32", 150, 105, 77, "fp32", 0.6, 1.0, 100, "all"),
        lattice("ragged 117x90x133 fp16", 117, 90, 133, "fp16", 0.6, 1.0, 100, "phi"),
        # A sweep of uneven cases advanced together in FP32 (the 'batch'
        # presets' sides and parameters), phi of every case read afterwards.
        {"name": "batch of 32 fp32", "kind": "batch", "cases": 32, "mix": 1, "storage": "fp32", "steps": 50},
        # The serving loop: requests of uneven size and length (the 'serve'
        # presets' ranges, step counts x 0.1) arriving at once, FP16.
        {"name": "serve 24 requests fp16", "kind": "serve", "requests": 24, "mix": 2, "storage": "fp16"},
        # The reference's kernels, one entry point each, over the caller's own
        # device buffers: one iteration of its loop on its own lattice.
        {"name": "operators 64x64x256", "kind": "ops", "nx": 64, "ny": 64, "nz": 256, "bc": "reference"},
    ]


def draw(rng):
    def side(lo, hi):
        v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        how = rng.random()
        return v if how < 0.5 else (max(lo, v // 2 * 2) if how < 0.7 else max(lo, min(hi, (v + 8) // 16 * 16)))

    kind = rng.choice(["lattice"] * 7 + ["batch", "serve", "ops", "ops", "reduce"])
    if kind == "reduce":
        return {"kind": kind, "nx": side(32, 256), "ny": side(32, 256), "nz": side(32, 256)}
    if kind == "ops":
        return {"kind": kind, "nx": side(32, 128), "ny": side(32, 128), "nz": side(32, 256),
                "bc": rng.choice(["reference", "periodic"])}
    if kind == "batch":
        return {"kind": kind, "cases": rng.randint(8, 32), "mix": rng.randint(100, 10 ** 6),
                "storage": rng.choice(["fp32", "fp32", "fp16", "bf16"]), "steps": rng.randint(20, 50)}
    if kind == "serve":
        return {"kind": kind, "requests": rng.randint(6, 20), "mix": rng.randint(100, 10 ** 6),
                "storage": rng.choice(["fp16", "bf16"])}
    bc = rng.choice(["periodic"] * 4 + ["reference"])
    storage = "fp32" if bc == "reference" else rng.choice(["fp32", "fp32", "fp16", "bf16"])
    tau_g = 1.0 if bc == "reference" else rng.choice([1.0, 1.0, 0.8])
    nx, ny, nz = side(32, 256), side(32, 256), side(32, 256)
    small = nx * ny * nz <= 3 << 20
    return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "storage": storage, "bc": bc,
            "tau_f": round(rng.uniform(0.55, 0.8), 3), "tau_g": tau_g, "sigma": round(rng.uniform(0.01, 0.1), 3),
            "bubbles": rng.randint(1, 2), "steps": rng.randint(20, 100),
            "fields": "all" if small and storage == "fp32" and rng.random() < 0.5 else "phi"}


# ------------------------------------------------------------------- inputs

def _f32(v):
    return float(np.float32(v))


def _bubbles(r, sides, n, bc):
    """n bubbles of 0.12 to 0.28 of the shortest side: anywhere in a periodic box, near the centre between walls."""
    out = []
    s = min(sides)
    for _ in range(n):
        if bc == "reference":
            c = [v * 0.5 + r.uniform(-0.05, 0.05) * v for v in sides]
        else:
            c = [r.uniform(0, v) for v in sides]
        out.append(tuple(_f32(v) for v in (*c, r.uniform(0.12, 0.28) * s)))
    return out


def _lattice_params(case):
    ref = case["bc"] == "reference"
    return mcb.make_params(case["nx"], case["ny"], case["nz"], bc_mode=mcb.BC_REFERENCE if ref else mcb.BC_PERIODIC,
                           weights=mcb.WEIGHTS_LITERAL if ref else mcb.WEIGHTS_UNIT_SUM,
                           storage=STORAGE[case["storage"]], tau_f=case["tau_f"], tau_g=case["tau_g"],
                           sigma=case["sigma"])


def _lattice_bubbles(case, seed):
    return _bubbles(random.Random(seed * 7919 + 1), (case["nx"], case["ny"], case["nz"]), case["bubbles"], case["bc"])


def _batch_cases(case, seed):
    """Cubes with the sides and parameter ranges of the 'batch' presets; the sides are the case's, the rest the seed's."""
    mix, r = random.Random(case["mix"]), random.Random(seed * 7919 + 2)
    out = []
    for _ in range(case["cases"]):
        side = mix.choice([32, 48, 64, 96, 128])
        out.append({"side": side, "sigma": r.uniform(0.01, 0.1), "tau_f": r.uniform(0.52, 0.8),
                    "bubble": tuple(_f32(v) for v in (*(r.uniform(0, side) for _ in range(3)),
                                                      r.uniform(0.15, 0.3) * side))})
    return out


def _serve_cases(case, seed):
    """Requests with the ranges of the 'serve' presets, step counts x 0.1; sides and step counts are the case's."""
    mix, r = random.Random(case["mix"]), random.Random(seed * 7919 + 3)
    out = []
    for _ in range(case["requests"]):
        side = 48 + 16 * mix.randrange(10)
        steps = int(round(50.0 * 10.0 ** mix.random()))
        out.append({"side": side, "steps": steps, "sigma": r.uniform(0.01, 0.1), "tau_f": r.uniform(0.52, 0.8),
                    "bubble": tuple(_f32(v) for v in (*(r.uniform(0, side) for _ in range(3)),
                                                      r.uniform(0.1, 0.3) * side))})
    return out


def _cube_params(c, storage):
    return mcb.make_params(c["side"], c["side"], c["side"], storage=STORAGE[storage], tau_f=c["tau_f"], tau_g=1.0,
                           sigma=c["sigma"])


def _flow(case, seed, dtype, device):
    """Fields of a bubble in a weak flow, as a program holds them between steps: phi, rho and u of a droplet with a
    swirl of a few hundredths, the same values whatever the type (they are made in 64 bits and rounded to 32)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    r = random.Random(seed * 7919 + 4)
    bub = _bubbles(r, (nx, ny, nz), 1, case.get("bc", "periodic"))
    phi = _phi0(nx, ny, nz, bub, case.get("bc", "periodic") == "reference", device)
    ax = [torch.arange(v, dtype=torch.float64, device=device) * (2 * math.pi / v) for v in (nx, ny, nz)]
    X, Y, Z = ax[0][None, None, :], ax[1][None, :, None], ax[2][:, None, None]
    p = [r.uniform(0, 2 * math.pi) for _ in range(4)]
    ux = 0.02 * torch.sin(Y + p[0]) * torch.cos(Z + p[1]) + 0 * X
    uy = 0.02 * torch.sin(Z + p[1]) * torch.cos(X + p[2]) + 0 * Y
    uz = 0.02 * torch.sin(X + p[2]) * torch.cos(Y + p[0]) + 0 * Z
    rho = 1.0 + 0.002 * torch.cos(X + Y + Z + p[3])
    return [v.to(torch.float32).to(dtype).contiguous() for v in (phi, rho, ux, uy, uz)]


# ------------------------------------------------------------------ prepare

OP_FIELDS = ("phi", "rho", "ux", "uy", "uz", "ffx", "ffy", "ffz", "normx", "normy", "normz", "indicator", "curvature",
             "pxx", "pyy", "pzz", "pxy", "pxz", "pyz")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "lattice":
        lat = mcb.Lattice(_lattice_params(case))
        lat.init_bubbles(_lattice_bubbles(case, seed), WIDTH)
        return {"kind": kind, "lat": lat, "steps": case["steps"], "fields": case["fields"]}
    if kind == "batch":
        b = mcb.Batch(STORAGE[case["storage"]])
        ids = [b.add(_cube_params(c, case["storage"]), [c["bubble"]], WIDTH) for c in _batch_cases(case, seed)]
        return {"kind": kind, "batch": b, "ids": ids, "steps": case["steps"]}
    if kind == "serve":
        todo = _serve_cases(case, seed)
        reqs = (mcb.Request * len(todo))()
        phi = [np.zeros((c["side"],) * 3, dtype=np.float32) for c in todo]
        for q, c, out in zip(reqs, todo, phi):
            q.c.params = _cube_params(c, case["storage"])
            q.c.n_bubbles, q.c.width, q.c.nsteps, q.c.save_every = 1, WIDTH, c["steps"], c["steps"]
            q.c.bubbles[0] = mcb.Bubble(*c["bubble"])
            q.arrival_s = 0.0
            q.phi_out = out.ctypes.data_as(ctypes.POINTER(ctypes.c_float))
        return {"kind": kind, "reqs": reqs, "phi": phi, "storage": STORAGE[case["storage"]]}
    phi, rho, ux, uy, uz = _flow(case, seed, torch.float32, DEVICE)
    if kind == "reduce":
        out = torch.zeros(2, dtype=torch.float64, device=DEVICE)
        return {"kind": kind, "fields": [phi, rho, ux, uy, uz], "shape": (case["nx"], case["ny"], case["nz"]),
                "out": out}
    # The reference's device buffers (src/var.cu:13-18): populations at equilibrium, which the caller's own set-up
    # leaves there, and every field of the loop.
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    f, g = _equilibrium(phi, rho, ux, uy, uz)
    buf = {k: torch.zeros((nz, ny, nx), dtype=torch.float32, device=DEVICE) for k in OP_FIELDS}
    for k, v in (("phi", phi), ("rho", rho), ("ux", ux), ("uy", uy), ("uz", uz)):
        buf[k].copy_(v)
    buf["f"], buf["g"], buf["g_out"] = f, g, torch.zeros_like(g)
    params = mcb.make_params(nx, ny, nz, bc_mode=mcb.BC_REFERENCE if case["bc"] == "reference" else mcb.BC_PERIODIC,
                             weights=mcb.WEIGHTS_LITERAL, tau_f=0.505, tau_g=1.0, sigma=0.1)
    return {"kind": kind, "buf": buf, "shape": (nx, ny, nz), "consts": mcb.op_consts(params),
            "walls": case["bc"] == "reference"}


def _equilibrium(phi, rho, ux, uy, uz):
    """f = w rho (1 + 3 c.u) and g = w phi in float32: a state to start the loop from."""
    f = torch.empty((19,) + tuple(phi.shape), dtype=torch.float32, device=phi.device)
    g = torch.empty_like(f)
    for l in range(19):
        w = float(np.float32(W[l]))
        f[l] = w * rho * (1 + 3 * (CX[l] * ux + CY[l] * uy + CZ[l] * uz))
        g[l] = w * phi
    return f, g


# ---------------------------------------------------------------------- run

def run(state):
    kind = state["kind"]
    if kind == "lattice":
        lat = state["lat"]
        lat.step(state["steps"])
        return lat.observables() if state["fields"] == "all" else {"phi": lat.read("phi")}
    if kind == "batch":
        b = state["batch"]
        b.step(state["steps"])
        return [b.read(i, "phi") for i in state["ids"]]
    if kind == "serve":
        res, _ = mcb.serve(state["reqs"], storage=state["storage"])
        return {"phi": state["phi"], "status": np.array([r.status for r in res])}
    stream = torch.cuda.current_stream().cuda_stream
    nx, ny, nz = state["shape"]
    if kind == "reduce":
        ptr = [v.data_ptr() for v in state["fields"]]
        mcb.check(mcb.lib().mcb_reduce_fields_noalloc(*ptr, nx, ny, nz, state["out"].data_ptr(), stream))
        return state["out"]
    b, c = state["buf"], state["consts"]

    def op(name, *fields):
        mcb.op(name, *[b[k].data_ptr() for k in fields], nx, ny, nz, c, stream)

    # One iteration of the reference's loop (src/main.cu:79-178).
    op("phiCalc", "phi", "g")
    op("gradCalc", "phi", "normx", "normy", "normz", "indicator")
    op("curvatureCalc", "curvature", "indicator", "normx", "normy", "normz", "ffx", "ffy", "ffz")
    op("momentiCalc", "ux", "uy", "uz", "rho", "ffx", "ffy", "ffz", "f", "pxx", "pyy", "pzz", "pxy", "pxz", "pyz")
    op("collisionFluid", "f", "ux", "uy", "uz", "ffx", "ffy", "ffz", "rho", "pxx", "pyy", "pzz", "pxy", "pxz", "pyz")
    op("collisionPhase", "g", "ux", "uy", "uz", "phi", "normx", "normy", "normz")
    op("streamingCalc", "g", "g_out")
    b["g"], b["g_out"] = b["g_out"], b["g"]
    if state["walls"]:
        op("fgBoundary", "f", "rho", "g", "phi")
        op("boundaryConditions", "phi")
    return {k: b[k] for k in ("f", "g", "phi", "rho", "ux", "uy", "uz")}


# --------------------------------------------------------------------- work

def work(case):
    """Bytes: each step reads and writes the state once (f; g as populations, or the few values per cell that
    determine it at tau_g = 1), and the outputs are written once. Operations: about 900 a cell and step."""
    def step_bytes(storage, tau_g):
        pop = 4 if storage == "fp32" else 2
        f = 2 * 19 * pop
        if tau_g != 1.0:
            return 2 * f
        return f + (2 * 16 if storage == "fp32" else 2 * 10)

    kind = case["kind"]
    if kind == "lattice":
        n = case["nx"] * case["ny"] * case["nz"]
        out = 4 * n * (5 if case["fields"] == "all" else 1)
        return {"bytes": case["steps"] * n * step_bytes(case["storage"], case["tau_g"]) + out,
                "flops": 900.0 * case["steps"] * n}
    if kind == "batch":
        n = sum(c["side"] ** 3 for c in _batch_cases(case, 0))
        return {"bytes": case["steps"] * n * step_bytes(case["storage"], 1.0) + 4 * n,
                "flops": 900.0 * case["steps"] * n}
    if kind == "serve":
        todo = _serve_cases(case, 0)
        n = sum(c["side"] ** 3 * c["steps"] for c in todo)
        return {"bytes": n * step_bytes(case["storage"], 1.0) + 4 * sum(c["side"] ** 3 for c in todo),
                "flops": 900.0 * n}
    n = case["nx"] * case["ny"] * case["nz"]
    if kind == "reduce":
        return {"bytes": 5 * 4 * n + 16, "flops": 9.0 * n}
    # Each operator reads its input fields and writes its output fields once.
    return {"bytes": n * 4 * ((19 + 1) + (1 + 4) + (4 + 4) + (3 + 19 + 10) + (13 + 19) + (7 + 19) + (19 + 19)),
            "flops": 900.0 * n}


# -------------------------------------------------------------------- exact
# The same model in 64 bits, from its equations: D3Q19, pull form, one array operation per term.

CX = [0, 1, -1, 0, 0, 0, 0, 1, -1, 1, -1, 0, 0, 1, -1, 1, -1, 0, 0]
CY = [0, 0, 0, 1, -1, 0, 0, 1, -1, 0, 0, 1, -1, -1, 1, 0, 0, 1, -1]
CZ = [0, 0, 0, 0, 0, 1, -1, 0, 0, 1, -1, 1, -1, 0, 0, -1, 1, -1, 1]
W = [1.0 / 3.0] + [1.0 / 18.0] * 6 + [1.0 / 36.0] * 12
SHARP = 0.15 * 3.0
PAIRS = ((1, 2), (3, 4), (5, 6), (7, 8), (9, 10), (11, 12), (13, 14), (15, 16), (17, 18))


def _phi0(nx, ny, nz, bubbles, walls, device):
    """The tanh profile of the bubbles, nearest images in a periodic box, zero on the faces between walls."""
    ax = [torch.arange(v, dtype=torch.float64, device=device) for v in (nx, ny, nz)]
    phi = torch.zeros((nz, ny, nx), dtype=torch.float64, device=device)
    for cx, cy, cz, r in bubbles:
        d = []
        for a, c, n in zip(ax, (cx, cy, cz), (nx, ny, nz)):
            v = a - c
            if not walls:
                v = torch.where(v > n * 0.5, v - n, torch.where(v < -n * 0.5, v + n, v))
            d.append(v * v)
        dist = torch.sqrt(d[0][None, None, :] + d[1][None, :, None] + d[2][:, None, None])
        phi = torch.maximum(phi, 0.5 + 0.5 * torch.tanh(2.0 * (r - dist) / WIDTH))
    if walls:
        phi *= _interior(phi.shape, device)
    return phi.to(torch.float32).to(torch.float64)


def _interior(shape, device):
    m = torch.zeros(shape, dtype=torch.float64, device=device)
    m[1:-1, 1:-1, 1:-1] = 1.0
    return m


def _clamped_faces(v):
    v = v.clone()
    v[0], v[-1] = v[1], v[-2]
    v[:, 0], v[:, -1] = v[:, 1], v[:, -2]
    v[:, :, 0], v[:, :, -1] = v[:, :, 1], v[:, :, -2]
    return v


def _from(v, l):
    """v(x - c_l), periodic."""
    return torch.roll(v, (CZ[l], CY[l], CX[l]), (0, 1, 2))


def _diff(v, axis):
    """Sum over links of 3 w_l c_l,axis v(x + c_l), by one derivative and the two smoothings across it."""
    a, b = [d for d in (0, 1, 2) if d != axis]
    dv = torch.roll(v, -1, axis) - torch.roll(v, 1, axis)
    side = torch.roll(dv, 1, a) + torch.roll(dv, -1, a) + torch.roll(dv, 1, b) + torch.roll(dv, -1, b)
    return dv / 6.0 + side / 12.0


def _normals(phi, keep):
    gx, gy, gz = _diff(phi, 2), _diff(phi, 1), _diff(phi, 0)
    sq = gx * gx + gy * gy + gz * gz
    k = 1.0 / torch.sqrt(torch.clamp(sq, min=1e-9))
    ind = sq * k
    return [v if keep is None else v * keep for v in (gx * k, gy * k, gz * k, ind)]


def _force(n, ind, sigma, keep):
    curv = -(_diff(n[0], 2) + _diff(n[1], 1) + _diff(n[2], 0))
    return [v if keep is None else v * keep for v in (sigma * curv * n[0] * ind, sigma * curv * n[1] * ind,
                                                      sigma * curv * n[2] * ind)]


def _dot(l, v):
    s = 0.0
    for c, a in ((CX[l], v[0]), (CY[l], v[1]), (CZ[l], v[2])):
        if c:
            s = s + a if c > 0 else s - a
    return s


def _moments(pull, F):
    """rho, u and the non-equilibrium stress from the 19 incoming populations pull(l)."""
    shape = F[0].shape
    z = lambda: torch.zeros(shape, dtype=torch.float64, device=F[0].device)  # noqa: E731
    rho, j, t = z(), [z(), z(), z()], {k: z() for k in ("xx", "yy", "zz", "xy", "xz", "yz")}
    for l in range(19):
        v = pull(l)
        rho += v
        _add_moments(l, v, j, t)
    u = [(a + 0.5 * b) / rho for a, b in zip(j, F)]
    base, uf = 1.5 * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2), u[0] * F[0] + u[1] * F[1] + u[2] * F[2]
    for l in range(19):
        a = 3.0 * _dot(l, u) if l else 0.0
        eq = W[l] * rho * (1.0 + a + 0.5 * a * a - base)
        he = 1.5 * eq * ((_dot(l, F) if l else 0.0) - uf) / rho
        _add_moments(l, he - eq, None, t)
    return rho, u, t


def _add_moments(l, v, j, t):
    c = (CX[l], CY[l], CZ[l])
    for k, a in enumerate("xyz"):
        if c[k]:
            if j is not None:
                j[k] += c[k] * v
            t[a + a] += v
    for i, k in ((0, 1), (0, 2), (1, 2)):
        if c[i] * c[k]:
            t["xyz"[i] + "xyz"[k]] += c[i] * c[k] * v


def _collide(l, rho, u, F, t, omega, base, uf):
    a = 3.0 * _dot(l, u) if l else 0.0
    eq = W[l] * rho * (1.0 + a + 0.5 * a * a - base)
    he = 1.5 * eq * ((_dot(l, F) if l else 0.0) - uf) / rho
    c = (CX[l], CY[l], CZ[l])
    q = (c[0] ** 2 - 1 / 3) * t["xx"] + (c[1] ** 2 - 1 / 3) * t["yy"] + (c[2] ** 2 - 1 / 3) * t["zz"]
    for i, k in ((0, 1), (0, 2), (1, 2)):
        if c[i] * c[k]:
            q = q + 2.0 * c[i] * c[k] * t["xyz"[i] + "xyz"[k]]
    return eq + (1.0 - omega) * 4.5 * W[l] * q + he


def _collide_phase(l, phi, u, n):
    s = SHARP * phi * (1.0 - phi)
    if l == 0:
        return W[0] * phi
    return W[l] * (phi * (1.0 + 3.0 * _dot(l, u)) + s * _dot(l, n))


def _simulate(nx, ny, nz, bubbles, walls, tau_f, tau_g, sigma, steps, macros):
    """phi as a program reads it after the steps; with macros the observables of the state instead."""
    dev = DEVICE
    phi = _phi0(nx, ny, nz, bubbles, walls, dev)
    keep = _interior(phi.shape, dev) if walls else None
    face = 1.0 - keep if walls else None
    omega, omega_g = 1.0 / _f32(tau_f), 1.0 / _f32(tau_g)
    sigma = _f32(sigma)
    f = torch.empty((19,) + tuple(phi.shape), dtype=torch.float64, device=dev)   # outgoing populations
    g = torch.empty_like(f)
    for l in range(19):
        f[l] = W[l]
        g[l] = W[l] * torch.roll(phi, (-CZ[l], -CY[l], -CX[l]), (0, 1, 2))
    for it in range(steps + 1):
        new = torch.zeros_like(phi)
        for l in range(19):
            new += _from(g[l], l)
        phi = new if keep is None else new * keep + phi * face
        if it == steps and not macros:
            break
        nx_, ny_, nz_, ind = _normals(phi, keep)
        n = (nx_, ny_, nz_)
        F = _force(n, ind, sigma, keep)
        rho, u, t = _moments(lambda l: _from(f[l], l), F)
        if it == steps:
            if walls:
                rho, u = rho * keep + face, [v * keep for v in u]
            return {"phi": phi, "rho": rho, "ux": u[0], "uy": u[1], "uz": u[2]}
        base, uf = 1.5 * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2), u[0] * F[0] + u[1] * F[1] + u[2] * F[2]
        for l in range(19):
            v = _collide(l, rho, u, F, t, omega, base, uf)
            f[l] = v if keep is None else v * keep + W[l] * face
        for l in range(19):
            v = _collide_phase(l, phi, u, n)
            if tau_g != 1.0:
                v = (1.0 - omega_g) * _from(g[l], l) + omega_g * v
            g[l] = v if keep is None else v * keep + W[l] * phi * face
        last = phi if keep is None else _clamped_faces(phi)
        phi = last
    # A step leaves the phi that it started from (phiCalc runs first), walls with their copied faces.
    return {"phi": last}


def exact(case, seed):
    kind = case["kind"]
    if kind == "lattice":
        out = _simulate(case["nx"], case["ny"], case["nz"], _lattice_bubbles(case, seed), case["bc"] == "reference",
                        case["tau_f"], case["tau_g"], case["sigma"], case["steps"], case["fields"] == "all")
        return {k: v.cpu().numpy() for k, v in out.items()}
    if kind == "batch":
        return [_simulate(c["side"], c["side"], c["side"], [c["bubble"]], False, c["tau_f"], 1.0, c["sigma"],
                          case["steps"], False)["phi"].cpu().numpy() for c in _batch_cases(case, seed)]
    if kind == "serve":
        # The loop reads a case out when its steps are done: phi of its final state.
        phi = [_simulate(c["side"], c["side"], c["side"], [c["bubble"]], False, c["tau_f"], 1.0, c["sigma"],
                         c["steps"], True)["phi"].cpu().numpy() for c in _serve_cases(case, seed)]
        return {"phi": phi, "status": None}
    phi, rho, ux, uy, uz = _flow(case, seed, torch.float64, DEVICE)
    if kind == "reduce":
        return torch.stack([phi.sum(), (0.5 * rho * (ux * ux + uy * uy + uz * uz)).sum()])
    return _exact_ops(case, phi, rho, ux, uy, uz)


def _exact_ops(case, phi, rho, ux, uy, uz):
    """One iteration on the buffers prepare() makes."""
    walls = case["bc"] == "reference"
    f, g = (v.double() for v in _equilibrium(*(v.float() for v in (phi, rho, ux, uy, uz))))
    keep = _interior(phi.shape, phi.device) if walls else torch.ones_like(phi)
    face = 1.0 - keep
    phi = g.sum(0) * keep + phi * face
    nx_, ny_, nz_, ind = _normals(phi, keep)
    n = (nx_, ny_, nz_)
    F = _force(n, ind, _f32(0.1), keep)
    r, u, t = _moments(lambda l: f[l], F)
    rho = r * keep + rho * face
    u = [a * keep + b * face for a, b in zip(u, (ux, uy, uz))]
    base, uf = 1.5 * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2), u[0] * F[0] + u[1] * F[1] + u[2] * F[2]
    f_new, g_new = torch.empty_like(f), torch.empty_like(g)
    inside = torch.zeros_like(phi)
    for l in range(19):
        # Destinations whose source x - c_l lies in the box: pushed by an interior cell, set by a face. A destination
        # without one keeps its f, and its g comes across the periodic wrap.
        inside.fill_(1.0)
        if walls:
            for axis, c in enumerate((CZ[l], CY[l], CX[l])):
                if c:
                    inside.select(axis, 0 if c > 0 else -1).zero_()
        post = _collide(l, rho, u, F, t, 1.0 / _f32(0.505), base, uf)
        f_new[l] = _from(post * keep + W[l] * rho * face, l) * inside + f[l] * (1.0 - inside)
        gp = _collide_phase(l, phi, u, n) * keep + g[l] * face
        g_new[l] = _from(gp * keep + W[l] * phi * face, l) * inside + _from(gp, l) * (1.0 - inside)
    if walls:
        phi = _clamped_faces(phi)
    return {"f": f_new, "g": g_new, "phi": phi, "rho": rho, "ux": u[0], "uy": u[1], "uz": u[2]}
