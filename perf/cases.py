"""What is timed: the stencil path as a user's program calls it.

The cases are calls of the public Python API (``npbench_amd.stencils`` and
``npbench_amd.batch``) on operands that already live on the GPU, as the
framework's copy function leaves them: the four structured-grid kernels and
the batched form of the sweeps, which carry the framework, and three of the
suite's other solvers, one of each kind of dependence (a time-stepping loop
around a pressure-Poisson iteration, a Gauss-Seidel sweep, an implicit line
solve).  Sizes are the suite's own presets, the measured configurations of
bench.py, and sizes of the same ranges that no vector width divides.

``work`` counts what a call cannot do without: every input read once, every
output written once, and the arithmetic of the update expressions.
"""

import math

import numpy as np
import torch

from npbench_amd import batch
from npbench_amd import device as dev
from npbench_amd import stencils as st
from npbench_amd import tune

DTYPE = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16}
SIZE = {"f64": 8, "f32": 4, "bf16": 2}


def listed():
    return [
        # the smallest call of the suite's sweeps (preset S): launches and
        # latency, the drop-in signature with FP64 device arrays
        {"name": "jacobi_2d_S_f64", "kind": "jacobi_2d", "n": 150, "steps": 49, "dtype": "f64"},
        # the measured 2-D configuration: 1000 x 1000, 100 ping-pong steps
        {"name": "jacobi_2d_1000_f64", "kind": "jacobi_2d", "n": 1000, "steps": 100,
         "dtype": "f64"},
        # one 3-D grid between the L and paper presets, side not a multiple
        # of any vector
        {"name": "heat_3d_101_f64", "kind": "heat_3d", "n": 101, "steps": 100, "dtype": "f64"},
        # the batched headline: eight 256^3 FP32 grids, 100 ping-pong steps
        {"name": "heat_3d_batch_256_f32", "kind": "plan", "mix": "heat", "count": 8, "n": 256,
         "steps": 100, "dtype": "f32", "tblock": 3},
        # a batch of uneven 2-D and 3-D grids with their own step counts, as
        # the serving mix draws them
        {"name": "uneven_batch_f32", "kind": "plan", "mix": "uneven", "count": 12, "n": 1024,
         "steps": 60, "dtype": "f32", "tblock": 2},
        # horizontal diffusion at the paper preset, the FP64 drop-in
        {"name": "hdiff_paper_f64", "kind": "hdiff", "I": 256, "J": 256, "K": 160,
         "dtype": "f64"},
        # a ragged FP32 domain: an odd level count, rows of odd length
        {"name": "hdiff_ragged_f32", "kind": "hdiff", "I": 190, "J": 203, "K": 137,
         "dtype": "f32"},
        # vertical advection at the measured configuration, FP32 fields with
        # FP64 elimination
        {"name": "vadv_256_f32", "kind": "vadv", "I": 256, "J": 256, "K": 160, "dtype": "f32"},
        # vertical advection at preset M, the FP64 drop-in
        {"name": "vadv_M_f64", "kind": "vadv", "I": 112, "J": 112, "K": 80, "dtype": "f64"},
        # lid-driven cavity at preset L: 100 time steps of 20 pressure
        # iterations
        {"name": "cavity_flow_L", "kind": "cavity_flow", "nx": 201, "ny": 201, "nt": 100,
         "nit": 20},
        # Gauss-Seidel at the paper preset
        {"name": "seidel_2d_paper", "kind": "seidel_2d", "n": 400, "tsteps": 100},
        # the implicit alternating-direction solver at the paper preset
        {"name": "adi_paper", "kind": "adi", "n": 200, "tsteps": 100},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the presets' ranges of each kind, any size in them."""
    kind = rng.choice(["jacobi_2d", "jacobi_2d", "heat_3d", "plan", "hdiff", "hdiff", "vadv",
                       "vadv", "cavity_flow", "seidel_2d", "adi"])
    if kind == "jacobi_2d":
        return {"kind": kind, "n": _log_int(rng, 128, 2800), "steps": rng.randint(20, 100),
                "dtype": rng.choice(["f64", "f32", "bf16"])}
    if kind == "heat_3d":
        return {"kind": kind, "n": _log_int(rng, 25, 256), "steps": rng.randint(20, 100),
                "dtype": rng.choice(["f64", "f32", "bf16"])}
    if kind == "plan":
        mix = rng.choice(["heat", "uneven"])
        # tile plans want whole 16-byte vectors: sides in eights, as served
        n = 8 * rng.randint(8, 32) if mix == "heat" else 8 * rng.randint(32, 160)
        return {"kind": kind, "mix": mix, "count": rng.randint(2, 8), "n": n,
                "steps": rng.randint(10, 60), "dtype": "f32",
                "tblock": rng.choice([2, 3]) if mix == "heat" else 2}
    if kind == "hdiff":
        return {"kind": kind, "I": _log_int(rng, 60, 384), "J": _log_int(rng, 60, 384),
                "K": rng.randint(40, 160), "dtype": rng.choice(["f64", "f32", "bf16"])}
    if kind == "vadv":
        return {"kind": kind, "I": _log_int(rng, 60, 256), "J": _log_int(rng, 60, 256),
                "K": rng.choice([40, 60, 80, 120, 160, rng.randint(40, 160)]),
                "dtype": rng.choice(["f64", "f32"])}
    if kind == "cavity_flow":
        return {"kind": kind, "nx": rng.randint(61, 201), "ny": rng.randint(61, 201),
                "nt": rng.randint(25, 100), "nit": rng.randint(5, 20)}
    if kind == "seidel_2d":
        return {"kind": kind, "n": _log_int(rng, 50, 400), "tsteps": rng.randint(8, 100)}
    return {"kind": "adi", "n": _log_int(rng, 100, 300), "tsteps": rng.randint(20, 80)}


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _rand(seed, shapes, dtype=torch.float64):
    """Uniform [0, 1) fields, drawn in FP64 and stored in ``dtype``."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    return [torch.rand(s, generator=gen, dtype=torch.float64, device="cuda").to(dtype)
            for s in shapes]


def _plan_grids(case):
    """(kind, side, sweeps) of a batch's grids: equal ones, or 2-D and 3-D in
    turn with sides and step counts falling off from the largest."""
    if case["mix"] == "heat":
        return [("heat_3d", case["n"], 2 * case["steps"])] * case["count"]
    out = []
    for g in range(case["count"]):
        share = 1.0 - 0.8 * g / max(1, case["count"] - 1)
        steps = max(5, int(case["steps"] * (1.0 - 0.07 * g)))
        if g % 2 == 0:
            side = max(128, int(case["n"] * share) // 8 * 8)
            out.append(("jacobi_2d", side, 2 * steps))
        else:
            side = max(32, int(case["n"] / 8 * share) // 8 * 8)
            out.append(("heat_3d", side, 2 * steps))
    return out


def prepare(case, seed):
    dev.require_device()
    kind = case["kind"]
    state = {"case": case}
    if kind in ("jacobi_2d", "heat_3d"):
        shape = (case["n"],) * (2 if kind == "jacobi_2d" else 3)
        state["f"] = _rand(seed, [shape, shape], DTYPE[case["dtype"]])
        if kind == "heat_3d":  # the suite starts heat from B = A.copy()
            state["f"][1] = state["f"][0].clone()
    elif kind == "plan":
        grids = []
        for g, (k, n, sweeps) in enumerate(_plan_grids(case)):
            shape = (n,) * (2 if k == "jacobi_2d" else 3)
            a, b = _rand(1000 * seed + g, [shape, shape], DTYPE[case["dtype"]])
            if case["mix"] == "heat":  # B = A.copy(), the suite's start
                b = a.clone()
            grids.append(batch.Grid(k, a, b, sweeps))
        # bench.py's launch shapes: the autotuner's choice for equal grids,
        # the serving mix's own for uneven ones; and a captured graph
        if case["mix"] == "heat":
            shape = {"T": case["tblock"], "rows": 14 if case["tblock"] == 3 else 12, "seg": 64}
        else:
            shape = {"T": case["tblock"], "rows": 10, "seg": 32}
        tune.apply(shape)
        plan = batch.Plan(grids, tblock=shape["T"], seg=shape["seg"])
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        plan.capture(side)
        state["plan"], state["side"] = plan, side
    elif kind == "hdiff":
        I, J, K = case["I"], case["J"], case["K"]
        f = _rand(seed, [(I + 4, J + 4, K), (I, J, K), (I, J, K)])
        f[2] *= 0.25  # coeff uniform [0, 0.25)
        state["f"] = [t.to(DTYPE[case["dtype"]]) for t in f]
    elif kind == "vadv":
        I, J, K = case["I"], case["J"], case["K"]
        state["f"] = _rand(seed, [(I, J, K), (I, J, K), (I + 1, J, K), (I, J, K), (I, J, K)],
                           DTYPE[case["dtype"]])
    elif kind == "cavity_flow":
        # near rest, as the suite starts it
        shape = (case["ny"], case["nx"])
        u, v, p = _rand(seed, [shape] * 3)
        state["f"] = [0.01 * u, 0.01 * (v - 0.5), 0.01 * p]
        dx, dy = 2 / (case["nx"] - 1), 2 / (case["ny"] - 1)
        state["d"] = (.1 / ((case["nx"] - 1) * (case["ny"] - 1)), dx, dy)
    else:  # seidel_2d, adi
        state["f"] = _rand(seed, [(case["n"], case["n"])])
    return state


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "plan":
        state["plan"].launch()
        return [t for g in state["plan"].grids for t in (g.A, g.B)]
    f = state["f"]
    if kind in ("jacobi_2d", "heat_3d"):
        if case["dtype"] == "f64":  # the suite's signature
            dropin = st.jacobi_2d if kind == "jacobi_2d" else st.heat_3d
            dropin(case["steps"] + 1, f[0], f[1])
        else:
            sweeps = st.jacobi2d_sweeps if kind == "jacobi_2d" else st.heat3d_sweeps
            sweeps(f[0], f[1], 2 * case["steps"])
        return f
    if kind == "hdiff":
        st.hdiff(f[0], f[1], f[2])
        return f[1]
    if kind == "vadv":
        st.vadv(*f, 0.15)
        return f[0]
    if kind == "cavity_flow":
        dt, dx, dy = state["d"]
        st.cavity_flow_dropin(case["nx"], case["ny"], case["nt"], case["nit"], f[0], f[1], dt,
                              dx, dy, f[2], 1.0, 0.1)
        return f
    if kind == "seidel_2d":
        st.seidel_2d(case["tsteps"], case["n"], f[0])
        return f[0]
    return st.adi_dropin(case["tsteps"], case["n"], f[0])


def work(case):
    kind = case["kind"]
    if kind in ("jacobi_2d", "heat_3d", "plan"):
        grids = (_plan_grids(case) if kind == "plan" else
                 [(kind, case["n"], 2 * case["steps"])])
        s = SIZE[case["dtype"]]
        nbytes = flops = 0
        for k, n, sweeps in grids:
            d = 2 if k == "jacobi_2d" else 3
            nbytes += 3 * s * n ** d  # A read, A and B written
            flops += (5 if d == 2 else 8) * sweeps * (n - 2) ** d
        return {"bytes": nbytes, "flops": flops}
    if kind == "hdiff":
        I, J, K = case["I"], case["J"], case["K"]
        return {"bytes": SIZE[case["dtype"]] * K * ((I + 4) * (J + 4) + 2 * I * J),
                "flops": 18 * I * J * K}
    if kind == "vadv":
        I, J, K = case["I"], case["J"], case["K"]
        return {"bytes": SIZE[case["dtype"]] * K * J * (6 * I + 1), "flops": 33 * I * J * K}
    if kind == "cavity_flow":
        points = case["nx"] * case["ny"]
        return {"bytes": 48 * points, "flops": points * case["nt"] * (8 * case["nit"] + 60)}
    n = case["n"]
    if kind == "seidel_2d":
        return {"bytes": 16 * n * n, "flops": 9 * (case["tsteps"] - 1) * (n - 2) ** 2}
    return {"bytes": 16 * n * n, "flops": 20 * case["tsteps"] * (n - 2) ** 2}


# --------------------------------------------------------------------------
# the same results in 64 bits, by plain torch and numpy
# --------------------------------------------------------------------------
def _jacobi(src, dst):
    c = src[1:-1, 1:-1]
    s = c + src[1:-1, :-2]
    s += src[1:-1, 2:]
    s += src[2:, 1:-1]
    s += src[:-2, 1:-1]
    dst[1:-1, 1:-1] = s.mul_(0.2)


def _heat(src, dst):
    mid = slice(1, -1)
    c = src[mid, mid, mid]
    c2 = 2.0 * c
    t = ((src[2:, mid, mid] - c2) + src[:-2, mid, mid]) * 0.125
    t += ((src[mid, 2:, mid] - c2) + src[mid, :-2, mid]) * 0.125
    t += ((src[mid, mid, 2:] - c2) + src[mid, mid, :-2]) * 0.125
    dst[mid, mid, mid] = t + c


def _swept(kind, a, b, sweeps):
    a, b = a.double(), b.double()
    step = _jacobi if kind == "jacobi_2d" else _heat
    for s in range(sweeps):
        step(*((a, b) if s % 2 == 0 else (b, a)))
    return [a, b]


def _hdiff(f, coeff):
    I, J, _ = coeff.shape
    lap = 4.0 * f[1:I + 3, 1:J + 3] - (f[2:I + 4, 1:J + 3] + f[0:I + 2, 1:J + 3] +
                                       f[1:I + 3, 2:J + 4] + f[1:I + 3, 0:J + 2])
    r = lap[1:, 1:J + 1] - lap[:-1, 1:J + 1]
    flx = torch.where(r * (f[2:I + 3, 2:J + 2] - f[1:I + 2, 2:J + 2]) > 0, 0.0, r)
    r = lap[1:I + 1, 1:] - lap[1:I + 1, :-1]
    fly = torch.where(r * (f[2:I + 2, 2:J + 3] - f[2:I + 2, 1:J + 2]) > 0, 0.0, r)
    div = flx[1:] - flx[:-1] + fly[:, 1:] - fly[:, :-1]
    return f[2:I + 2, 2:J + 2] - coeff * div


def _vadv(ustage_t, u, wcon, u_pos, utens, dtr):
    K = u.shape[2]
    u, u_pos, rest = (x.permute(2, 0, 1).contiguous() for x in (u, u_pos, utens))
    ut = ustage_t.permute(2, 0, 1).contiguous()
    w = (wcon[1:] + wcon[:-1]).permute(2, 0, 1).contiguous()
    cc, dd = torch.zeros_like(u), torch.zeros_like(u)
    for k in range(K):
        a = -0.25 * w[k] * 0.5 if k else torch.zeros_like(w[0])
        c = 0.25 * w[k + 1] * 0.5 if k < K - 1 else torch.zeros_like(w[0])
        corr = torch.zeros_like(w[0])
        if k:
            corr = corr - a * (u[k - 1] - u[k])
        if k < K - 1:
            corr = corr - c * (u[k + 1] - u[k])
        d = dtr * u_pos[k] + rest[k] + ut[k] + corr
        b = dtr - a - c
        if k:
            b = b - cc[k - 1] * a
            d = d - dd[k - 1] * a
        inv = 1.0 / b
        cc[k], dd[k] = c * inv, d * inv
    x = dd[K - 1]
    out = torch.empty_like(dd)
    for k in range(K - 1, -1, -1):
        if k < K - 1:
            x = dd[k] - cc[k] * x
        out[k] = dtr * (x - u_pos[k])
    return out.permute(1, 2, 0).contiguous()


def _cavity(nt, nit, u, v, p, dt, dx, dy, rho, nu):
    m, lo, hi = slice(1, -1), slice(None, -2), slice(2, None)
    den = 2 * (dx ** 2 + dy ** 2)
    for _ in range(nt):
        un, vn = u.copy(), v.copy()
        ux = (u[m, hi] - u[m, lo]) / (2 * dx)
        vy = (v[hi, m] - v[lo, m]) / (2 * dy)
        cross = (u[hi, m] - u[lo, m]) / (2 * dy) * (v[m, hi] - v[m, lo]) / (2 * dx)
        b = rho * (1 / dt * (ux + vy) - ux ** 2 - 2 * cross - vy ** 2)
        for _ in range(nit):
            q = p.copy()
            p[m, m] = (((q[m, hi] + q[m, lo]) * dy ** 2 + (q[hi, m] + q[lo, m]) * dx ** 2) / den
                       - dx ** 2 * dy ** 2 / den * b)
            p[:, -1] = p[:, -2]
            p[0, :] = p[1, :]
            p[:, 0] = p[:, 1]
            p[-1, :] = 0
        uc, vc = un[m, m], vn[m, m]
        for x, xn, grad, d in ((u, un, p[m, hi] - p[m, lo], dx),
                               (v, vn, p[hi, m] - p[lo, m], dy)):
            c = xn[m, m]
            x[m, m] = (c - uc * dt / dx * (c - xn[m, lo]) - vc * dt / dy * (c - xn[lo, m])
                       - dt / (2 * rho * d) * grad
                       + nu * (dt / dx ** 2 * (xn[m, hi] - 2 * c + xn[m, lo])
                               + dt / dy ** 2 * (xn[hi, m] - 2 * c + xn[lo, m])))
        for x, lid in ((u, 1), (v, 0)):
            x[0, :] = x[:, 0] = x[:, -1] = 0
            x[-1, :] = lid
    return [u, v, p]


def _seidel(tsteps, a):
    """Points (t, i, j) of one 4 t + 2 i + j depend only on earlier ones and
    are updated together."""
    n = a.shape[0]
    sweeps = tsteps - 1
    flat = a.reshape(-1)
    t, i = (x.reshape(-1) for x in np.meshgrid(np.arange(sweeps), np.arange(1, n - 1),
                                               indexing="ij"))
    start = 4 * t + 2 * i
    order = np.argsort(start, kind="stable")
    start, i = start[order], i[order]
    for tau in range(int(start[0]) + 1, int(start[-1]) + n - 1):
        first = np.searchsorted(start, tau - (n - 2), "left")
        last = np.searchsorted(start, tau - 1, "right")
        x = i[first:last] * n + (tau - start[first:last])
        s = flat[x - n - 1] + flat[x - n]
        for d in (1 - n, 1, n - 1, n, n + 1):
            s = s + flat[x + d]
        flat[x] = ((flat[x] + s) + flat[x - 1]) / 9.0
    return a


def _adi(tsteps, u):
    n = u.shape[0]
    dt, h = 1.0 / tsteps, 1.0 / n
    mul1, mul2 = 2.0 * dt / (h * h), 1.0 * dt / (h * h)
    a, d, mid = -mul1 / 2.0, -mul2 / 2.0, 1.0 + mul2

    def lines(x, lo, side):
        """Solves along axis 0 of x for every interior column, whose
        neighbours enter the right-hand side with weight side."""
        p, q = np.zeros(n), np.ones((n, n - 2))
        for j in range(1, n - 1):
            den = lo * p[j - 1] + mid
            p[j] = -lo / den
            rhs = -side * x[j, :-2] + (1.0 + 2.0 * side) * x[j, 1:-1] - side * x[j, 2:]
            q[j] = (rhs - lo * q[j - 1]) / den
        out = np.ones((n, n - 2))
        for j in range(n - 2, 0, -1):
            out[j] = p[j] * out[j + 1] + q[j]
        return out

    v = np.empty_like(u)
    for _ in range(tsteps):
        v[:, 1:-1] = lines(u, a, d)
        u[1:-1, :] = lines(np.ascontiguousarray(v.T), d, a).T
    return u


def exact(case, seed):
    kind = case["kind"]
    state = prepare(case, seed)
    if kind == "plan":
        return [t for g in state["plan"].grids for t in _swept(g.kind, g.A, g.B, g.nsweeps)]
    f = state["f"]
    if kind in ("jacobi_2d", "heat_3d"):
        return _swept(kind, f[0], f[1], 2 * case["steps"])
    if kind == "hdiff":
        return _hdiff(f[0].double(), f[2].double())
    if kind == "vadv":
        return _vadv(*(t.double() for t in f), 0.15)
    host = [t.cpu().numpy() for t in f]
    if kind == "cavity_flow":
        dt, dx, dy = state["d"]
        return _cavity(case["nt"], case["nit"], *host, dt, dx, dy, 1.0, 0.1)
    if kind == "seidel_2d":
        return _seidel(case["tsteps"], host[0])
    return _adi(case["tsteps"], host[0])
