"""Workloads of the pressure-projection library, as a program calls it.

A case is a dict of plain values; `prepare` builds what a program holds before
the call (device fields made from the seed, the Poisson plan, the recorded
graph), `run` makes one pass through the entry points of `flutas_amd.api` and
returns its outputs as torch views of the device fields.

kinds
  solve     out-of-place FP64 Poisson solve on one plan
  refined   the same through the FP32 transforms with FP64 refinement (1e-10)
  f32       in-place solve of a single-precision field (the FP32 builds)
  step      one two-phase projection step with constant-coefficient pressure
            splitting, call by call in the reference's order
  graph     the same step through the fused entry points, recorded once and
            replayed
  batch     many independent uneven solves in one call
  lines     the stand-alone r2r transforms along x and y of a field
"""
import ctypes
import math

import numpy as np
import torch

from flutas_amd import api

DT, RHO_HEAVY = 1e-3, 1000.0
TWO_PI = 2 * math.pi


def _grid(kind, nx, ny, nz, bc, lx=1.0, ly=1.0, lz=1.0, alpha=0.0):
    return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "bc": bc, "lx": lx, "ly": ly, "lz": lz,
            "alpha": alpha}


def listed():
    def c(name, *a, **k):
        return dict(_grid(*a, **k), name=name)

    return [
        # the quasi-2-D lid-driven cavity (two periodic cells across): a step
        # of such a run is all latency
        c("solve_2x64x64", "solve", 2, 64, 64, "PPNNNN"),
        # an ordinary small box: the uniform 128^3 channel
        c("solve_128", "solve", 128, 128, 128, "PPPPNN"),
        # a channel at mesh sizes that are no powers of two
        c("solve_360x300x240", "solve", 360, 300, 240, "PPPPNN", TWO_PI, math.pi, 1.0, 1.5),
        # a closed box at ragged sizes, with factors 7 and 11
        c("solve_210x154x90", "solve", 210, 154, 90, "DDNNNN", 1.0, 0.7, 0.5, 1.2),
        # the stretched channel at production size
        c("solve_512", "solve", 512, 512, 512, "PPPPNN", TWO_PI, math.pi, 1.0, 1.5),
        # the largest: the cavity with Neumann walls all round
        c("solve_1024x1024x512", "solve", 1024, 1024, 512, "NNNNNN"),
        # the mixed-precision option on the production channel
        c("refined_512", "refined", 512, 512, 512, "PPPPNN", TWO_PI, math.pi, 1.0, 1.5),
        # a single-precision run
        c("f32_256", "f32", 256, 256, 256, "PPPPNN", TWO_PI, math.pi, 1.0, 1.5),
        # the two-phase step of a triply periodic box (one heavy sphere)
        c("step_256x256x512", "step", 256, 256, 512, "PPPPPP", 1.0, 1.0, 2.0),
        # the same between walls on a small box, as a replayed graph
        c("graph_128", "graph", 128, 128, 128, "PPPPNN", 1.0, 1.0, 1.0),
        # an ensemble of 64 uneven problems with mixed walls
        {"name": "batch_64", "kind": "batch", "count": 64, "pick": 5, "precision": 64},
        # the transforms of fft.f90 on their own, x then y
        {"name": "lines_256x192x128", "kind": "lines", "nx": 256, "ny": 192, "nz": 128, "bc": "PPNN"},
    ]


def _largest_prime(n):
    q = 2
    while q * q <= n:
        if n % q:
            q += 1
        else:
            n //= q
    return n


# Mesh sizes spread over the logarithm: the transformed directions take
# products of 2, 3 and 5 mostly and factors up to 13 now and then, z any even
# number.
def _size(rng, lo, hi, most):
    n = 2 * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / 2)
    while _largest_prime(n) > most:
        n += 2
    return n


_XY = ("PPPP", "PPPP", "NNNN", "PPNN", "DDPP", "NNDD", "NDPP", "PPDN")
_Z = ("NN", "NN", "DD", "ND", "PP")


def draw(rng):
    kind = rng.choice(("solve", "solve", "solve", "solve", "refined", "f32", "step", "graph",
                       "batch", "lines"))
    if kind == "batch":
        return {"kind": "batch", "count": rng.randint(3, 64), "pick": rng.randint(10, 10 ** 6),
                "precision": rng.choice((64, 32))}
    cap = {"solve": 2 ** 27, "refined": 2 ** 26, "f32": 2 ** 27, "step": 2 ** 25, "graph": 2 ** 23,
           "lines": 2 ** 24}[kind]
    lo = 32 if kind in ("refined", "step", "graph") else 16
    while True:
        nx, ny, nz = (_size(rng, lo, 640, m) for m in (rng.choice((5, 5, 5, 13)),
                                                       rng.choice((5, 5, 5, 13)), 10 ** 6))
        if cap / 2 ** 13 <= nx * ny * nz <= cap and nz >= 16:
            break
    if kind == "lines":
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz,
                "bc": rng.choice(("PPPP", "PPNN", "NNNN", "DDNN", "NDDD"))}
    if kind in ("step", "graph"):
        bc = "PPPP" + rng.choice(("PP", "NN"))
    else:
        bc = rng.choice(_XY) + rng.choice(_Z)
    # cells of like width; the stretched grids cluster at both walls
    alpha = 0.0 if bc[4] == "P" else rng.choice((0.0, round(rng.uniform(1.0, 2.0), 3)))
    lx = 1.0
    if kind == "f32":
        # in place, pass after pass: a box in which no mode grows (the lowest
        # eigenvalue stays a little over one)
        low = [(math.pi / (1.0, ny / nx, nz / nx)[d] * {"P": 2, "NN": 1, "DD": 1}.get(
            "P" if bc[2 * d] == "P" else bc[2 * d:2 * d + 2], 0.5)) ** 2 for d in range(3)]
        fixed = [low[d] for d in range(3) if "D" in bc[2 * d:2 * d + 2]]
        lx = 0.9 * math.sqrt(sum(fixed) if fixed else min(low))
    return _grid(kind, nx, ny, nz, bc, lx, lx * ny / nx, lx * nz / nx, alpha)


# ---- inputs -----------------------------------------------------------------

class _Memory:
    """A DeviceArray as torch sees it: (nz, ny, nx), x fastest."""

    def __init__(self, arr):
        self.arr = arr
        self.__cuda_array_interface__ = {
            "shape": arr.shape[::-1], "typestr": arr.dtype.str, "data": (arr.ptr, False),
            "strides": None, "version": 2}


def _field(shape, dtype=np.float64):
    arr = api.DeviceArray(shape, dtype)
    t = torch.as_tensor(_Memory(arr), device="cuda")
    t.zero_()
    return arr, t


def _inner(t):
    return t[1:-1, 1:-1, 1:-1]


def _upload(a):
    return api.DeviceArray.from_host(np.ascontiguousarray(a, np.float64))


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(case, g):
    return torch.randn((case["nz"], case["ny"], case["nx"]), dtype=torch.float64, device="cuda",
                       generator=g)


def _metrics(case):
    """dzc, dzf over (0 : nz+1): both ends clustered by a tanh law."""
    n, al, lz = case["nz"], case["alpha"], case["lz"]
    z0 = np.arange(n + 1) / n
    zf = lz * (0.5 * (1.0 + np.tanh((z0 - 0.5) * al) / np.tanh(al / 2)) if al else z0)
    dzf = np.zeros(n + 2)
    dzf[1:-1] = np.diff(zf)
    dzf[0], dzf[-1] = dzf[1], dzf[-2]
    dzc = np.zeros(n + 2)
    dzc[:-1] = 0.5 * (dzf[:-1] + dzf[1:])
    dzc[-1] = dzc[-2]
    return dzc, dzf


def _dli(case):
    return case["nx"] / case["lx"], case["ny"] / case["ly"], case["nz"] / case["lz"]


def _rhs(case, seed):
    """N(0,1); solvable (weighted mean removed) when no side is Dirichlet."""
    f = _normal(case, _generator(seed))
    if "D" not in case["bc"]:
        w = torch.from_numpy(_metrics(case)[1][1:-1]).cuda()
        f -= (f.mean(dim=(1, 2)) * w).sum() / w.sum()
    return f


def _batch(case):
    """The problems of an uneven batch, drawn from `pick`."""
    g = np.random.Generator(np.random.Philox(case["pick"]))
    out = []
    for q in range(case["count"]):
        nx, ny = (int(g.choice([64, 96, 128, 192, 256])) for _ in range(2))
        nz = int(g.choice([64, 128, 256]))
        bc = ["PPPPNN", "NNNNNN", "PPPPDD"][int(g.integers(0, 3))]
        out.append(_grid("solve", nx, ny, nz, bc, alpha=float(g.uniform(1, 2)) if q % 2 else 0.0))
    return out


def _step_inputs(case, seed):
    """Interior u, v, w ~ U[-0.1, 0.1], p, pold ~ N(0,1) and the density of a
    heavy sphere in the middle, smoothed over 1.5 cells."""
    g = _generator(seed)
    shape = (case["nz"], case["ny"], case["nx"])
    u, v, w = (0.2 * torch.rand(shape, dtype=torch.float64, device="cuda", generator=g) - 0.1
               for _ in range(3))
    if case["bc"][4] == "N":
        w[-1] = 0.0
    p, pold = _normal(case, g), _normal(case, g)
    r2 = 0.0
    for d, (n, l) in enumerate(((case["nz"], case["lz"]), (case["ny"], case["ly"]),
                                (case["nx"], case["lx"]))):
        x = (torch.arange(n, dtype=torch.float64, device="cuda") + 0.5) * (l / n) - l / 2
        r2 = r2 + x.pow(2).reshape([-1 if q == d else 1 for q in range(3)])
    psi = 0.5 * (1 - torch.tanh((r2.sqrt() - 0.25 * case["lx"]) / (1.5 * case["lx"] / case["nx"])))
    return u, v, w, p, pold, psi * RHO_HEAVY + (1 - psi)


def _plan(case, precision=api.FP64):
    dzc, dzf = _metrics(case)
    return api.PoissonPlan((case["nx"], case["ny"], case["nz"]), _dli(case), 1 / dzc, 1 / dzf,
                           case["bc"], precision=precision, tol=1e-10)


def _prepare_step(case, seed):
    nx, ny, nz = n = case["nx"], case["ny"], case["nz"]
    dzc, dzf = _metrics(case)
    bc, zero = case["bc"], (0.0,) * 6
    dli = _dli(case)
    dl = tuple(1 / d for d in dli)
    s = {"case": case, "n": n, "dli": dli, "dl": dl, "dzc": dzc, "dzf": dzf, "bc": bc,
         "dzci_d": _upload(1 / dzc), "dzfi_d": _upload(1 / dzf), "plan": _plan(case),
         "bcu": bc.replace("N", "D") * 3, "zero": zero, "turn": 0}
    for name, x in zip(("u", "v", "w", "p", "pold", "rho"), _step_inputs(case, seed)):
        s[name], t = _field(tuple(v + 2 for v in n))
        s[name + "_t"] = t
        _inner(t).copy_(x)
    for name in ("p", "pold", "rho"):
        api.boundp(bc, n, zero, dl, dzc[0], dzc[nz], s[name])
    _bounduvw(s)
    return s


def _bounduvw(s):
    api.bounduvw(s["bcu"], s["n"], (0.0,) * 18, 1, 1, [0] * 6, s["dl"], s["dzc"], s["dzf"],
                 s["u"], s["v"], s["w"])


def _source(s, p, pold):
    nx, ny, nz = s["n"]
    api.pres_tw_src(nx, ny, nz, *s["dli"], 1, 1, s["dzci_d"], 1.0, DT, DT, p, pold, s["rho"],
                    s["u"], s["v"], s["w"])
    _bounduvw(s)


def _step_calls(s):
    """The reference's call order."""
    nx, ny, nz = n = s["n"]
    u, v, w, p, pold, bc = s["u"], s["v"], s["w"], s["p"], s["pold"], s["bc"]
    ends = s["dzc"][0], s["dzc"][nz]
    _source(s, p, pold)
    api.copy_interior(nx, ny, nz, p, pold)
    api.boundp(bc, n, s["zero"], s["dl"], *ends, pold)
    api.fillps(nx, ny, nz, 1, 1, *s["dli"], s["dzfi_d"], 1 / DT, 1.0, u, v, w, p)
    api.updt_rhs_b(nx, ny, nz, "ccc", bc, *s["plan"].rhsb_device(), p)
    s["plan"].solve(p)
    api.boundp(bc, n, s["zero"], s["dl"], *ends, p)
    api.correc(nx, ny, nz, 1, 1, *s["dli"], s["dzci_d"], DT, 1.0, p, u, v, w)
    _bounduvw(s)
    api.add_interior(nx, ny, nz, pold, p)
    api.boundp(bc, n, s["zero"], s["dl"], *ends, p)


def _fused_calls(s, p, pold):
    """The fused order; the new pressure goes to pold's buffer."""
    nx, ny, nz = n = s["n"]
    u, v, w, phi, bc = s["u"], s["v"], s["w"], s["phi"], s["bc"]
    _source(s, p, pold)
    api.fillps_rhs(nx, ny, nz, 1, 1, *s["dli"], s["dzfi_d"], 1 / DT, 1.0, u, v, w, "ccc", bc,
                   *s["plan"].rhsb_device(), phi)
    s["plan"].solve_async(phi)
    api.correc_update_bc(nx, ny, nz, 1, 1, *s["dli"], s["dzci_d"], DT, 1.0, phi, p, pold, u, v, w,
                         bc, s["zero"], s["dl"], s["dzc"][0], s["dzc"][nz])
    _bounduvw(s)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("step", "graph"):
        s = _prepare_step(case, seed)
        if kind == "graph":
            s["phi"], s["phi_t"] = _field(tuple(v + 2 for v in s["n"]))
            s["graphs"] = []
            for p, pold in ((s["p"], s["pold"]), (s["pold"], s["p"])):
                with api.Graph() as graph:
                    _fused_calls(s, p, pold)
                s["graphs"].append(graph)
        return s
    if kind == "batch":
        s = {"case": case, "f": [], "p": [], "p_t": []}
        problems = []
        for q, c in enumerate(_batch(case)):
            dzc, dzf = _metrics(c)
            shape = (c["nx"] + 2, c["ny"] + 2, c["nz"] + 2)
            f, ft = _field(shape)
            _inner(ft).copy_(_rhs(c, seed * 1000 + q))
            p, pt = _field(shape)
            s["f"].append(f)
            s["p"].append(p)
            s["p_t"].append(pt)
            problems.append(((c["nx"], c["ny"], c["nz"]), _dli(c), 1 / dzc, 1 / dzf, c["bc"]))
        s["plan"] = api.BatchPlan(problems, precision=case["precision"], tol=1e-10)
        s["plan"].set_fields(s["f"], s["p"])
        return s
    if kind == "lines":
        s = {"case": case}
        s["f"], s["f_t"] = _field((case["nx"], case["ny"], case["nz"]))
        s["f_t"].copy_(_normal(case, _generator(seed)))
        return s
    shape = (case["nx"] + 2, case["ny"] + 2, case["nz"] + 2)
    if kind == "f32":
        s = {"case": case, "plan": _plan(case)}
        s["p"], s["p_t"] = _field(shape, np.float32)
        _inner(s["p_t"]).copy_(_rhs(case, seed))
        return s
    s = {"case": case, "plan": _plan(case, api.FP64 if kind == "solve" else api.FP32_REFINE)}
    s["f"], s["f_t"] = _field(shape)
    _inner(s["f_t"]).copy_(_rhs(case, seed))
    s["p"], s["p_t"] = _field(shape)
    return s


# ---- one pass -----------------------------------------------------------------

_FORWARD = {"PP": "R2HC", "NN": "REDFT10", "DD": "RODFT10", "ND": "REDFT11", "DN": "RODFT11"}


def _unit(case):
    """What keeps the spectrum of the unnormalised transforms at unit size."""
    return 1.0 / math.sqrt(math.prod(n * (1 if b == "PP" else 2) for n, b in (
        (case["nx"], case["bc"][:2]), (case["ny"], case["bc"][2:4]))))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("solve", "refined"):
        state["plan"].solve_into(state["f"], state["p"])
        return _inner(state["p_t"])
    if kind == "f32":
        plan, p = state["plan"], state["p"]
        rc = api.lib.flutas_psolve_solve_f32(ctypes.c_void_p(plan._h), ctypes.c_void_p(p.ptr))
        if rc:
            raise api.FlutasError(rc, api.lib.flutas_last_error().decode())
        return _inner(state["p_t"])
    if kind == "batch":
        state["plan"].solve()
        return [_inner(t) for t in state["p_t"]]
    if kind == "lines":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        api.fft_guru(_FORWARD[case["bc"][:2]], state["f"], nx, 1, ny, nx, nz, nx * ny)
        api.fft_guru(_FORWARD[case["bc"][2:4]], state["f"], ny, nx, nx, 1, nz, nx * ny)
        return state["f_t"].mul_(_unit(case))
    if kind == "step":
        _step_calls(state)
    else:
        state["graphs"][state["turn"]].launch()
        state["turn"] ^= 1
    new, old = ("pold_t", "p_t") if state["turn"] else ("p_t", "pold_t")
    return {"u": _inner(state["u_t"]), "v": _inner(state["v_t"]), "w": _inner(state["w_t"]),
            "p": _inner(state[new]), "pold": _inner(state[old])}


# ---- what a pass cannot do without ----------------------------------------------

def _solve_work(c, width=8):
    n = c["nx"] * c["ny"] * c["nz"]
    return {"bytes": 2 * width * n,
            "flops": n * (2 * 2.5 * (math.log2(c["nx"]) + math.log2(c["ny"])) + 10)}


def work(case):
    kind = case["kind"]
    if kind == "batch":
        each = [_solve_work(c) for c in _batch(case)]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    if kind == "lines":
        n = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": 16 * n, "flops": 2.5 * n * math.log2(case["nx"] * case["ny"])}
    w = _solve_work(case, 4 if kind == "f32" else 8)
    if kind in ("step", "graph"):
        # u, v, w, p, pold, rho in; u, v, w, p, pold out; source, divergence, correction
        n = case["nx"] * case["ny"] * case["nz"]
        w = {"bytes": 88 * n, "flops": w["flops"] + 60 * n}
    return w


# ---- the same in 64 bits, from the mathematics ------------------------------------

def _basis(n, b, dli):
    """Eigenvectors (columns, orthonormal) and eigenvalues of the second
    difference on n cells between the boundary pair b."""
    j = torch.arange(n, dtype=torch.float64, device="cuda")[:, None]
    k = torch.arange(n, dtype=torch.float64, device="cuda")[None, :]
    if b == "PP":
        m = torch.where(2 * k > n, n - k, k)
        ang = 2 * math.pi * ((j * m) % n) / n
        vec = torch.where(2 * k > n, torch.sin(ang), torch.cos(ang))
        arg = math.pi * m[0] / n
    elif b == "NN":
        vec, arg = torch.cos(math.pi * (j + 0.5) * k / n), math.pi * k[0] / (2 * n)
    elif b == "DD":
        vec, arg = torch.sin(math.pi * (j + 0.5) * (k + 1) / n), math.pi * (k[0] + 1) / (2 * n)
    else:
        fn = torch.cos if b == "ND" else torch.sin
        vec, arg = fn(math.pi * (j + 0.5) * (k + 0.5) / n), math.pi * (2 * k[0] + 1) / (4 * n)
    return vec / vec.pow(2).sum(0).sqrt(), -4 * torch.sin(arg).pow(2) * dli * dli


def _poisson(case, f):
    """Solution of the seven-point Poisson problem, f and the result as
    (nz, ny, nx); the free constant is fixed by a zero mean in the last plane."""
    bc, n = case["bc"], case["nz"]
    dli = _dli(case)
    vx, lx = _basis(case["nx"], bc[:2], dli[0])
    vy, ly = _basis(case["ny"], bc[2:4], dli[1])
    h = torch.matmul(vy.t().contiguous(), torch.matmul(f, vx))
    lam = ly[:, None] + lx[None, :]
    free = "D" not in bc
    if free:
        lam[0, 0] = 0.0
    if bc[4:] == "PP":
        vz, lz = _basis(n, "PP", dli[2])
        h = torch.matmul(vz.t().contiguous(), h.reshape(n, -1)).reshape(h.shape)
        d = lz[:, None, None] + lam
        d[0, 0, 0] = 1.0
        h /= d
        h[0, 0, 0] = 0.0
        h = torch.matmul(vz, h.reshape(n, -1)).reshape(h.shape)
    else:
        dzc, dzf = _metrics(case)
        a, c = 1 / (dzf[1:-1] * dzc[:-2]), 1 / (dzf[1:-1] * dzc[1:-1])
        b = -(a + c)
        b[0] += a[0] if bc[4] == "N" else -a[0]
        b[-1] += c[-1] if bc[5] == "N" else -c[-1]
        d = torch.empty_like(h)
        for k in range(n):
            piv = float(b[k]) + lam - (float(a[k]) * d[k - 1] if k else 0.0)
            if free and k == n - 1 and bc[4:] == "NN":
                piv[0, 0] = math.inf
            d[k] = float(c[k]) / piv
            h[k] = (h[k] - (float(a[k]) * h[k - 1] if k else 0.0)) / piv
        for k in range(n - 2, -1, -1):
            h[k] -= d[k] * h[k + 1]
        del d
    h = torch.matmul(torch.matmul(vy, h), vx.t().contiguous())
    if free:
        h -= h[-1].mean()
    return h


def _up(t, dim, wall=None):
    """The upper neighbour; beyond a wall `wall` of the last plane, else periodic."""
    r = torch.roll(t, -1, dim)
    if wall is not None:
        r[-1] = wall * t[-1]
    return r


def _exact_step(case, seed):
    u, v, w, p, pold, rho = _step_inputs(case, seed)
    dxi, dyi, _ = _dli(case)
    dzc, dzf = _metrics(case)
    dzci = torch.from_numpy(1 / dzc[1:-1]).cuda()[:, None, None]
    dzfi = torch.from_numpy(1 / dzf[1:-1]).cuda()[:, None, None]
    wall = None if case["bc"][4] == "P" else 1.0

    def close(w):
        if wall:
            w[-1] = 0.0

    hat = 2 * p - pold
    for vel, dim, di, wl in ((u, 2, dxi, None), (v, 1, dyi, None), (w, 0, dzci, wall)):
        inv = 2 / (_up(rho, dim, wl) + rho)
        vel -= DT * ((_up(p, dim, wl) - p) + (inv - 1) * (_up(hat, dim, wl) - hat)) * di
    close(w)
    below = torch.roll(w, 1, 0)
    f = ((w - below) * dzfi + (v - torch.roll(v, 1, 1)) * dyi + (u - torch.roll(u, 1, 2)) * dxi) / DT
    phi = _poisson(case, f)
    for vel, dim, di, wl in ((u, 2, dxi, None), (v, 1, dyi, None), (w, 0, dzci, wall)):
        vel -= DT * (_up(phi, dim, wl) - phi) * di
    close(w)
    return {"u": u, "v": v, "w": w, "p": p + phi, "pold": p}


def _r2r(b, n):
    """The forward transform of a boundary pair as a matrix (n outputs, n inputs)."""
    j = torch.arange(n, dtype=torch.float64, device="cuda")[None, :]
    k = torch.arange(n, dtype=torch.float64, device="cuda")[:, None]
    if b == "PP":
        m = torch.where(2 * k > n, n - k, k)
        ang = 2 * math.pi * ((j * m) % n) / n
        return torch.where(2 * k > n, -torch.sin(ang), torch.cos(ang))
    if b == "NN":
        return 2 * torch.cos(math.pi * (j + 0.5) * k / n)
    if b == "DD":
        return 2 * torch.sin(math.pi * (j + 0.5) * (k + 1) / n)
    return 2 * (torch.cos if b == "ND" else torch.sin)(math.pi * (j + 0.5) * (k + 0.5) / n)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "graph"):
        return _exact_step(case, seed)
    if kind == "batch":
        return [_poisson(c, _rhs(c, seed * 1000 + q)) for q, c in enumerate(_batch(case))]
    if kind == "lines":
        f = _normal(case, _generator(seed))
        mx, my = _r2r(case["bc"][:2], case["nx"]), _r2r(case["bc"][2:4], case["ny"])
        return torch.matmul(my, torch.matmul(f, mx.t().contiguous())) * _unit(case)
    f = _rhs(case, seed)
    return _poisson(case, f.float().double() if kind == "f32" else f)
