"""Performance cases: what programs of this framework have it do, through the
public entry points (physis_amd.runtime, .programs, .poisson, .warmstart).

Ranges.  Stencil maps over 3-D grids from 32 points per axis (launch bound) to
512^3, with extents that are multiples of nothing as often as not: 7-point
diffusion with clamped and periodic boundaries, with the reductions a program
follows a run with; 19-point Jacobi sweeps (the residual of each sweep
returned, or not); red-black relaxation; a stencil over user-defined points;
2-D 5- and 9-point maps.  The Poisson solver in each storage type (FP32, BF16,
FP16), single problems and batches.  The warm-start network's prediction
(forward) and its loss gradient (forward and backward) for problems of 32 to
128 points per axis, one to eight at a time.

A case's state holds device grids filled on the GPU from the seed; run() makes
the calls a program makes between copy-in and copy-out, and returns the whole
grids (tensors over the grids' own memory) and whatever numbers the calls
return.  Every call can be made again on the same state: the iterations then
go on from where the last pass left the grids, as a program's would.
"""
from __future__ import annotations

import os

import numpy as np
import torch

import physis_amd
from physis_amd import runtime as ps
from physis_amd.poisson import PoissonSolver
from physis_amd.programs import (Diffusion7, Himeno, RedBlack7, Stencil2D,
                                 Udt7)
from physis_amd.warmstart import UNet

COEF = (0.1, 0.1, 0.1, 0.1, 0.1, 0.1, 0.4)  # ce cw cn cs ct cb cc
OMEGA = float(np.float32(0.8))
WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(physis_amd.__file__)),
                       "weights", "unet128.npz")
# channels in and out of the network's 3x3x3 layers and the level of each;
# only 2 of the first layer's 8 input channels carry data
LAYERS = ((8, 8, 1), (8, 8, 1), (8, 16, 2), (16, 16, 2), (16, 32, 3),
          (32, 32, 3), (48, 16, 2), (16, 16, 2), (24, 8, 1), (8, 8, 1))


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # a small solve: launches and latency are what it costs
        {"name": "diffusion 64^3", "path": "diffusion", "nx": 64, "ny": 64,
         "nz": 64, "sweeps": 100, "periodic": False, "reduce": "sum"},
        # the large diffusion run between two of its reductions
        {"name": "diffusion 512^3", "path": "diffusion", "nx": 512, "ny": 512,
         "nz": 512, "sweeps": 50, "periodic": False, "reduce": "sum max"},
        # an ordinary periodic run whose extents are multiples of nothing
        {"name": "diffusion periodic ragged", "path": "diffusion", "nx": 321,
         "ny": 190, "nz": 157, "sweeps": 20, "periodic": True,
         "reduce": "max"},
        # the 19-point benchmark's size, with the residual of every sweep
        {"name": "himeno 512x256x256", "path": "himeno", "nx": 512, "ny": 256,
         "nz": 256, "sweeps": 20, "residual": True},
        # the same program on a small grid of odd extents
        {"name": "himeno 129x65x65", "path": "himeno", "nx": 129, "ny": 65,
         "nz": 65, "sweeps": 40, "residual": True},
        # red-black relaxation of an ordinary grid
        {"name": "redblack 256^3", "path": "redblack", "nx": 256, "ny": 256,
         "nz": 256, "iterations": 20},
        # a stencil over points with two members
        {"name": "user points 250x200x180", "path": "udt", "nx": 250,
         "ny": 200, "nz": 180, "sweeps": 10},
        # an image-sized 2-D map
        {"name": "2-D 9-point 4096x4096", "path": "stencil2d", "nx": 4096,
         "ny": 4096, "points": 9, "pairs": 5},
        # two refinement steps of a batch of problems, BF16 storage
        {"name": "poisson bf16 8x128^3", "path": "poisson", "nx": 128,
         "ny": 128, "nz": 128, "batch": 8, "storage": "bf16", "inner": 50,
         "steps": 2},
        # the plain FP32 solve of one smaller problem, with its checks
        {"name": "poisson fp32 162x150x140", "path": "poisson", "nx": 162,
         "ny": 150, "nz": 140, "batch": 1, "storage": "fp32", "inner": 20,
         "steps": 3},
        # initial guesses of a batch of problems
        {"name": "network predict 8x128^3", "path": "predict", "nx": 128,
         "ny": 128, "nz": 128, "batch": 8},
        # loss and gradient of a training batch
        {"name": "network gradient 8x128^3", "path": "gradient", "nx": 128,
         "ny": 128, "nz": 128, "batch": 8},
    ]


def _extent(rng, lo, hi):
    """An extent between lo and hi, spread over its logarithm; half of them
    multiples of 4, the others whatever comes."""
    n = int(round(lo * (hi / lo) ** rng.random()))
    return max(lo, n - n % 4) if rng.random() < 0.5 else n


def _box(rng, lo, hi, most):
    """Three extents between lo and hi with at most `most` points."""
    while True:
        n = [_extent(rng, lo, hi) for _ in range(3)]
        if n[0] * n[1] * n[2] <= most:
            return n


def draw(rng):
    path = rng.choice(["diffusion", "diffusion", "himeno", "redblack", "udt",
                       "stencil2d", "poisson", "predict", "gradient"])
    if path == "diffusion":
        nx, ny, nz = _box(rng, 32, 512, 1 << 27)
        return {"path": path, "nx": nx, "ny": ny, "nz": nz,
                "sweeps": 2 * rng.randint(1, 25),
                "periodic": rng.random() < 0.5,
                "reduce": rng.choice(["sum", "max", "sum max", ""])}
    if path == "himeno":
        nx, ny, nz = _box(rng, 32, 512, 1 << 25)
        return {"path": path, "nx": nx, "ny": ny, "nz": nz,
                "sweeps": 2 * rng.randint(1, 10),
                "residual": rng.random() < 0.7}
    if path == "redblack":
        nx, ny, nz = _box(rng, 32, 512, 1 << 26)
        return {"path": path, "nx": nx, "ny": ny, "nz": nz,
                "iterations": rng.randint(1, 20)}
    if path == "udt":
        nx, ny, nz = _box(rng, 32, 512, 1 << 26)
        return {"path": path, "nx": nx, "ny": ny, "nz": nz,
                "sweeps": rng.randint(1, 10)}
    if path == "stencil2d":
        return {"path": path, "nx": _extent(rng, 128, 16384),
                "ny": _extent(rng, 128, 16384), "points": rng.choice([5, 9]),
                "pairs": rng.randint(1, 5)}
    if path == "poisson":
        batch = rng.choice([1, 1, 2, 4, 8])
        nx, ny, nz = _box(rng, 32, 256, (1 << 24) // batch)
        return {"path": path, "nx": nx - nx % 2, "ny": ny, "nz": nz,
                "batch": batch, "storage": rng.choice(["bf16", "fp16", "fp32"]),
                "inner": 2 * rng.randint(5, 16), "steps": rng.randint(1, 3)}
    return {"path": path, "nx": 16 * rng.randint(2, 8),
            "ny": 16 * rng.randint(2, 8), "nz": 16 * rng.randint(2, 8),
            "batch": rng.randint(1, 8)}


# ------------------------------------------------------------- grids, inputs
class _Memory:
    """A grid's device memory for torch, holding the grid alive."""

    def __init__(self, owner, address, count, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {
            "shape": (count,), "typestr": typestr, "data": (address, False),
            "version": 2, "strides": None}


class _Owned:
    """A grid that is freed with the last state or tensor that uses it."""

    def __init__(self, grid, free):
        self.grid, self._free = grid, free

    def __del__(self):
        self._free(self.grid)


def _grid(shape, dtype=np.float32):
    """(grid, tensor over its memory)."""
    g = ps.PSGridNew(list(shape), dtype)
    own = _Owned(g, ps.PSGridFree)
    n = int(np.prod(shape))
    typestr = "<f4" if g.dtype == np.float32 else "<f8"
    return g, torch.as_tensor(_Memory(own, g.handle.contents.p, n, typestr),
                              device="cuda")


def _random(case, seed, count):
    """Tensors in [0, 1), [nz][ny][nx], one after another from the seed."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 7919 + 17)
    shape = ((case.get("batch", 1) * case["nz"],) if "nz" in case else ()) + \
        (case["ny"], case["nx"])
    for _ in range(count):
        yield torch.rand(shape, generator=gen, device="cuda")


def _inside(case):
    """1 at the interior points of every problem, 0 on its faces."""
    m = torch.zeros((case.get("batch", 1), case["nz"], case["ny"],
                     case["nx"]), device="cuda")
    m[:, 1:-1, 1:-1, 1:-1] = 1.0
    return m.reshape(-1, case["ny"], case["nx"])


def _gaussians(case, seed, lo, hi):
    """Every problem a sum of lo .. hi Gaussians of amplitude +-1 and width 2
    cells to an eighth of its smallest extent."""
    g = np.random.default_rng(int(seed) * 31 + 5)
    n = (case["nz"], case["ny"], case["nx"])
    wide = max(3.0, min(n) / 8.0)
    out = torch.empty((case["batch"],) + n, device="cuda")
    for q in range(case["batch"]):
        count = int(g.integers(lo, hi + 1))
        width = g.uniform(2.0, wide, count)
        sign = g.choice([-1.0, 1.0], count)
        ax = []
        for d in range(3):
            at = torch.arange(n[d], dtype=torch.float64)[None, :]
            c = torch.as_tensor(g.uniform(0, n[d], count))[:, None]
            w = torch.as_tensor(width)[:, None]
            ax.append(torch.exp(-0.5 * ((at - c) / w) ** 2).cuda())
        yx = (ax[1][:, :, None] * ax[2][:, None, :]).reshape(count, -1)
        az = ax[0] * torch.as_tensor(sign).cuda()[:, None]
        out[q] = (az.T @ yx).reshape(n).float()
    return out.reshape(-1, case["ny"], case["nx"])


def _himeno_inputs(case, seed):
    """The benchmark's coefficients (1% noise on each) and pressure."""
    r = _random(case, seed, 11)
    noise = lambda: 0.01 * (2.0 * next(r) - 1.0)  # noqa: E731
    c = [1.0 + noise() for _ in range(3)]
    c.append((1.0 + noise()) / 6.0)
    c += [noise() for _ in range(3)]
    c += [1.0 + noise() for _ in range(3)]
    c.append(_inside(case))
    c.append(torch.zeros_like(c[0]))
    k = torch.linspace(0, 1, case["nz"], device="cuda") ** 2
    return c, k[:, None, None] + 1e-3 * next(r)


def _poisson_inputs(case, seed):
    """A variable-conductivity operator (5% noise on the face coefficients,
    rows that balance) and a right-hand side of Gaussians."""
    r = _random(case, seed, 6)
    face = [1.0 + 0.05 * (2.0 * next(r) - 1.0) for _ in range(6)]
    zero = torch.zeros_like(face[0])
    inside = _inside(case)
    return face[:3] + [1.0 / sum(face)] + [zero] * 3 + face[3:] + \
        [inside, _gaussians(case, seed, 4, 16) * inside]


def _network_inputs(case, seed):
    """Right-hand sides, boundary masks and solutions as large and smooth as
    those the network is trained on."""
    inside = _inside(case)
    return (_gaussians(case, seed, 4, 24) * inside, inside,
            30.0 * _gaussians(case, seed + 1, 4, 24) * inside)


# -------------------------------------------------------------- prepare, run
def prepare(case, seed):
    ps.PSInit()
    path = case["path"]
    s = {"case": case}

    def grid(name, value=None, shape=None, dtype=np.float32):
        shape = shape or (case["nx"], case["ny"],
                          case.get("batch", 1) * case["nz"])
        s[name], s[name + "_t"] = _grid(shape, dtype)
        if value is not None:
            s[name + "_t"].copy_(value.reshape(-1))

    if path == "diffusion":
        u = next(_random(case, seed, 1))
        s["program"] = Diffusion7()
        grid("a", u)
        grid("b", u)
    elif path == "himeno":
        c, p = _himeno_inputs(case, seed)
        s["program"] = Himeno()
        for k, v in enumerate(c):
            grid("c%d" % k, v)
        grid("a", p)
        grid("b", p)
    elif path == "redblack":
        s["program"] = RedBlack7()
        grid("a", next(_random(case, seed, 1)))
    elif path == "udt":
        p, q = _random(case, seed, 2)
        n = p.numel()
        s["program"] = Udt7()
        g = s["program"].new((case["nx"], case["ny"], case["nz"]),
                             torch.stack([p.reshape(-1), q.reshape(-1)], 1)
                             .cpu().numpy())
        own = _Owned(g, s["program"].free)
        s["a"] = g
        at = ps.C.cast(g, ps.PSGridPtr)
        member = ps.runtime().__PSGridUserMember
        member.argtypes = [ps.PSGridPtr, ps.C.c_int]
        member.restype = ps.C.c_void_p
        s["p_t"], s["q_t"] = (torch.as_tensor(
            _Memory(own, member(at, m), n, "<f4"), device="cuda")
            for m in (0, 1))
    elif path == "stencil2d":
        u = next(_random(case, seed, 1))
        s["program"] = Stencil2D()
        grid("a", u, (case["nx"], case["ny"]))
        grid("b", u, (case["nx"], case["ny"]))
    elif path == "poisson":
        c = _poisson_inputs(case, seed)
        for k, v in enumerate(c):
            grid("c%d" % k, v)
        grid("a", dtype=np.float32 if case["storage"] == "fp32"
             else np.float64)
        torch.cuda.synchronize()
        s["solver"] = PoissonSolver([s["c%d" % k] for k in range(12)],
                                    case["batch"], case["storage"])
    else:
        rhs, inside, target = _network_inputs(case, seed)
        w = np.load(WEIGHTS)
        s["net"] = UNet(case["nx"], case["ny"], case["nz"], case["batch"],
                        float(w["out_scale"]))
        s["net"].set_params(w["params"])
        grid("rhs", rhs)
        grid("bnd", inside)
        if path == "predict":
            grid("a", dtype=np.float64)
        else:
            grid("target", target)
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    path = case["path"]
    if path == "diffusion":
        s["program"].run(s["a"], s["b"], case["sweeps"], COEF,
                         periodic=case["periodic"])
        out = {"a": s["a_t"], "b": s["b_t"]}
        if "sum" in case["reduce"]:
            out["sum"] = ps.PSReduce(ps.PS_SUM, s["a"])
        if "max" in case["reduce"]:
            out["max"] = ps.PSReduce(ps.PS_MAX, s["a"])
        return out
    if path == "himeno":
        coefs = [s["c%d" % k] for k in range(12)]
        if case["residual"]:
            res = s["program"].run_gosa(case["sweeps"], s["a"], s["b"], coefs,
                                        OMEGA)
            return {"a": s["a_t"], "b": s["b_t"], "residual": res}
        s["program"].run(case["sweeps"], s["a"], s["b"], coefs, OMEGA)
        return {"a": s["a_t"], "b": s["b_t"]}
    if path == "redblack":
        s["program"].run(s["a"], case["iterations"], COEF)
        return s["a_t"]
    if path == "udt":
        s["program"].run(s["a"], case["sweeps"], COEF)
        return {"p": s["p_t"], "q": s["q_t"]}
    if path == "stencil2d":
        s["program"].run(s["a"], s["b"], case["points"], case["pairs"],
                         1.0 / case["points"])
        return {"a": s["a_t"], "b": s["b_t"]}
    if path == "poisson":
        solve = s["solver"].solve_plain if case["storage"] == "fp32" else \
            s["solver"].solve_mixed
        st = solve(s["a"], OMEGA, 0.0, case["inner"],
                   case["inner"] * case["steps"])
        return {"a": s["a_t"], "residual": st["rel_residual"]}
    if path == "predict":
        s["net"].predict(s["rhs"], s["bnd"], 0, case["batch"], s["a"])
        return s["a_t"]
    loss, grad = s["net"].loss_grad(s["rhs"], s["bnd"], s["target"], 0,
                                    case["batch"])
    return {"loss": loss, "gradient": grad}


# ----------------------------------------------------------- work, tolerance
def work(case):
    path = case["path"]
    n = case["nx"] * case["ny"] * case.get("nz", 1) * case.get("batch", 1)
    if path == "diffusion":
        return {"bytes": 12 * n, "flops": 13 * n * case["sweeps"]}
    if path == "himeno":
        return {"bytes": 60 * n, "flops": 34 * n * case["sweeps"]}
    if path == "redblack":
        return {"bytes": 8 * n, "flops": 13 * n * case["iterations"]}
    if path == "udt":
        return {"bytes": 8 * n, "flops": 13 * n * case["sweeps"]}
    if path == "stencil2d":
        return {"bytes": 12 * n,
                "flops": case["points"] * n * 2 * case["pairs"]}
    if path == "poisson":
        sweeps, e = case["inner"] * case["steps"], \
            8 if case["storage"] != "fp32" else 4
        return {"bytes": (48 + 2 * e) * n,
                "flops": 34 * n * (sweeps + case["steps"] + 1)}
    pts = {1: n, 2: n / 64, 3: n / 4096}
    conv = sum(2 * 27 * ci * co * pts[lv] for ci, co, lv in LAYERS) - \
        2 * 27 * 6 * 8 * n
    if path == "predict":
        return {"bytes": 16 * n, "flops": conv + 16 * n}
    return {"bytes": 12 * n, "flops": 3 * conv + 48 * n}


def tolerance(case):
    # about four times the difference from the 64-bit results below: 7e-7
    # after 100 sweeps of diffusion, 2e-7 and less for the other FP32 maps,
    # 6e-3 with BF16 coefficients, 6e-3 through the BF16 network
    path = case["path"]
    if path in ("diffusion", "himeno"):
        return {"rel": 3e-6}
    if path in ("redblack", "udt", "stencil2d"):
        return {"rel": 1e-6}
    if path == "poisson":
        return {"rel": {"fp32": 1e-6, "fp16": 5e-3,
                        "bf16": 2.5e-2}[case["storage"]]}
    return {"rel": 2.5e-2}


# --------------------------------------------------------------------- exact
def exact(case, seed):
    path = case["path"]
    if path in ("predict", "gradient"):
        return _network_exact(case, seed)
    if path == "diffusion":
        a = next(_random(case, seed, 1)).double()
        b = a
        for _ in range(case["sweeps"]):
            b, a = a, _diffuse(a, case["periodic"])
        out = {"a": a.reshape(-1), "b": b.reshape(-1)}
        if "sum" in case["reduce"]:
            out["sum"] = float(a.sum())
        if "max" in case["reduce"]:
            out["max"] = float(a.max())
        return out
    if path == "himeno":
        c, p = _himeno_inputs(case, seed)
        c, a = [v.double() for v in c], p.double()
        b, res = a, []
        for _ in range(case["sweeps"]):
            ss = _jacobi(c, a, a * c[3].reciprocal())[1] * c[3]
            ss = ss[1:-1, 1:-1, 1:-1]
            res.append(float((ss * ss).sum()))
            b, a = a, a.clone()
            a[1:-1, 1:-1, 1:-1] += OMEGA * ss
        out = {"a": a.reshape(-1), "b": b.reshape(-1)}
        if case["residual"]:
            out["residual"] = np.array(res)
        return out
    if path == "redblack":
        a = next(_random(case, seed, 1)).double()
        z, y, x = (torch.arange(n, device="cuda") for n in a.shape)
        odd = (z[:, None, None] + y[None, :, None] + x[None, None, :]) % 2
        inside = _inside(case) > 0
        for _ in range(case["iterations"]):
            for colour in (0, 1):
                a = torch.where(inside & (odd == colour),
                                _diffuse(a, True), a)
        return a.reshape(-1)
    if path == "udt":
        p, q = (v.double() for v in _random(case, seed, 2))
        q = torch.where(_inside(case) > 0, _diffuse(p, True), q)
        return {"p": p.reshape(-1), "q": q.reshape(-1)}
    if path == "stencil2d":
        a = next(_random(case, seed, 1)).double()
        b = a.clone()
        for _ in range(2 * case["pairs"]):
            t = a.clone()
            if case["points"] == 5:
                v = a[1:-1, 1:-1] + a[1:-1, :-2] + a[1:-1, 2:] + \
                    a[:-2, 1:-1] + a[2:, 1:-1]
            else:
                v = a[:, 1:-1] + a[:, :-2] + a[:, 2:]
                v = v[1:-1] + v[:-2] + v[2:]
            t[1:-1, 1:-1] = v / case["points"]
            b, a = a, t
        return {"a": a.reshape(-1), "b": b.reshape(-1)}
    c = [v.double() for v in _poisson_inputs(case, seed)]
    n = (case["batch"], case["nz"], case["ny"], case["nx"])
    c = [v.reshape(n) for v in c]
    a = torch.zeros(n, dtype=torch.float64, device="cuda")
    for _ in range(case["inner"] * case["steps"]):
        for q in range(case["batch"]):
            d = _jacobi([v[q] for v in c], a[q], a[q] / c[3][q])[1]
            a[q] += OMEGA * c[3][q] * d
    rel = 0.0
    for q in range(case["batch"]):
        r = _jacobi([v[q] for v in c], a[q], a[q] / c[3][q])[1]
        rel = max(rel, float(r.norm() / (c[11][q] * c[10][q]).norm()))
    return {"a": a.reshape(-1), "residual": rel}


def _diffuse(a, periodic):
    out = float(np.float32(0.4)) * a
    for d in range(3):
        for s in (1, -1):
            v = torch.roll(a, s, d)
            if not periodic:  # the edge value again
                e = 0 if s == 1 else a.shape[d] - 1
                v.select(d, e).copy_(a.select(d, e))
            out += float(np.float32(0.1)) * v
    return out


def _jacobi(c, p, diagonal):
    """(neighbour sum, residual masked by bnd) of the 19-point operator."""
    def at(dx, dy, dz):
        return torch.roll(p, (-dz, -dy, -dx), (0, 1, 2))
    s = c[0] * at(0, 0, 1) + c[1] * at(0, 1, 0) + c[2] * at(1, 0, 0)
    s += c[7] * at(0, 0, -1) + c[8] * at(0, -1, 0) + c[9] * at(-1, 0, 0)
    s += c[11]
    for k, (u, v) in zip((4, 5, 6), (((0, 1, 0), (0, 0, 1)),
                                     ((1, 0, 0), (0, 1, 0)),
                                     ((1, 0, 0), (0, 0, 1)))):
        t = torch.zeros_like(p)
        for e in (1, -1):
            for f in (1, -1):
                t += e * f * at(*(e * i + f * j for i, j in zip(u, v)))
        s += c[k] * t
    return s, (s - diagonal) * c[10]


class _Conv(torch.autograd.Function):
    """3x3x3 convolution, zero padded, as products tap by tap: x
    [z, y, x, in], w [out, 27, in]."""

    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        d, h, v = x.shape[:3]
        y = 0
        for t in range(27):
            k, j, i = t // 9, t // 3 % 3, t % 3
            y = y + xp[k:k + d, j:j + h, i:i + v] @ w[:, t].T
        return y

    @staticmethod
    def backward(ctx, g):
        x, w = ctx.saved_tensors
        d, h, v = x.shape[:3]
        gx = torch.zeros((d + 2, h + 2, v + 2, x.shape[3]), dtype=x.dtype,
                         device=x.device)
        xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        gw = torch.empty_like(w)
        gf = g.reshape(d * h, v, -1).transpose(1, 2).contiguous()
        for t in range(27):
            k, j, i = t // 9, t // 3 % 3, t % 3
            gx[k:k + d, j:j + h, i:i + v] += g @ w[:, t]
            part = xp[k:k + d, j:j + h, i:i + v].reshape(d * h, v, -1)
            gw[:, t] = torch.bmm(gf, part).sum(0)
        return gx[1:-1, 1:-1, 1:-1], gw


def _network_exact(case, seed):
    rhs, inside, target = _network_inputs(case, seed)
    w = np.load(WEIGHTS)
    scale = float(w["out_scale"])
    p = torch.tensor(w["params"], dtype=torch.float64, device="cuda",
                     requires_grad=case["path"] == "gradient")
    n = (case["nz"], case["ny"], case["nx"])
    total = case["batch"] * n[0] * n[1] * n[2]
    layers, off = [], 0
    for ci, co, _ in LAYERS:
        k = co * 27 * ci
        layers.append((p[off:off + k].reshape(co, 27, ci),
                       p[off + k:off + k + co]))
        off += k + co

    def conv(l, x):
        return torch.relu(_Conv.apply(x, layers[l][0]) + layers[l][1])

    def pool(x):
        d, h, v, ch = x.shape
        return x.reshape(d // 4, 4, h // 4, 4, v // 4, 4, ch).mean((1, 3, 5))

    def up(x):
        for d in range(3):
            x = x.repeat_interleave(4, d)
        return x

    loss, out = 0.0, []
    for q in range(case["batch"]):
        r, m, t = (v.reshape((-1,) + n)[q].double()
                   for v in (rhs, inside, target))
        x = torch.stack([r, m] + [torch.zeros_like(r)] * 6, 3)
        e1 = conv(1, conv(0, x))
        e2 = conv(3, conv(2, pool(e1)))
        e3 = conv(5, conv(4, pool(e2)))
        d2 = conv(7, conv(6, torch.cat([up(e3), e2], 3)))
        d1 = conv(9, conv(8, torch.cat([up(d2), e1], 3)))
        y = d1 @ p[off:off + 8] + p[off + 8]
        if case["path"] == "predict":
            out.append((scale * y * m).detach().reshape(-1))
        else:
            part = ((y - t / scale) ** 2).sum() / total
            part.backward()
            loss += float(part.detach())
    if case["path"] == "predict":
        return torch.cat(out)
    return {"loss": loss, "gradient": p.grad}
