"""The work that users of this package have it do, as cases with a run time and a result.

Kinds of case:
  apply   one application of the Stokes/Brinkman operator to a device vector
          (an outer Krylov method or a nonlinear loop around LinearMapping);
  hooks   one design update of a user's own optimiser loop on host arrays: objective,
          its gradient, sensitivity, density filter both ways, OC update;
  solve   a new design and one solve from zero, the solution fetched to the host;
  to      a short topology-optimization run on the device from a given design,
          OC or MMA, the final design fetched to the host;
  learn   training epochs of the learned initial guess on recorded solutions.
Grid sides are the ones the solver takes (4 * 2^k).
"""
import ctypes
import functools
import math

import numpy as np
import torch

from stokes_to_amd.problems import channel_problem, dof_sizes, reference_test0
from stokes_to_amd.steady import FluidSteadyState

BYTES = {"fp64": 8, "fp32": 4, "bf16": 2}
PDOUBLE = ctypes.POINTER(ctypes.c_double)


def listed():
    return [
        # the smallest call in use: the operator inside a user's own iteration on a coarse 3D grid
        {"name": "apply_3d_32", "kind": "apply", "dim": 3, "n": 32, "mean": 0.3, "sigma": 4.0},
        # the same at the size of the large runs, where HBM bounds it
        {"name": "apply_3d_256", "kind": "apply", "dim": 3, "n": 256, "mean": 0.2, "sigma": 8.0},
        # a user's own optimiser on host arrays, one update (the reference's call pattern)
        {"name": "hooks_3d_64", "kind": "hooks", "dim": 3, "n": 64, "mean": 0.3, "radius": 1.5, "volfrac": 0.3},
        # the 2D 64^2 configuration: plain FP64, 1e-10; launch latency bounds it
        {"name": "solve_2d_64_fp64", "kind": "solve", "dim": 2, "n": 64, "precision": "fp64", "rtol": 1e-10,
         "mean": 0.15, "sigma": 6.0},
        # the 3D 64^3 configuration, plain FP64 and BF16 smoothing
        {"name": "solve_3d_64_fp64", "kind": "solve", "dim": 3, "n": 64, "precision": "fp64", "rtol": 1e-8,
         "mean": 0.3, "sigma": 8.0},
        {"name": "solve_3d_64_bf16", "kind": "solve", "dim": 3, "n": 64, "precision": "bf16", "rtol": 1e-8,
         "mean": 0.3, "sigma": 8.0},
        # a single 128^3 solve in mixed precision
        {"name": "solve_3d_128_fp32", "kind": "solve", "dim": 3, "n": 128, "precision": "fp32", "rtol": 1e-8,
         "mean": 0.25, "sigma": 8.0},
        # the plain FP64 solve of the largest configuration
        {"name": "solve_3d_256_fp64", "kind": "solve", "dim": 3, "n": 256, "precision": "fp64", "rtol": 1e-8,
         "mean": 0.2, "sigma": 8.0},
        # the 2D 256^2 configuration with FP32 smoothing: the first design iterations of an OC run
        {"name": "to_2d_256_fp32", "kind": "to", "problem": "channel", "dim": 2, "n": 256, "precision": "fp32",
         "rtol": 1e-10, "volfrac": 0.15, "radius": 1.5, "optimizer": "oc", "init": "keep", "steps": 4},
        # the reference's own demo: closed box, MMA on the unfiltered density, solves from zero
        {"name": "to_3d_64_mma", "kind": "to", "problem": "box", "dim": 3, "n": 64, "precision": "fp64",
         "rtol": 1e-8, "volfrac": 0.3, "radius": 1.0, "optimizer": "mma", "init": "zero", "steps": 3},
        # the 256^3 configuration: mixed precision with warm starts, OC
        {"name": "to_3d_256_fp32", "kind": "to", "problem": "channel", "dim": 3, "n": 256, "precision": "fp32",
         "rtol": 1e-8, "volfrac": 0.2, "radius": 1.5, "optimizer": "oc", "init": "keep", "steps": 4},
        # online training of the 128^3 configuration's network (forward, backward, Adam)
        {"name": "learn_3d_128", "kind": "learn", "dim": 3, "n": 128, "precision": "fp32", "mean": 0.25,
         "sigma": 8.0, "samples": 2, "epochs": 3},
    ]


def _log(rng, lo, hi):
    return round(math.exp(rng.uniform(math.log(lo), math.log(hi))), 3)


def draw(rng):
    kind = rng.choice(["apply", "hooks", "solve", "solve", "solve", "to", "to", "to", "learn"])
    dim = rng.choice([2, 3, 3])
    mean = round(rng.uniform(0.15, 0.45), 4)
    if kind == "apply":
        n = rng.choice([32, 64, 128, 256, 512, 1024] if dim == 2 else [16, 32, 64, 128, 256])
        return {"kind": "apply", "dim": dim, "n": n, "mean": mean, "sigma": _log(rng, 2.0, n / 4)}
    if kind == "hooks":
        n = rng.choice([32, 64, 128, 256] if dim == 2 else [16, 32, 64, 128])
        return {"kind": "hooks", "dim": dim, "n": n, "mean": mean, "radius": round(rng.uniform(1.1, 3.4), 3),
                "volfrac": round(mean + rng.uniform(-0.03, 0.03), 4)}
    if kind == "solve":
        n = rng.choice([32, 64, 128, 256, 512] if dim == 2 else [16, 32, 64, 128, 256])
        return {"kind": "solve", "dim": dim, "n": n, "precision": rng.choice(["fp64", "fp32", "bf16"]),
                "rtol": rng.choice([1e-8, 1e-8, 1e-10]), "mean": mean, "sigma": _log(rng, 4.0, max(5.0, n / 8))}
    if kind == "to":
        n = rng.choice([32, 64, 128, 256] if dim == 2 else [16, 32, 64, 128])
        opt = rng.choice(["oc", "oc", "mma"])
        return {"kind": "to", "problem": "channel", "dim": dim, "n": n, "precision": rng.choice(["fp64", "fp32"]),
                "rtol": rng.choice([1e-8, 1e-10]), "volfrac": round(rng.uniform(0.15, 0.4), 4),
                "radius": 1.0 if opt == "mma" else round(rng.uniform(1.2, 2.9), 3), "optimizer": opt,
                "init": rng.choice(["zero", "keep", "keep"]), "steps": rng.randint(2, 5)}
    return {"kind": "learn", "dim": 3, "n": rng.choice([32, 64, 128]), "precision": rng.choice(["fp64", "fp32"]),
            "mean": mean, "sigma": _log(rng, 4.0, 9.0), "samples": rng.randint(1, 3), "epochs": rng.randint(1, 4)}


# ------------------------------------------------------------------ inputs

@functools.lru_cache(maxsize=4)
def _problem(kind, dim, n):
    return channel_problem(dim, n) if kind == "channel" else reference_test0(dim, n)


def _field(dim, n, sigma, gen):
    """Gaussian random field of correlation length sigma cells, zero mean, unit variance."""
    w = torch.randn((n,) * dim, generator=gen, device="cuda", dtype=torch.float64)
    f = torch.fft.fftfreq(n, device="cuda", dtype=torch.float64)
    k2 = sum(f.reshape([n if a == b else 1 for b in range(dim)]) ** 2 for a in range(dim))
    g = torch.fft.ifftn(torch.fft.fftn(w) * torch.exp(-2.0 * math.pi ** 2 * sigma ** 2 * k2)).real
    return (g - g.mean()) / g.std()


def _density(dim, n, mean, sigma, gen):
    """Logistic squash of a random field with the shift that gives the wanted mean."""
    g = _field(dim, n, sigma, gen)
    lo, hi = -20.0, 20.0
    for _ in range(40):
        s = 0.5 * (lo + hi)
        lo, hi = (lo, s) if torch.sigmoid(g + s).mean().item() > mean else (s, hi)
    return torch.sigmoid(g + 0.5 * (lo + hi)).clamp_min(1e-3).reshape(-1).contiguous()


def _start_design(dim, n, volfrac, gen):
    """The design of a run's first steps: near the uniform one."""
    return (volfrac * (1.0 + 0.1 * _field(dim, n, max(2.0, n / 16), gen))).clamp(0.02, 0.98).reshape(-1).contiguous()


def _state_vector(P, gen, amplitude):
    """A smooth velocity and pressure field, with the boundary values on the fixed faces."""
    parts = []
    for f in range(P.dim + 1):
        g = amplitude * _field(P.dim, P.n + 1, max(2.0, P.n / 12), gen)
        parts.append(g[tuple(slice(0, P.n + (f == 1 + a)) for a in range(P.dim))].reshape(-1))
    x = torch.cat(parts)
    return torch.where(_dev(P.fixed).bool(), _dev(P.dirichlet), x)


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _ptr(t):
    return ctypes.cast(ctypes.c_void_p(t.data_ptr()), PDOUBLE)


def _solver(P, **kw):
    a = P.alpha
    s = FluidSteadyState(P.dim, P.n, alpha_max=a.alpha_max, alpha_min=a.alpha_min, q=a.q, power=a.power,
                         alpha_scale=a.scale, **kw)
    s.init_boundary(P.fixed, closed=P.closed)
    s.update_b(body=P.body if P.closed else None, dirichlet=None if P.closed else P.dirichlet)
    return s


def _inputs(case, seed):
    """What a case's inputs are, from the seed alone."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    dim, n, kind = case["dim"], case["n"], case["kind"]
    P = _problem(case.get("problem", "channel"), dim, n)
    if kind == "apply":
        return P, {"rho": _density(dim, n, case["mean"], case["sigma"], gen), "x": _state_vector(P, gen, 1.0)}
    if kind == "hooks":
        return P, {"rho": _density(dim, n, case["mean"], n / 8, gen), "x": _state_vector(P, gen, 1.0),
                   "lam": _state_vector(P, gen, 0.05)}
    if kind == "solve":
        return P, {"rho": _density(dim, n, case["mean"], case["sigma"], gen)}
    if kind == "to":
        return P, {"rho": _start_design(dim, n, case["volfrac"], gen)}
    return P, {"rhos": [_density(dim, n, case["mean"], case["sigma"], gen) for _ in range(case["samples"])]}


def prepare(case, seed):
    P, st = _inputs(case, seed)
    kind = case["kind"]
    st["case"] = case
    if kind == "apply":
        st["s"] = _solver(P)
        st["s"].set_design(st["rho"].cpu().numpy())
        st["y"] = torch.zeros_like(st["x"])
    elif kind == "hooks":
        st.update({k: st[k].cpu().numpy() for k in ("rho", "x", "lam")})
        st["s"] = _solver(P, filter_radius=case["radius"])
        st["s"].set_design(st["rho"])
    elif kind == "solve":
        st["s"] = _solver(P, precision=case["precision"], rtol=case["rtol"])
    elif kind == "to":
        st["s"] = _solver(P, precision=case["precision"], rtol=case["rtol"], filter_radius=case["radius"],
                          optimizer=case["optimizer"])
    else:
        s = st["s"] = _solver(P, precision=case["precision"])
        for rho in st.pop("rhos"):
            s.set_design(rho.cpu().numpy())
            s.solve(init="zero", fetch=False)
            s.record_sample()
        st["params"] = s.net_params()
    torch.cuda.synchronize()
    return st


def run(st):
    case, s = st["case"], st["s"]
    kind = case["kind"]
    if kind == "apply":
        s._check(s.lib.st_apply_device(s.h, st["x"].data_ptr(), st["y"].data_ptr()))
        return st["y"]
    if kind == "hooks":
        J = s.compute_energy(st["x"])
        gx = s.compute_gradient_x(st["x"])
        dj = s.sensitivity(st["rho"], st["x"], st["lam"])
        dc = s.filter(dj, transpose=True)
        rho, change = s.oc_update(st["rho"], dc, case["volfrac"])
        return {"J": J, "gx": gx, "dj": dj, "dc": dc, "rho": rho, "change": change, "rhof": s.filter(rho)}
    if kind == "solve":
        s._check(s.lib.st_set_design_device(s.h, _ptr(st["rho"])))
        return s.solve(init="zero")[0]
    if kind == "to":
        s._check(s.lib.st_set_design_device(s.h, _ptr(st["rho"])))
        s.reset_solution()
        s.mma_reset()
        rho_min = 0.01 if case["optimizer"] == "mma" else 1e-3
        J = [s.to_step(case["volfrac"], rho_min=rho_min, init=case["init"])["J"] for _ in range(case["steps"])]
        return {"J": J, "rho": s.get_design()}
    s.net_set_params(st["params"])
    loss = s.net_train(case["epochs"], 1e-3)
    return {"loss": loss, "params": s.net_params()}


# ------------------------------------------------------- what a pass needs

def work(case):
    dim, n, kind = case["dim"], case["n"], case["kind"]
    nc, _, _, _, tot = dof_sizes(dim, n)
    nf = tot - nc
    if kind == "apply":
        return {"bytes": 8.0 * (2 * nc + 3 * nf), "flops": 60.0 * nc}
    if kind == "hooks":  # x and alpha in; gx out; rho, x, lam in; dj, dc, rho, filtered rho out
        return {"bytes": 8.0 * (2 * tot + 2 * nf + 2 * tot + 8 * nc), "flops": 400.0 * nc}
    if kind == "learn":
        v = (n // 4) ** 3
        # 16/32/64 channels over three grids: multiply-adds of the forward pass per voxel of the finest
        macs = 27.0 * (16 * 16 + 16 * 16 + (16 * 32 + 32 * 32) / 8 + (32 * 64 + 64 * 64) / 64
                       + (96 * 32 + 32 * 32) / 8 + 48 * 16 + 16 * 16) + 16 * 16
        passes = case["epochs"] * case["samples"]
        return {"bytes": 8.0 * v * 4 * passes, "flops": 6.0 * macs * v * passes}
    # a solve: FGMRES iterations (a nominal number of them: 12 from zero, 5 from a previous solution) of
    # one operator application, a V(1,2) cycle over the levels (x, b, alpha read and x written once per
    # sweep; residual, restriction and prolongation beside them) and the orthogonalisation
    sv = BYTES[case["precision"]]
    geo = 8.0 / 7.0 if dim == 3 else 4.0 / 3.0
    cycle = sv * ((2 * nc + 3 * nf) + geo * (3 * (3 * nc + 4 * nf) + 3 * (nc + nf)) + 6 * (nc + nf))
    per = {"bytes": cycle, "flops": (60.0 + geo * 3 * 260.0) * nc}
    io = 8.0 * (nc + nf + tot)
    if kind == "solve":
        return {"bytes": 12 * per["bytes"] + io, "flops": 12 * per["flops"]}
    its = 24 * case["steps"] if case["init"] == "zero" else 24 + 10 * (case["steps"] - 1)
    return {"bytes": its * per["bytes"] + case["steps"] * (2 * io + 80.0 * nc),
            "flops": its * per["flops"] + 400.0 * nc * case["steps"]}


# ------------------------------------------- the same in plain torch, 64 bits

def _shift(a, axis, by, dim):
    """a[index + by along axis], zero outside; axis counts the last dim axes."""
    ax = a.dim() - dim + axis
    out = torch.zeros_like(a)
    m = a.shape[ax]
    if by > 0:
        out.narrow(ax, 0, m - by).copy_(a.narrow(ax, by, m - by))
    else:
        out.narrow(ax, -by, m + by).copy_(a.narrow(ax, 0, m + by))
    return out


def _split(dim, n, v):
    """A (batch of) dof vector(s) as [p, u_x, ...] on the (n+1)^dim node box, zero outside each field."""
    out, o = [], 0
    for f in range(dim + 1):
        sh = [n + (f == 1 + a) for a in range(dim)]
        m = math.prod(sh)
        w = torch.zeros(*v.shape[:-1], *([n + 1] * dim), dtype=v.dtype, device=v.device)
        w[(...,) + tuple(slice(0, q) for q in sh)] = v[..., o:o + m].reshape(*v.shape[:-1], *sh)
        out.append(w)
        o += m
    return out


def _join(dim, n, fields):
    cut = [f[(...,) + tuple(slice(0, n + (i == 1 + a)) for a in range(dim))] for i, f in enumerate(fields)]
    return torch.cat([c.reshape(*c.shape[:c.dim() - dim], -1) for c in cut], dim=-1)


def _operator(dim, n, fixed, alpha, x, objective=False, masked=True):
    """A x (or the objective's G x) of the Stokes/Brinkman system on the MAC grid; alpha per face."""
    ones = torch.ones_like(fixed, dtype=torch.float64)
    m = [a * (1 - b) for a, b in zip(_split(dim, n, ones), _split(dim, n, fixed.double()))]
    X, al = _split(dim, n, x), _split(dim, n, alpha)
    w = [X[1 + d] * (m[1 + d] if masked else 1.0) for d in range(dim)]
    div = sum(_shift(w[d], d, 1, dim) - w[d] for d in range(dim))
    g = div * m[0]
    rows = [torch.zeros_like(X[0]) if objective else g + (1 - m[0]) * X[0]]
    for d in range(dim):
        r = _shift(g, d, -1, dim) - g
        for e in range(dim):
            if e != d:
                c = w[d] - _shift(w[d], e, -1, dim) - w[e] + _shift(w[e], d, -1, dim)
                r = r + c - _shift(c, e, 1, dim)
        if objective and dim == 2:  # the 2D objective: face Laplacian of the unmasked velocity
            u = X[1 + d]
            r = 2 * dim * u - sum(_shift(u, e, s, dim) for e in range(dim) for s in (-1, 1))
        elif not objective:
            r = r + _shift(X[0], d, -1, dim) - X[0]
        r = r + al[1 + d] * X[1 + d]
        rows.append(r * m[1 + d] + (0.0 if objective else (1 - m[1 + d]) * X[1 + d]))
    return _join(dim, n, rows)


def _cell_alpha(P, rho):
    a, r = P.alpha, rho ** P.alpha.power
    return a.scale * (a.alpha_max + (a.alpha_min - a.alpha_max) * r * (1 + a.q) / (r + a.q))


def _face_alpha(P, rho):
    """Half of each adjacent cell's penalty, on free faces, as a dof vector."""
    dim, n = P.dim, P.n
    c = torch.zeros([n + 1] * dim, dtype=torch.float64, device=rho.device)
    c[tuple(slice(0, n) for _ in range(dim))] = 0.5 * _cell_alpha(P, rho).reshape([n] * dim)
    v = _join(dim, n, [torch.zeros_like(c)] + [c + _shift(c, d, -1, dim) for d in range(dim)])
    return v * (1 - _dev(P.fixed).double())


def _filter(dim, n, R, v, transpose):
    """Cone filter of radius R cells, normalised by the weight sum of the cell."""
    r = math.ceil(R) - 1
    box = torch.ones([n] * dim, dtype=torch.float64, device=v.device)

    def sums(a):
        out = torch.zeros_like(a)
        for o in np.ndindex(*([2 * r + 1] * dim)):
            off = [q - r for q in o]
            h = R - math.sqrt(sum(q * q for q in off))
            if h > 0:
                t = a
                for ax, q in enumerate(off):
                    t = _shift(t, ax, q, dim) if q else t
                out += h * t
        return out

    W, a = sums(box), v.reshape([n] * dim)
    return (sums(a / W) if transpose else sums(a) / W).reshape(-1)


def exact(case, seed):
    kind, dim, n = case["kind"], case["dim"], case["n"]
    if kind in ("to", "learn") or (kind == "solve" and n ** dim > 4096):
        return None  # a 64-bit solve without this package would take minutes
    P, st = _inputs(case, seed)
    fixed, alpha = _dev(P.fixed), _face_alpha(P, st["rho"])
    if kind == "apply":
        return _operator(dim, n, fixed, alpha, st["x"])
    if kind == "solve":  # dense solve of the lifted system
        xd = _dev(P.dirichlet)
        fx = fixed.double()
        A = torch.cat([_operator(dim, n, fixed, alpha, c) for c in
                       torch.eye(xd.numel(), dtype=torch.float64, device=xd.device).split(512)]).T
        lift = _operator(dim, n, fixed, torch.zeros_like(alpha), xd * fx, masked=False)
        return torch.linalg.solve(A, fx * xd - (1 - fx) * lift)
    x, lam, rho = st["x"], st["lam"], st["rho"]
    nc = n ** dim
    gx = _operator(dim, n, fixed, alpha, x, objective=True)
    a = P.alpha
    dalpha = a.scale * (a.alpha_min - a.alpha_max) * (1 + a.q) * a.q / (rho + a.q) ** 2  # power 1
    e = _split(dim, n, (0.5 * x * x - x * lam) * (1 - fixed.double()))
    s = sum(e[1 + d] + _shift(e[1 + d], d, 1, dim) for d in range(dim))
    dj = 0.5 * dalpha * s[tuple(slice(0, n) for _ in range(dim))].reshape(-1)
    dc = _filter(dim, n, case["radius"], dj, True)
    dv = _filter(dim, n, case["radius"], torch.full_like(rho, 1.0 / nc), True)
    base = torch.clamp(-dc / dv, min=0.0) ** 0.5
    low, high = torch.clamp(rho - 0.2, min=1e-3), torch.clamp(rho + 0.2, max=1.0)
    l1, l2 = 0.0, 1e9
    while l2 - l1 > 1e-15 * (l1 + l2):
        lm = 0.5 * (l1 + l2)
        if lm in (l1, l2):
            break
        vol = (torch.minimum(torch.maximum(rho * base / math.sqrt(lm), low), high) * dv).sum().item()
        l1, l2 = (lm, l2) if vol > case["volfrac"] else (l1, lm)
    new = torch.minimum(torch.maximum(rho * base / math.sqrt(0.5 * (l1 + l2)), low), high)
    return {"J": 0.5 * float((x * gx).sum()), "gx": gx.cpu().numpy(), "dj": dj.cpu().numpy(), "dc": dc.cpu().numpy(),
            "rho": new.cpu().numpy(), "change": float((new - rho).abs().max()),
            "rhof": _filter(dim, n, case["radius"], new, False).cpu().numpy()}
