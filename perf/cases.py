"""Performance cases of the Stokes hot path: what a user's program runs through
the public entry points of gale_amd, over the sizes and options it is used with.

Kinds of case:

apply     one operator of the Uzawa loop on device vectors (apply_K_moments,
          apply_K, apply_K_fp32, apply_G, apply_Gt): what every iteration of
          every solve is made of
setup     one linear execute up to the Schur right-hand side: the constitutive
          pass with yielding from the previous solution, the multigrid levels,
          GetRhs, and an application of the operator that was set up
solve     setup and Uzawa solve from a zero pressure
learned   the same with the learned Schur preconditioner
picard    the nonlinear execute of a Drucker-Prager lid, from a restart
step      the particle half of a time step from a restart: time step size, RK2
          advection, relocation, remap (with constant or Voronoi weights) and
          the particles read back for a checkpoint
batch     many independent sinkers in one launch
forward,  the learned preconditioner's network on a grid: one application, and
backward  the gradient of a training batch
"""
import math
import os

import numpy as np
import torch

import gale_amd as G

# The layers of the network as oracle and library define them: channels per
# grid level, two convolutions per level down and up.
LEVELS, CHAN = 5, (16, 32, 48, 64, 96)


def listed():
    return [
        # the smallest call: one operator apply on a test-sized mesh that no tile divides; the launches are what counts
        {"name": "apply_moments_17x15x13", "kind": "apply", "form": "moments", "dim": 3, "nx": 17, "ny": 15, "nz": 13,
         "ppc": 8},
        # the operator of every inner iteration at the size of the 96^3 random-viscosity workload
        {"name": "apply_moments_96", "kind": "apply", "form": "moments", "dim": 3, "nx": 96, "ny": 96, "nz": 96,
         "ppc": 16},
        # what every Picard iteration and time step of the 96^3 workload begins with
        {"name": "setup_yield_96", "kind": "setup", "dim": 3, "nx": 96, "ny": 96, "nz": 96, "ppc": 16},
        # the 2D sinker, the smallest whole solve
        {"name": "solve_sinker_32", "kind": "solve", "problem": "sinker", "dim": 2, "nx": 32, "ny": 32, "nz": 1,
         "ppc": 20, "mixed": False, "tol": 1e-6},
        # the 3D Rayleigh-Taylor solve of one time step, all in 64 bits
        {"name": "solve_rayleigh_taylor_48", "kind": "solve", "problem": "layers", "dim": 3, "nx": 48, "ny": 48,
         "nz": 48, "ppc": 20, "mixed": False, "tol": 1e-6},
        # the random-viscosity solve with the learned preconditioner, mixed precision and relaxed inner solves
        {"name": "learned_48", "kind": "learned", "dim": 3, "nx": 48, "ny": 48, "nz": 48, "ppc": 16, "tol": 1e-4},
        # the 2D extension of a plastic lid: nonlinear, with a free surface
        {"name": "picard_lithosphere_2d", "kind": "picard", "dim": 2, "nx": 64, "ny": 16, "nz": 1, "ppc": 40,
         "picard_tol": 1e-4},
        # the particle half of a 3D time step with a checkpoint, constant weights
        {"name": "step_45x50x47", "kind": "step", "dim": 3, "nx": 45, "ny": 50, "nz": 47, "ppc": 20,
         "weights": "constant"},
        # the same in 2D with the Voronoi weights that PCDVC models integrate with
        {"name": "step_voronoi_127x63", "kind": "step", "dim": 2, "nx": 127, "ny": 63, "nz": 1, "ppc": 25,
         "weights": "voronoi"},
        # a batch of sinkers of uneven mesh size, reference loop
        {"name": "batch_sinkers", "kind": "batch", "count": 32, "lo8": 2, "hi8": 6, "ppc": 20, "relaxed": False},
        # the learned preconditioner applied once per Uzawa iteration of the 96^3 workload
        {"name": "net_forward_96", "kind": "forward", "nx": 96, "ny": 96, "nz": 96, "batch": 1},
        # one training batch at the resolution the shipped network was trained at
        {"name": "net_backward_32", "kind": "backward", "nx": 32, "ny": 32, "nz": 32, "batch": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["apply", "apply", "apply", "setup", "solve", "picard", "step", "batch", "forward", "backward",
                       "learned"])
    if kind == "apply":
        form = rng.choice(["moments", "particles", "particles32", "gradient", "divergence"])
        dim = rng.choice([2, 3, 3])
        hi = 96 if dim == 3 else 600
        n = [_log(rng, 8, hi) for _ in range(dim)] + [1] * (3 - dim)
        return {"kind": kind, "form": form, "dim": dim, "nx": n[0], "ny": n[1], "nz": n[2], "ppc": rng.randint(4, 16)}
    if kind == "setup":
        dim = rng.choice([2, 3])
        q = [8 * _log(rng, 1, 8 if dim == 3 else 32) for _ in range(dim)] + [1] * (3 - dim)
        return {"kind": kind, "dim": dim, "nx": q[0], "ny": q[1], "nz": q[2], "ppc": rng.randint(4, 24)}
    if kind == "solve":
        dim = rng.choice([2, 3])
        if dim == 2:
            n = [rng.randint(8, 40), rng.randint(8, 40), 1]
            problem = "sinker"
        else:
            n = [8 * _log(rng, 1, 6) for _ in range(3)]
            problem = "layers"
        return {"kind": kind, "problem": problem, "dim": dim, "nx": n[0], "ny": n[1], "nz": n[2],
                "ppc": rng.randint(8, 24), "mixed": rng.random() < 0.5, "tol": rng.choice([1e-5, 1e-6])}
    if kind == "learned":
        n = [48, rng.choice([32, 48]), rng.choice([32, 48])]
        rng.shuffle(n)
        return {"kind": kind, "dim": 3, "nx": n[0], "ny": n[1], "nz": n[2], "ppc": rng.randint(4, 16), "tol": 1e-4}
    if kind == "picard":
        return {"kind": kind, "dim": 2, "nx": 8 * rng.randint(3, 8), "ny": 4 * rng.randint(2, 4), "nz": 1,
                "ppc": rng.randint(20, 40), "picard_tol": 1e-4}
    if kind == "step":
        dim = rng.choice([2, 3])
        w = rng.choice(["constant", "voronoi"])
        n = [_log(rng, 8, (48 if w == "constant" else 24) if dim == 3 else 160) for _ in range(dim)] + [1] * (3 - dim)
        return {"kind": kind, "dim": dim, "nx": n[0], "ny": n[1], "nz": n[2], "ppc": rng.randint(8, 20), "weights": w}
    if kind == "batch":
        return {"kind": kind, "count": _log(rng, 2, 32), "lo8": 2, "hi8": rng.randint(2, 6), "ppc": rng.randint(8, 20),
                "relaxed": rng.random() < 0.5}
    n = [16 * _log(rng, 1, 6 if kind == "forward" else 3) for _ in range(3)]
    most = 96 ** 3 if kind == "forward" else 8 * 32 ** 3
    return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2],
            "batch": rng.randint(1, max(1, min(8, most // (n[0] * n[1] * n[2]))))}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _gen(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(1000003 + int(seed))
    return g


def _res(case):
    return [case["nx"], case["ny"], case["nz"]][:case["dim"]]


def _box(case):
    """The unit box, or the 4 x 1 box of the lithosphere."""
    dim = case["dim"]
    return [0.0] * dim, ([4.0] + [1.0] * (dim - 1) if case["kind"] == "picard" else [1.0] * dim)


def _cells(case):
    """(E, dim) integer cell of every element, x fastest."""
    res = _res(case)
    e = torch.arange(int(np.prod(res)), device=_dev())
    out = []
    for r in res:
        out.append(e % r)
        e = e // r
    return torch.stack(out, 1)


def _points(case, g):
    """(E, ppc, dim) points, uniform in every cell of the box, cell after cell
    as the reference's random layout fills them."""
    res = torch.tensor(_res(case), dtype=torch.float64, device=_dev())
    lo, hi = (torch.tensor(v, dtype=torch.float64, device=_dev()) for v in _box(case))
    c = _cells(case).double()
    f = torch.rand((c.shape[0], case["ppc"], case["dim"]), generator=g, dtype=torch.float64, device=_dev())
    return lo + (c[:, None, :] + f.clamp(1e-6, 1 - 1e-6)) / res * (hi - lo)


def _field(x, g, decades):
    """A smooth random field of the points x in [-decades/2, decades/2]:
    log10 of the viscosity of the random-viscosity workload."""
    dim = x.shape[-1]
    k = torch.randint(1, 6, (12, dim), generator=g, device=x.device).double()
    ph = 2 * math.pi * torch.rand(12, generator=g, dtype=torch.float64, device=x.device)
    v = torch.zeros(x.shape[:-1], dtype=torch.float64, device=x.device)
    for m in range(12):
        a = torch.full_like(v, float(ph[m]))
        for d in range(dim):
            a += math.pi * float(k[m, d]) * x[..., d]
        v += torch.cos(a)
    return v * (0.5 * decades / v.abs().max())


def _pad3(x):
    """(P, 3) host coordinates as the swarm keeps them."""
    x = x.reshape(-1, x.shape[-1])
    if x.shape[1] < 3:
        x = torch.cat([x, torch.zeros((x.shape[0], 3 - x.shape[1]), dtype=x.dtype, device=x.device)], 1)
    return x.cpu().numpy()


def _nodes(case):
    """(N, dim) node positions, x fastest."""
    res = _res(case)
    lo, hi = _box(case)
    ax = [torch.linspace(0.0, 1.0, r + 1, dtype=torch.float64, device=_dev()) * (h - l) + l
          for r, l, h in zip(res, lo, hi)]
    grid = torch.meshgrid(*ax[::-1], indexing="ij")
    return torch.stack([grid[case["dim"] - 1 - d].reshape(-1) for d in range(case["dim"])], 1)


def _roll(x, amplitude):
    """A convection roll with no flow through the walls of the unit box."""
    u = torch.zeros_like(x)
    u[:, 0] = amplitude * torch.sin(math.pi * x[:, 0]) * torch.cos(math.pi * x[:, 1])
    u[:, 1] = -amplitude * torch.cos(math.pi * x[:, 0]) * torch.sin(math.pi * x[:, 1])
    if x.shape[1] == 3:
        u[:, 2] = 0.5 * amplitude * torch.sin(math.pi * x[:, 2]) * torch.sin(2 * math.pi * x[:, 0])
    return u


LID = dict(eta0=1e2, density=0.0, yield_type=G.YIELD_DRUCKER_PRAGER, cohesion=1e-2,
           friction=math.tan(math.radians(30.0)), min_viscosity=1e-3)
CLAMP = (1e-3, 1e3)


def _lid_problem(case, g):
    """The random-viscosity workload: smooth six-decade viscosity, a plastic
    lid on top, a dense sphere, free slip.  Returns problem arguments and the
    device copies that exact() needs."""
    dim = case["dim"]
    x = _points(case, g)
    eta = 10.0 ** _field(x, g, 6.0)
    mat = torch.zeros(x.shape[:-1], dtype=torch.int32, device=x.device)
    mat[x[..., 1] >= 0.75] = 1
    mat[((x - 0.5) ** 2).sum(-1) <= 0.15 ** 2] = 2
    eta = torch.where(mat == 1, torch.full_like(eta, 1e2), eta)
    mask, vals = G.free_slip(dim, _res(case))
    mats = [G.material(eta0=1.0), G.material(**LID), G.material(eta0=1.0, density=1.0)]
    lo, hi = _box(case)
    kw = dict(dim=dim, res=_res(case), lo=lo, hi=hi, coord=_pad3(x), material_index=mat.reshape(-1).cpu().numpy(),
              materials=mats, bc_mask=mask, bc_value=vals, gravity=1.0, eta_clamp=CLAMP,
              eta0_particle=eta.reshape(-1).cpu().numpy())
    return kw, x, eta, mat


def _flow(case, kind):
    """Previous velocity (N*dim, host) and pressure (E, host) of a restart."""
    x = _nodes(case)
    if kind == "extension":
        u = torch.zeros_like(x)
        u[:, 0] = 0.5 * (x[:, 0] - 2.0)
        u[:, 1] = -0.5 * x[:, 1]
    else:
        u = _roll(x, 0.1)
    res = _res(case)
    c = _cells(case)[:, 1].double()
    p = 0.01 * (1.0 - (c + 0.5) / res[1])
    return u.reshape(-1), p


def _apply_inputs(case, g):
    x = _points(case, g)
    eta = 10.0 ** _field(x, g, 6.0)
    N = G.num_nodes(case["dim"], _res(case))
    if case["form"] == "gradient":
        v = torch.randn(x.shape[0], generator=g, dtype=torch.float64, device=_dev())
    else:
        v = torch.randn(N * case["dim"], generator=g, dtype=torch.float64, device=_dev())
    if case["form"] == "particles32":
        v = v.float()
    return x, eta, v


def _sinker_arrays(case, g):
    """Dense disc or two layers; returns points, material index and materials."""
    x = _points(case, g)
    mat = torch.zeros(x.shape[:-1], dtype=torch.int32, device=x.device)
    r = torch.rand(8, generator=g, dtype=torch.float64, device=x.device)
    if case["problem"] == "sinker":
        c = 0.4 + 0.2 * r[:2]
        mat[((x - c) ** 2).sum(-1) <= 0.15 ** 2] = 1
        return x, mat, [G.material(eta0=1.0, density=1.0), G.material(eta0=1e3, density=1.1)]
    y0 = torch.full_like(x[..., 0], 0.5)
    for m in range(4):
        y0 += 0.005 * torch.cos(2 * math.pi * (0.5 * (m + 1) * x[..., 0] + 0.5 * (4 - m) * x[..., 2] + float(r[m])))
    mat[x[..., 1] < y0] = 1
    return x, mat, [G.material(eta0=1e2, density=1.0), G.material(eta0=1.0, density=0.0)]


def _batch_problems(case, seed):
    rng = np.random.default_rng(7 + int(seed))
    out = []
    for i in range(case["count"]):
        # mesh sizes span the range evenly; the seed places discs and particles
        q = case["lo8"] + i % (case["hi8"] - case["lo8"] + 1)
        sub = dict(kind="batch", problem="sinker", dim=2, nx=8 * q, ny=8 * q, nz=1, ppc=case["ppc"])
        x = rng.random((8 * q, 8 * q, case["ppc"], 2)).clip(1e-6, 1 - 1e-6)
        x[..., 0] += np.arange(8 * q)[None, :, None]
        x[..., 1] += np.arange(8 * q)[:, None, None]
        x = x.reshape(-1, 2) / (8 * q)
        mat = np.zeros(len(x), np.int32)
        mats = [G.material(eta0=1.0, density=1.0)]
        for k in range(int(rng.integers(1, 6))):
            rad = rng.uniform(0.05, 0.15)
            c = rng.uniform(rad, 1 - rad, 2)
            mat[((x - c) ** 2).sum(1) <= rad * rad] = k + 1
            mats.append(G.material(eta0=10.0 ** rng.uniform(-2, 4), density=1.0 + rng.uniform(0.05, 0.2)))
        mask, vals = G.free_slip(2, _res(sub))
        coord = np.zeros((len(x), 3))
        coord[:, :2] = x
        out.append(dict(dim=2, res=_res(sub), lo=[0.0, 0.0], hi=[1.0, 1.0], coord=coord, material_index=mat,
                        materials=mats, bc_mask=mask, bc_value=vals))
    return out


def _weights():
    return np.load(os.path.join(os.path.dirname(G.__file__), "lpc_weights.npy"), allow_pickle=False)


def _net_inputs(case, g):
    """A residual scaled to unit RMS and log10 of the viscosity over 3, per
    element, and a gradient of the loss."""
    B, n = case["batch"], (case["nz"], case["ny"], case["nx"])
    r = torch.randn((B,) + n, generator=g, dtype=torch.float64, device=_dev())
    ax = [(torch.arange(k, dtype=torch.float64, device=_dev()) + 0.5) / k for k in n]
    gz, gy, gx = torch.meshgrid(*ax, indexing="ij")
    pts = torch.stack([gx, gy, gz], -1)
    eta = torch.stack([_field(pts, g, 6.0) / 3.0 for _ in range(B)])
    # residuals are smooth with noise on top
    r = 0.5 * r + torch.stack([_field(pts, g, 2.0) for _ in range(B)])
    r = r / r.square().mean((1, 2, 3), keepdim=True).sqrt()
    inp = torch.stack([r, eta], -1).float().contiguous()
    go = torch.randn((B,) + n, generator=g, dtype=torch.float64, device=_dev()).float() / r[0].numel()
    return inp, go.contiguous()


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "apply":
        x, eta, v = _apply_inputs(case, g)
        lo, hi = _box(case)
        dim = case["dim"]
        mask, vals = G.free_slip(dim, _res(case))
        pb = G.Problem(dim, _res(case), lo, hi, _pad3(x), np.zeros(x.shape[0] * x.shape[1], np.int32),
                       [G.material(eta0=1.0)], bc_mask=mask, bc_value=vals,
                       eta0_particle=eta.reshape(-1).cpu().numpy())
        inner = G.INNER_MULTIGRID if case["form"] == "moments" else G.INNER_JACOBI
        s = G.Stokes_SLE_UzawaSolver(pb, G.uzawa_params(inner_preconditioner=inner))
        s.setup()
        out = torch.empty(x.shape[0] if case["form"] == "divergence" else pb.N * dim, dtype=v.dtype, device=v.device)
        return dict(case=case, pb=pb, s=s, v=v, out=out)
    if kind == "setup":
        kw, *_ = _lid_problem(case, g)
        u, p = _flow(case, "roll")
        pb = G.Problem(**kw)
        s = G.Stokes_SLE_UzawaSolver(pb, G.uzawa_params(tolerance=1e-6))
        v = torch.randn(pb.N * case["dim"], generator=g, dtype=torch.float64, device=_dev())
        return dict(case=case, pb=pb, s=s, u=u.cpu().numpy(), p=p.cpu().numpy(), v=v, out=torch.empty_like(v))
    if kind == "solve":
        x, mat, mats = _sinker_arrays(case, g)
        mask, vals = G.free_slip(case["dim"], _res(case))
        lo, hi = _box(case)
        pb = G.Problem(case["dim"], _res(case), lo, hi, _pad3(x), mat.reshape(-1).cpu().numpy(), mats, bc_mask=mask,
                       bc_value=vals)
        s = G.Stokes_SLE_UzawaSolver(pb, G.uzawa_params(
            tolerance=case["tol"], maxIterations=20000, precision=G.PREC_MIXED if case["mixed"] else G.PREC_FP64))
        return dict(case=case, pb=pb, s=s)
    if kind == "learned":
        kw, *_ = _lid_problem(case, g)
        pb = G.Problem(**kw)
        s = G.Stokes_SLE_UzawaSolver(pb, G.uzawa_params(tolerance=case["tol"], maxIterations=20000, learned=True,
                                                        precision=G.PREC_MIXED, inner_relax_max=0.1))
        net = G.LearnedPreconditioner()
        net.set_params(_weights())
        s.set_learned(net)
        return dict(case=case, pb=pb, s=s)
    if kind == "picard":
        x = _points(case, g)
        mat = torch.zeros(x.shape[:-1], dtype=torch.int32, device=x.device)
        mat[x[..., 1] >= 0.75] = 1
        mat[((x[..., 0] - 2.0).abs() <= 0.05) & ((x[..., 1] - 0.875).abs() <= 0.05)] = 2
        mask, vals = G.wall_bc(2, _res(case), [("left", 0, -1.0), ("right", 0, 1.0), ("bottom", 1, 0.0)])
        lo, hi = _box(case)
        pb = G.Problem(2, _res(case), lo, hi, _pad3(x), mat.reshape(-1).cpu().numpy(),
                       [G.material(eta0=1.0), G.material(**LID), G.material(eta0=1e-2)], bc_mask=mask, bc_value=vals,
                       gravity=0.0, eta_clamp=CLAMP)
        s = G.Stokes_SLE_UzawaSolver(pb, G.uzawa_params(tolerance=1e-6, maxIterations=20000))
        u, p = _flow(case, "extension")
        return dict(case=case, pb=pb, s=s, u=u.cpu().numpy(), p=p.cpu().numpy())
    if kind == "step":
        x = _points(case, g)
        lo, hi = _box(case)
        order = torch.randperm(x.shape[0] * x.shape[1], generator=g, device=x.device)  # after many steps
        coord = _pad3(x.reshape(-1, case["dim"])[order])
        pb = G.Problem(case["dim"], _res(case), lo, hi, coord, np.zeros(len(coord), np.int32), [G.material(eta0=1.0)])
        if case["weights"] == "voronoi":
            pb.set_weights(G.WEIGHTS_DVC)
        s = G.Stokes_SLE_UzawaSolver(pb, G.uzawa_params())
        u, p = _flow(case, "roll")
        return dict(case=case, pb=pb, s=s, coord=coord, u=u.cpu().numpy(), p=p.cpu().numpy())
    if kind == "batch":
        bs = G.BatchSolver(_batch_problems(case, seed))
        prm = (G.batch_params(tolerance=1e-6, inner_relax_max=0.03, flexible_window=8) if case["relaxed"]
               else G.batch_params(tolerance=1e-6))
        return dict(case=case, bs=bs, prm=prm)
    inp, go = _net_inputs(case, g)
    net = G.LearnedPreconditioner()
    net.set_params(_weights())
    return dict(case=case, net=net, inp=inp, go=go, out=torch.empty(inp.shape[:-1], device=inp.device))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "apply":
        s, v, out = state["s"], state["v"], state["out"]
        {"moments": s.apply_K_moments, "particles": s.apply_K, "particles32": s.apply_K_fp32,
         "gradient": s.apply_G, "divergence": s.apply_Gt}[case["form"]](v, out)
        return out
    if kind == "setup":
        s = state["s"]
        s.setup(state["u"], state["p"], yield_on=True)
        rhs = s.GetRhs()
        s.apply_K_moments(state["v"], state["out"])
        return {"y": state["out"], "rhs": rhs}
    if kind in ("solve", "learned"):
        s = state["s"]
        s.set_pressure(None)
        s.setup()
        u, p, _ = s.Solve()
        return {"u": u, "p": p}
    if kind == "picard":
        s = state["s"]
        s.set_solution(state["u"], state["p"])
        u, p, _ = s.NonLinearExecute(nonLinearTolerance=case["picard_tol"], nonLinearMaxIterations=20)
        return {"u": u, "p": p}
    if kind == "step":
        pb, s = state["pb"], state["s"]
        pb.set_coords(state["coord"])
        s.set_solution(state["u"], state["p"])
        dt = s.compute_dt()
        s.advect_rk2(dt)
        coord, owner, xi, w = pb.particles()
        return {"dt": dt, "coord": coord, "owner": owner, "xi": xi, "weight": w}
    if kind == "batch":
        bs = state["bs"]
        bs.solve(state["prm"])
        sol = [bs.solution(i) for i in range(bs.count)]
        return {"u": np.concatenate([u for u, _ in sol]), "p": np.concatenate([p for _, p in sol])}
    if kind == "forward":
        state["net"].forward(state["inp"], state["out"])
        return state["out"]
    state["net"].forward(state["inp"], state["out"])
    return {"out": state["out"], "grad": state["net"].backward(state["inp"], state["go"])}


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------
def _layers():
    """(cin, cout, level) of the network's convolutions, in parameter order."""
    out = []
    for lev in range(LEVELS):
        cin = 4 if lev == 0 else CHAN[lev - 1]
        out.append((cin, CHAN[lev], lev))
        out.append((CHAN[lev], CHAN[LEVELS - 2] if lev == LEVELS - 1 else CHAN[lev], lev))
    for lev in range(LEVELS - 2, -1, -1):
        out.append((CHAN[lev], CHAN[lev], lev))
        out.append((CHAN[lev], CHAN[lev - 1] if lev else 1, lev))
    return out


def work(case):
    kind = case["kind"]
    if kind in ("forward", "backward"):
        V = case["batch"] * case["nx"] * case["ny"] * case["nz"]
        fl = sum(2.0 * 27 * ci * co * V / 8 ** lev for ci, co, lev in _layers())
        w = 4.0 * sum(27 * ci * co + co for ci, co, _ in _layers())
        if kind == "forward":
            return {"bytes": 12.0 * V + w, "flops": fl}
        return {"bytes": 16.0 * V + 2 * w, "flops": 3 * fl}
    if kind == "batch":
        E = sum((8 * (case["lo8"] + i % (case["hi8"] - case["lo8"] + 1))) ** 2 for i in range(case["count"]))
        return {"bytes": E * (8.0 * 9 + 8 * 5 + 8 * 3), "flops": E * 150.0}
    dim = case["dim"]
    res = _res(case)
    E = float(np.prod(res))
    N = float(np.prod([r + 1 for r in res]))
    P = E * case["ppc"]
    mom = 27 if dim == 3 else 9
    per_el = 700.0 if dim == 3 else 110.0  # flops of one element from its moments
    if kind == "apply":
        form = case["form"]
        if form == "moments":
            return {"bytes": 16 * dim * N + 8 * mom * E, "flops": per_el * E}
        if form == "particles":
            return {"bytes": 16 * dim * N + 32 * P + 4 * E, "flops": (150.0 if dim == 3 else 50.0) * P}
        if form == "particles32":
            return {"bytes": 8 * dim * N + 16 * P + 4 * E, "flops": (150.0 if dim == 3 else 50.0) * P}
        return {"bytes": 8 * dim * N + 8 * E, "flops": 2.0 * dim * 2 ** dim * E}
    if kind == "step":
        # positions in and out (host and device), the sort's key and index, local coordinates and weights
        return {"bytes": P * (24 * 4 + 16 + 8 * dim + 8) + 8 * dim * N, "flops": 200.0 * P}
    # setup, solve and nonlinear execute: particles read, viscosity written, fields in and out once
    return {"bytes": P * (32 + 12 + 16) + 8 * mom * E + 8 * dim * N * 5 + 8 * E * 4, "flops": 250.0 * P + per_el * E}


def tolerance(case):
    """About four times what the path showed against exact(), or against itself
    with its sums in another order (other coarse levels, smoothing steps, tile
    shapes or matrix-core steps), whichever was larger."""
    kind = case["kind"]
    if kind == "apply":
        return {"rel": 3e-7 if case["form"] == "particles32" else 3e-14}
    if kind == "setup":
        return {"rel": 1e-6}  # the right-hand side is an inner solve to 1e-6
    if kind == "solve":
        return {"rel": 1.3e-3}  # what a Schur residual of 1e-5 to 1e-6 leaves open: 3e-4 seen
    if kind == "learned":
        return {"rel": 0.2}  # pressure of a six-decade problem to 1e-4: 5e-2 seen
    if kind == "picard":
        return {"rel": 1e-5}
    if kind == "step":
        return {"rel": 6e-14}
    if kind == "batch":
        return {"rel": 1.2e-4}
    if kind == "forward":
        return {"rel": 1.7e-2}
    return {"rel": 0.1}  # gradients through BF16 activations, whose ReLUs flip: 2.4e-2 seen


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------
def _corner_nodes(case):
    """(E, 2^dim) nodes of every element, x fastest."""
    res, dim = _res(case), case["dim"]
    c = _cells(case)
    nn = [r + 1 for r in res]
    out = []
    for a in range(2 ** dim):
        idx = torch.zeros(c.shape[0], dtype=torch.int64, device=c.device)
        stride = 1
        for d in range(dim):
            idx += (c[:, d] + ((a >> d) & 1)) * stride
            stride *= nn[d]
        out.append(idx)
    return torch.stack(out, 1)


def _spacing(case):
    lo, hi = _box(case)
    return [(h - l) / r for l, h, r in zip(lo, hi, _res(case))]


def _shape_grad(case, cells, x):
    """dN/dx of the corner functions at the points x (E', ppc, dim) of the given cells: (E', ppc, 2^dim, dim)."""
    dim, h = case["dim"], torch.tensor(_spacing(case), dtype=torch.float64, device=x.device)
    lo = torch.tensor(_box(case)[0], dtype=torch.float64, device=x.device)
    xi = 2.0 * ((x - lo) / h - cells[:, None, :].double()) - 1.0
    out = []
    for a in range(2 ** dim):
        s = [1.0 if (a >> d) & 1 else -1.0 for d in range(dim)]
        g = []
        for d in range(dim):
            v = torch.full_like(xi[..., 0], s[d] / 2 ** dim * 2.0) / h[d]
            for d2 in range(dim):
                if d2 != d:
                    v = v * (1.0 + s[d2] * xi[..., d2])
            g.append(v)
        out.append(torch.stack(g, -1))
    return torch.stack(out, -2)


def _exact_K(case, x, eta, v):
    """K v integrated point by point: sum_p w detJ B^T (2 eta) B, no boundary conditions."""
    dim = case["dim"]
    nodes, cells = _corner_nodes(case), _cells(case)
    vol = float(np.prod(_spacing(case)))
    v = v.double().reshape(-1, dim)
    y = torch.zeros_like(v)
    step = max(1, (1 << 19) // case["ppc"])
    for e0 in range(0, x.shape[0], step):
        sl = slice(e0, min(e0 + step, x.shape[0]))
        dN = _shape_grad(case, cells[sl], x[sl])  # e p a j
        ue = v[nodes[sl]]  # e a i
        L = (ue[:, None, :, :, None] * dN[..., None, :]).sum(2)  # e p i j
        sig = (vol / case["ppc"]) * eta[sl][..., None, None] * (L + L.transpose(-1, -2))
        f = (sig[:, :, None] * dN[..., None, :]).sum(-1).sum(1)  # e a i
        y.index_add_(0, nodes[sl].reshape(-1), f.reshape(-1, dim))
    return y.reshape(-1)


def _face_signs(case):
    """G_e[a, d] = -s_ad (product of the other spacings) / 2^(dim-1)."""
    dim, h = case["dim"], _spacing(case)
    out = torch.zeros((2 ** dim, dim), dtype=torch.float64, device=_dev())
    for a in range(2 ** dim):
        for d in range(dim):
            area = np.prod([h[k] for k in range(dim) if k != d])
            out[a, d] = -(1.0 if (a >> d) & 1 else -1.0) * area / 2 ** (dim - 1)
    return out


def _yielded(case, x, eta, mat, u, p):
    """Viscosity of every point after the Drucker-Prager lid yields from u, p, and the clamp."""
    dim = case["dim"]
    nodes, cells = _corner_nodes(case), _cells(case)
    u = u.reshape(-1, dim)
    out = torch.empty_like(eta)
    mu = LID["friction"]
    cphi = 1 / math.sqrt(1 + mu * mu)
    k = cphi if dim == 2 else 2 * cphi / (math.sqrt(3.0) * (3 - mu * cphi))
    step = max(1, (1 << 19) // case["ppc"])
    for e0 in range(0, x.shape[0], step):
        sl = slice(e0, min(e0 + step, x.shape[0]))
        dN = _shape_grad(case, cells[sl], x[sl])
        L = (u[nodes[sl]][:, None, :, :, None] * dN[..., None, :]).sum(2)
        sr = 0.5 * (L + L.transpose(-1, -2))
        tr = sr.diagonal(dim1=-2, dim2=-1).sum(-1) / dim
        sr = sr - tr[..., None, None] * torch.eye(dim, dtype=sr.dtype, device=sr.device)
        srII = (0.5 * sr.square().sum((-1, -2))).sqrt()
        fs = mu * k * p[sl][:, None] + LID["cohesion"] * k * (1 if dim == 2 else 3)
        fs = torch.clamp(fs, min=LID["cohesion"] * k).expand_as(srII)
        e = eta[sl]
        yields = (mat[sl] == 1) & (fs < 2 * e * srII)
        e = torch.where(yields, torch.clamp(fs / (2 * srII), min=LID["min_viscosity"]), e)
        out[sl] = e.clamp(*CLAMP)
    return out


def _exact_solve(case, x, mat, mats):
    """Velocity of the saddle problem by dense elimination (2D, small)."""
    dim, dev = case["dim"], x.device
    nodes, cells = _corner_nodes(case), _cells(case)
    vol = float(np.prod(_spacing(case)))
    eta = torch.tensor([m["eta0"] for m in mats], dtype=torch.float64, device=dev)[mat.long()]
    rho = torch.tensor([m["density"] for m in mats], dtype=torch.float64, device=dev)[mat.long()]
    N, E, nen = G.num_nodes(dim, _res(case)), x.shape[0], 2 ** dim
    dN = _shape_grad(case, cells, x)
    w = vol / case["ppc"] * eta
    K = torch.zeros((N * dim, N * dim), dtype=torch.float64, device=dev)
    dof = (nodes[:, :, None] * dim + torch.arange(dim, device=dev)).reshape(E, -1)
    ke = torch.zeros((E, nen, dim, nen, dim), dtype=torch.float64, device=dev)
    for a in range(nen):
        for b in range(nen):
            gg = (w * (dN[:, :, a] * dN[:, :, b]).sum(-1)).sum(1)
            for i in range(dim):
                ke[:, a, i, b, i] += gg
                for j in range(dim):
                    # sigma_ij contributes dN_a,j (du_i/dx_j + du_j/dx_i)
                    ke[:, a, i, b, j] += (w * dN[:, :, a, j] * dN[:, :, b, i]).sum(1)
    ke = ke.reshape(E, nen * dim, nen * dim)
    K.reshape(-1).index_add_(0, (dof[:, :, None] * (N * dim) + dof[:, None, :]).reshape(-1), ke.reshape(-1))
    # shape functions of the points for the body force (0, -1) rho
    lo = torch.tensor(_box(case)[0], dtype=torch.float64, device=dev)
    h = torch.tensor(_spacing(case), dtype=torch.float64, device=dev)
    xi = 2.0 * ((x - lo) / h - cells[:, None, :].double()) - 1.0
    f = torch.zeros(N * dim, dtype=torch.float64, device=dev)
    for a in range(nen):
        n = torch.full_like(xi[..., 0], 1.0 / nen)
        for d in range(dim):
            n = n * (1.0 + (1.0 if (a >> d) & 1 else -1.0) * xi[..., d])
        f.index_add_(0, nodes[:, a] * dim + 1, -(vol / case["ppc"] * rho * n).sum(1))
    Gm = torch.zeros((N * dim, E), dtype=torch.float64, device=dev)
    sg = _face_signs(case).reshape(-1)
    Gm[dof, torch.arange(E, device=dev)[:, None]] = sg.expand(E, -1)
    mask, _ = G.free_slip(dim, _res(case))
    free = torch.from_numpy(np.flatnonzero(mask == 0)).to(dev)
    K, f, Gm = (t.cpu().numpy() for t in (K[free][:, free], f[free], Gm[free]))
    X = np.linalg.solve(K, np.concatenate([f[:, None], Gm], 1))
    S = Gm.T @ X[:, 1:]
    S = S + np.mean(np.diag(S)) / E  # the constant pressure is in its null space and orthogonal to the right side
    p = np.linalg.solve(S, Gm.T @ X[:, 0])
    u = np.zeros(N * dim)
    u[free.cpu().numpy()] = X[:, 0] - X[:, 1:] @ p
    return u


def _exact_step(case, coord, u):
    """RK2 positions, owners, local coordinates and constant weights."""
    dim, res = case["dim"], _res(case)
    r = torch.tensor(res, dtype=torch.float64, device=_dev())
    x0 = torch.from_numpy(coord[:, :dim]).to(_dev())  # the unit box
    U = u.reshape(-1, dim).to(_dev())
    nn = [k + 1 for k in res]
    vmax = U.square().sum(1).max().sqrt()
    dt = 0.5 * (1.0 / max(res)) / vmax

    def where(x):
        t = x * r
        c = torch.minimum(t.floor(), r - 1)
        return c, 2.0 * (t - c) - 1.0

    def vel(x):
        c, xi = where(x)
        v = torch.zeros_like(x)
        for a in range(2 ** dim):
            n = torch.full_like(x[:, 0], 1.0 / 2 ** dim)
            idx = torch.zeros(len(x), dtype=torch.int64, device=x.device)
            stride = 1
            for d in range(dim):
                b = (a >> d) & 1
                n = n * (1.0 + (1.0 if b else -1.0) * xi[:, d])
                idx += (c[:, d].long() + b) * stride
                stride *= nn[d]
            v += n[:, None] * U[idx]
        return v

    x1 = x0 + dt * vel(x0 + 0.5 * dt * vel(x0))
    c, xi = where(x1)
    owner = torch.zeros(len(x1), dtype=torch.int64, device=x1.device)
    stride = 1
    for d in range(dim):
        owner += c[:, d].long() * stride
        stride *= res[d]
    cnt = torch.bincount(owner, minlength=stride)
    out = coord.copy()
    out[:, :dim] = x1.cpu().numpy()
    return {"dt": float(dt), "coord": out, "owner": owner.int().cpu().numpy(), "xi": xi.cpu().numpy(),
            "weight": (2.0 ** dim / cnt[owner].double()).cpu().numpy()}


def _exact_net(case, params, inp):
    """The network's output in 64 bits from its FP32 parameters."""
    B, n = case["batch"], (case["nz"], case["ny"], case["nx"])
    pos = [0]

    def conv(x, cin, cout, relu):
        W = params[pos[0]:pos[0] + 27 * cin * cout].reshape(27, cin, cout)
        b = params[pos[0] + 27 * cin * cout:pos[0] + 27 * cin * cout + cout]
        pos[0] += 27 * cin * cout + cout
        m = x.shape[1:4]
        xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        y = b.expand(x.shape[:4] + (cout,))
        for t in range(27):
            dx, dy, dz = t % 3, (t // 3) % 3, t // 9
            y = y + (xp[:, dz:dz + m[0], dy:dy + m[1], dx:dx + m[2]].reshape(-1, cin) @ W[t]).reshape(y.shape)
        return torch.relu(y) if relu else y

    x = torch.cat([inp.double(), torch.zeros((B,) + n + (2,), dtype=torch.float64, device=inp.device)], -1)
    L = _layers()
    skip = []
    for lev in range(LEVELS):
        if lev:
            s = x.shape
            x = x.reshape(s[0], s[1] // 2, 2, s[2] // 2, 2, s[3] // 2, 2, s[4]).mean((2, 4, 6))
        x = conv(x, L[2 * lev][0], L[2 * lev][1], True)
        x = conv(x, L[2 * lev + 1][0], L[2 * lev + 1][1], True)
        skip.append(x)
    for i, lev in enumerate(range(LEVELS - 2, -1, -1)):
        x = x.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3) + skip[lev]
        a, b = L[2 * LEVELS + 2 * i], L[2 * LEVELS + 2 * i + 1]
        x = conv(x, a[0], a[1], True)
        x = conv(x, b[0], b[1], lev > 0)
    return x[..., 0]


def exact(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    dim = case.get("dim")
    if kind == "apply":
        x, eta, v = _apply_inputs(case, g)
        if case["form"] in ("gradient", "divergence"):
            nodes, sg = _corner_nodes(case), _face_signs(case)
            if case["form"] == "divergence":
                return (v.reshape(-1, dim)[nodes] * sg).sum((1, 2))
            y = torch.zeros((G.num_nodes(dim, _res(case)), dim), dtype=torch.float64, device=v.device)
            y.index_add_(0, nodes.reshape(-1), (v[:, None, None] * sg).reshape(-1, dim))
            return y.reshape(-1)
        return _exact_K(case, x, eta, v)
    if kind == "setup":
        _, x, eta, mat = _lid_problem(case, g)
        u, p = _flow(case, "roll")
        v = torch.randn(u.numel(), generator=g, dtype=torch.float64, device=_dev())
        return {"y": _exact_K(case, x, _yielded(case, x, eta, mat, u, p), v), "rhs": None}
    if kind == "solve" and dim == 2 and case["nx"] * case["ny"] <= 1100:
        return {"u": _exact_solve(case, *_sinker_arrays(case, g)), "p": None}
    if kind == "step" and case["weights"] == "constant":
        x = _points(case, g)
        order = torch.randperm(x.shape[0] * x.shape[1], generator=g, device=x.device)
        return _exact_step(case, _pad3(x.reshape(-1, dim)[order]), _flow(case, "roll")[0])
    if kind in ("forward", "backward"):
        inp, go = _net_inputs(case, g)
        prm = torch.from_numpy(_weights()).to(inp.device).double()
        if kind == "forward":
            return _exact_net(case, prm, inp)
        prm.requires_grad_(True)
        out = _exact_net(case, prm, inp)
        out.backward(go.double())
        return {"out": out.detach(), "grad": prm.grad}
    return None
