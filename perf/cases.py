"""The work that users of this package have it do, as measurable cases.

Kinds of case (`case["kind"]`), each through public entry points:

* "solve":   one streamfunction solve at the drop-in boundary, as a driver
             that keeps the energy equation on the host makes it in every RK
             stage: T and the warm start go in, smoother_time_T, multigrid and
             compute_velocities run, SF, u and w come back.
* "step":    one whole time step (RK4, RK_update=1) with the state on the
             device, and the grid fields read back as a snapshot reads them
             (with the tracer positions where they are few).
* "tracers": the tracer part of a step in a flow that stays as it is: four RK
             stages, each with the tracer-ratio binning, the C filter and the
             conductivity.
* "bin":     the binning alone on the caller's device buffers.
* "ensemble": one step of several independent cases run concurrently.
* "net":     one training step of the learned initial guess: sample in,
             forward, backward, Adam, prediction, gradients and weights out.

Sizes and physics are those of the package's presets (config.PRESETS), of its
ensemble distribution (ensemble.draw_cases) and of its tests.
"""
import ctypes
import math

import numpy as np
import torch

from tracer_code_amd import Solver, _abi, config, ensemble, ic, learn
from tracer_code_amd.model import library

# tracers of a step case whose positions come back with the fields
TRACERS_BACK = 2_000_000
# defect-correction settings of a tuned program: sweeps per visit on level 1,
# on level 2 and below, with the widened level-1 Chebyshev interval and GCR
TUNED = dict(common=20, level2=16, coarse=8, la=-0.25, gcr=16, refresh=4)


def listed():
    return [
        # the 128x128 preset in the reference's own FP64 form, the library's
        # default mode: the smallest grid that a study starts from
        dict(name="solve_fp64_128x128", kind="solve", mode="fp64", preset="cfg0", nx=128, nz=128, tol=1e-8),
        # a grid whose spacings are no powers of two, FP64 form
        dict(name="solve_fp64_608x352", kind="solve", mode="fp64", preset="drawn", nx=608, nz=352, visT=1e3, tol=1e-7),
        # the largest preset in the FP64 form, at the smallest tolerance it reaches there
        dict(name="solve_fp64_2048x1024", kind="solve", mode="fp64", preset="cfg2", nx=2048, nz=1024, tol=1e-7),
        # defect correction with FP64 corrections, untuned
        dict(name="solve_dc64_512x256", kind="solve", mode="dc64", preset="drawn", nx=512, nz=256, visT=1e4, tol=1e-8),
        # a whole step of the smallest preset, FP64 form
        dict(name="step_fp64_128x128", kind="step", mode="fp64", preset="cfg0", nx=128, nz=128, tpc=20, tol=1e-8),
        # mixed mode as it comes (no tuning call), a small ragged grid, two
        # composition types
        dict(name="step_mixed_152x104", kind="step", mode="mixed", preset="two", nx=152, nz=104, tpc=16, tol=1e-8),
        # the middle preset, mixed mode, tuned
        dict(name="step_mixed_768x256", kind="step", mode="mixed", preset="cfg1", nx=768, nz=256, tpc=40, tol=1e-8,
             tuned=True),
        # the largest preset with its 42M tracers, mixed mode, tuned: the benchmark's workload
        dict(name="step_mixed_2048x1024", kind="step", mode="mixed", preset="cfg2", nx=2048, nz=1024, tpc=20, tol=1e-8,
             tuned=True, sort=20),
        # tracers, binning and C filter of an ordinary grid
        dict(name="tracers_1024x512", kind="tracers", mode="mixed", preset="drawn", nx=1024, nz=512, visT=1e3, tpc=20,
             sort=0),
        # binning on the caller's buffers, tracers in creation order
        dict(name="bin_1024x512x40", kind="bin", nx=1024, nz=512, ntype=2, tpc=40, order="created"),
        # six cases over the ensemble's grids, mixed mode, tuned
        dict(name="ensemble_mixed_6", kind="ensemble", mode="mixed", cases=6, scale=1, tpc=12, tol=1e-8),
        # a training step of the network of the 768x256 preset (its multigrid level 4)
        dict(name="net_train_32x96", kind="net", H=32, W=96),
    ]


def draw(rng):
    def size(lo, hi, mult):
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / mult))
        return max(1, n) * mult

    def grid(lo, hi):
        # six-level grids above 256 nodes a side, ragged ones below
        nx = size(lo, hi, 32 if hi > 256 else 8)
        nz = min(max(size(max(lo, nx // 4), max(lo, nx), 32 if hi > 256 else 8), 32), 1024)
        return nx, nz

    kind = rng.choice(("solve", "solve", "solve", "step", "step", "step", "tracers", "bin", "ensemble", "net"))
    if kind == "solve":
        mode = rng.choice(("fp64", "fp64", "dc64", "mixed"))
        nx, nz = grid(64, 256) if rng.random() < 0.5 else grid(256, 1024)
        return dict(kind=kind, mode=mode, preset="drawn", nx=nx, nz=nz, visT=round(10.0 ** rng.uniform(2, 3.5), 1),
                    tol=1e-7 if mode == "fp64" else 1e-8, tuned=mode == "mixed" and rng.random() < 0.5)
    if kind == "step":
        mode = rng.choice(("fp64", "mixed", "mixed", "dc64"))
        nx, nz = grid(64, 256) if mode == "fp64" or rng.random() < 0.6 else grid(256, 768)
        return dict(kind=kind, mode=mode, preset="drawn", nx=nx, nz=nz, visT=round(10.0 ** rng.uniform(2, 3.5), 1),
                    tol=1e-7 if mode == "fp64" else 1e-8, tpc=rng.randint(10, 40), tuned=mode == "mixed" and rng.random() < 0.6,
                    sort=rng.choice((0, 0, 5)))
    if kind == "tracers":
        nx, nz = grid(96, 1024)
        return dict(kind=kind, mode="mixed", preset=rng.choice(("drawn", "two")), nx=nx, nz=nz, visT=1e3, tpc=rng.randint(8, 40),
                    sort=rng.choice((0, 10)))
    if kind == "bin":
        return dict(kind=kind, nx=rng.randint(33, 1200), nz=rng.randint(33, 700), ntype=rng.randint(1, 4),
                    tpc=rng.randint(5, 40), order=rng.choice(("created", "rows", "mixed")))
    if kind == "ensemble":
        return dict(kind=kind, mode="mixed", cases=rng.randint(2, 5), scale=rng.choice((1, 2, 4)), tpc=rng.randint(6, 12),
                    tol=1e-8)
    return dict(kind=kind, H=16 * rng.randint(1, 8), W=16 * rng.randint(1, 16))


# ---- inputs ------------------------------------------------------------------
def _physics(case):
    """Parameters of config.make_params plus the keys of the initial fields."""
    p = case["preset"]
    size = dict(nx=case["nx"], nz=case["nz"])
    if p in config.PRESETS:
        cfg = dict(config.PRESETS[p], **size)
        if p == "cfg1":
            # the reference's unzeroed coarse corrections diverge at this contrast
            cfg["fixes"] = 1
    else:
        # the middle of the ensemble's distribution
        ra = 1e6
        cfg = dict(aspect=case["nx"] / case["nz"], RaT=ra, RaC=(0.5 * ra,), ivis=2, visT=case.get("visT", 1e3),
                   visC=(1.0 / 30.0,), tpc=10, dlayer=0.15, initial_comp=0, t_variant="fourier4", fixes=1,
                   delta_visC=(1.2,), **size)
        if p == "two":
            cfg.update(ntype=2, RaC=(0.5 * ra, 0.25 * ra), visC=(1.0 / 10.0, 1.0 / 3.0), delta_visC=(1.5, 1.5),
                       conduct_factor=(1.0, 2.0))
    cfg["tpc"] = case.get("tpc", 8)
    if "tol" in case:
        cfg["tolerance"] = case["tol"]
    return cfg


def _solver(case, cfg, seed):
    params = config.make_params(**cfg)
    cfg = dict(cfg, nx=params.nx, nz=params.nz)
    T, r, s, ty = ic.workload(cfg, seed=seed)
    if params.ntype == 2:
        # a second, shallower layer above the first
        ty = np.where((ty == 0) & (s < 0.4), 2, ty).astype(np.int32)
    g = Solver(params, len(r))
    g.set_mode(case.get("mode", "fp64"))
    g.initialize(T, r, s, ty)
    if case.get("tuned"):
        _tune(g, params, case)
    if case.get("sort"):
        g.set_tracer_sort(case["sort"])
    return g, T


def _tune(g, params, case):
    common = 10 if case.get("preset") == "cfg2" else TUNED["common"]
    g.guess_enable("extrap")
    g.set_gcr(TUNED["gcr"])
    g.set_coarse_refresh(TUNED["refresh"])
    g.set_dc_cheb_interval(-2.0, TUNED["la"])
    g.set_dc_sweeps(common)
    for L in range(2, params.grids):
        g.set_dc_level_sweeps(L, TUNED["level2"] if L == 2 else TUNED["coarse"])


def _bin_inputs(case, seed):
    nx, nz = case["nx"], case["nz"]
    aspect = nx / nz
    n = (nx + 1) * (nz + 1) * case["tpc"]
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    node = torch.arange(n, device="cuda") // case["tpc"]
    if case["order"] == "rows":
        i, k = node % (nx + 1), node // (nx + 1)
    else:
        i, k = node // (nz + 1), node % (nz + 1)
    dr, ds = aspect / nx, 1.0 / nz
    # jitter over the node's own cell; "mixed": tracers that have moved up to two cells
    amp = 4.0 if case["order"] == "mixed" else 1.0
    u = torch.rand(n, device="cuda", dtype=torch.float64, generator=gen) - 0.5
    v = torch.rand(n, device="cuda", dtype=torch.float64, generator=gen) - 0.5
    r = (i * dr + amp * u * dr).clamp(1e-4 * dr, aspect - 1e-4 * dr)
    s = (k * ds + amp * v * ds).clamp(1e-4 * ds, 1.0 - 1e-4 * ds)
    # layers by depth, with a smooth boundary
    ty = ((1.0 - s + 0.02 * torch.cos(math.pi * r / aspect)) * (case["ntype"] + 1)).to(torch.int32).clamp(0, case["ntype"])
    return r, s, ty, aspect


def _net_inputs(case, seed):
    rng = np.random.default_rng(int(seed))
    H, W = case["H"], case["W"]
    kz, kx = np.meshgrid(np.arange(H) / H, np.arange(W) / W, indexing="ij")
    x = np.empty((H, W, 6), dtype=np.float32)
    for c in range(6):
        f = sum(rng.normal() * np.cos(math.pi * (a * kx + b * kz) + rng.uniform(0, 6)) for a in range(1, 4)
                for b in range(1, 4))
        x[:, :, c] = f / 4.0
    t = (0.3 * np.tanh(x[:, :, 1] + x[:, :, 4]) + 0.05 * rng.normal(size=(H, W))).astype(np.float32)
    m = np.ones((H, W), dtype=np.float32)
    m[0, :] = 0
    m[:, 0] = 0
    w = learn.init_weights(int(seed) % 100003)
    w[-17:-1] = rng.normal(size=16) * 0.25   # a head that has left its zero start
    return x, t, m, w


def prepare(case, seed):
    kind = case["kind"]
    if kind == "net":
        x, t, m, w = _net_inputs(case, seed)
        net = learn.Network(case["H"], case["W"])
        net.set_weights(w)
        return dict(kind=kind, net=net, x=x, t=t, m=m)
    if kind == "bin":
        r, s, ty, aspect = _bin_inputs(case, seed)
        nx, nz, nt = case["nx"], case["nz"], case["ntype"]
        plane = (nz + 5, nx + 5)
        return dict(kind=kind, case=case, aspect=aspect, r=r, s=s, ty=ty, lib=library(),
                    count=torch.empty((nt + 1,) + plane, dtype=torch.int32, device="cuda"),
                    nempty=torch.empty(plane, dtype=torch.int32, device="cuda"),
                    C=torch.zeros((nt,) + plane, dtype=torch.float64, device="cuda"))
    if kind == "ensemble":
        rng = np.random.default_rng(int(seed))
        grids = [ensemble.GRIDS[j % len(ensemble.GRIDS)] for j in range(case["cases"])]
        solvers = []
        for j, (nx, nz) in enumerate(grids):
            nx, nz = nx // case["scale"], nz // case["scale"]
            ra = float(math.exp(rng.uniform(math.log(1e5), math.log(1e7))))
            B = float(rng.uniform(0.3, 0.8))
            cfg = dict(aspect=nx / nz, nx=nx, nz=nz, RaT=ra, RaC=(B * ra,), ivis=2,
                       visT=float(math.exp(rng.uniform(math.log(1e2), math.log(1e4)))),
                       visC=(1.0 / float(rng.uniform(10.0, 100.0)),), tpc=case["tpc"], dlayer=0.15, initial_comp=0,
                       t_variant="fourier4", fixes=1, delta_visC=(1.2,), tolerance=case["tol"])
            g, _ = _solver(dict(mode=case["mode"], tuned=True), cfg, int(seed) + j)
            solvers.append(g)
        ensemble.ensemble_step(solvers, 1)   # a run's first step comes before those that are waited for
        return dict(kind=kind, solvers=solvers)
    cfg = _physics(case)
    g, T = _solver(case, cfg, int(seed))
    if kind == "solve":
        # the previous stage's solution is the warm start; T has moved on
        # by about what a time step changes
        g.multigrid()
        rng = np.random.default_rng(int(seed))
        nz, nx = g.nz, g.nx
        z, x = np.meshgrid(np.arange(-2, nz + 3) / nz, np.arange(-2, nx + 3) / nx, indexing="ij")
        dT = sum(rng.normal() * np.cos(a * math.pi * x) * np.sin(b * math.pi * z) for a in range(1, 4) for b in range(1, 4))
        T1 = ic.enforce_bcs_T(T + 1e-3 * dT, nx, nz)
        return dict(kind=kind, g=g, T=T1, SF=g.get("SF"))
    if kind == "tracers":
        g.multigrid()
        g.compute_velocities()
        return dict(kind=kind, g=g, dt=g.stability_RK4(), sort=case.get("sort"), n=0)
    # a step from within a run: its first step is behind it
    g.time_step(1)
    return dict(kind=kind, g=g, back=g.ntr <= TRACERS_BACK)


# ---- one pass -----------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "net":
        net = state["net"]
        net.set_sample(state["x"], state["t"], state["m"])
        out = net.forward()
        loss = net.backward()
        grads = net.get_grads()
        net.adam(1e-3)
        return dict(out=out, loss=loss, grads=grads, weights=net.get_weights())
    if kind == "bin":
        c = state["case"]
        p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
        st = state["lib"].tc_bin_tracers_noalloc(c["nx"], c["nz"], state["aspect"], c["ntype"], 1, p(state["r"]),
                                                 p(state["s"]), p(state["ty"]), state["r"].numel(), p(state["count"]),
                                                 p(state["nempty"]), p(state["C"]),
                                                 ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        if st != 0:
            raise RuntimeError(f"tc_bin_tracers_noalloc: status {st}")
        return dict(count=state["count"], nempty=state["nempty"], C=state["C"])
    if kind == "ensemble":
        ensemble.ensemble_step(state["solvers"], 1)
        return [{f: g.get(f) for f in ("T", "SF", "u", "w", "Cnew")} for g in state["solvers"]]
    g = state["g"]
    if kind == "solve":
        g.put("T", state["T"])
        g.put("SF", state["SF"])
        g.smoother_time_T("T")
        g.multigrid()
        g.compute_velocities()
        return dict(SF=g.get("SF"), u=g.get("u"), w=g.get("w"))
    if kind == "tracers":
        if state["sort"]:
            if state["n"] % state["sort"] == 0:
                g.sort_tracers()
            state["n"] += 1
        for stage, which in ((1, "x1"), (2, "x2"), (3, "x1"), (4, "x")):
            g.tracer_stage(stage, state["dt"])
            g.tracers_to_corners(which)
        return dict(Cnew=g.get("Cnew"), Cvis=g.get("Cvis"), conduct=g.get("conduct"), count=g.get("count_type"))
    g.time_step(1)
    out = {f: g.get(f) for f in ("T", "SF", "u", "w", "Cnew", "nempty")}
    if state["back"]:
        out["r"], out["s"] = g.get_tracers("x")
    return out


# ---- what a pass cannot do without ---------------------------------------------
def _net_flops(H, W):
    px = [H * W >> (2 * q) for q in range(4)]
    level = [0, 0, 1, 1, 2, 2, 3, 3, 2, 2, 1, 1, 0, 0]
    return 3 * sum(2 * 9 * ci * co * px[lv] for (ci, co), lv in zip(learn.LAYERS, level))


def work(case):
    kind = case["kind"]
    if kind == "net":
        n = learn.param_count()
        return dict(bytes=4.0 * (case["H"] * case["W"] * 9 + 5 * n), flops=float(_net_flops(case["H"], case["W"])))
    if kind == "ensemble":
        total = dict(bytes=0.0, flops=0.0)
        for j in range(case["cases"]):
            nx, nz = ensemble.GRIDS[j % len(ensemble.GRIDS)]
            w = work(dict(kind="step", mode="mixed", nx=nx // case["scale"], nz=nz // case["scale"], tpc=case["tpc"]))
            total = {k: total[k] + w[k] for k in total}
        return total
    pts = float((case["nx"] + 5) * (case["nz"] + 5))
    ntr = float((case["nx"] + 1) * (case["nz"] + 1) * case.get("tpc", 0))
    if kind == "bin":
        return dict(bytes=20.0 * ntr + pts * (4 * (case["ntype"] + 2) + 8 * case["ntype"]), flops=4.0 * ntr)
    # a solve: T, the warm start, C and the solution and velocities, and one
    # smoothing pass over the operator (six coefficients, the right-hand side
    # and the step) per digit of the residual; 13 taps a point
    digits = -math.log10(case.get("tol", 1e-8))
    solve = dict(bytes=pts * 8.0 * (6 + 9 * digits), flops=pts * 26.0 * digits)
    if kind == "solve":
        return solve
    # RK4 positions (304 B a tracer) and a binning per stage (20 B a tracer)
    tr = dict(bytes=ntr * (304.0 + 4 * 20.0) + 4 * 32.0 * pts, flops=ntr * 4 * 60.0)
    if kind == "tracers":
        return tr
    return dict(bytes=4 * solve["bytes"] + tr["bytes"] + 20.0 * ntr, flops=4 * solve["flops"] + tr["flops"])


def tolerance(case):
    kind = case["kind"]
    if kind == "net":
        # bfloat16 activations and activation gradients
        return dict(rel=2e-2, max=0.5)
    if kind == "bin":
        return "exact"
    if kind == "tracers":
        # FP64 in one order: a tracer within rounding of a cell's edge may be counted next door
        return dict(rel=1e-6, max=0.5, differ=1e-5)
    if kind == "solve":
        # the solve stops at a relative residual of `tol`; converged solutions
        # of the three modes are up to 1.6e-7 (FP64 form, 1e-7) and 5e-8
        # (1e-8) apart, 5e-7 at the worst node
        return dict(rel=7e-7 if case["mode"] == "fp64" else 2e-7, max=2e-6)
    if case.get("mode") == "fp64":
        return dict(rel=1e-7, max=1e-6, differ=1e-6)
    # fields as for a solve; a tracer within that of a cell's edge may be
    # counted next door, which changes a node's composition by 1/tpc: two such
    # tracers over the norm of the composition (a layer of 0.15)
    if kind == "ensemble":
        nodes = (ensemble.GRIDS[0][0] // case["scale"]) * (ensemble.GRIDS[0][1] // case["scale"])
    else:
        nodes = case["nx"] * case["nz"]
    return dict(rel=2.0 / case["tpc"] / math.sqrt(0.15 * nodes), max=0.6, differ=1e-4)


# ---- 64-bit answers -------------------------------------------------------------
def _exact_net(case, seed):
    x, t, m, w = _net_inputs(case, seed)
    th = torch.tensor(w.astype(np.float64), requires_grad=True)
    layers, o = [], 0
    for ci, co in learn.LAYERS:
        k = th[o:o + co * 9 * ci].reshape(co, 3, 3, ci).permute(0, 3, 1, 2)
        o += co * 9 * ci
        layers.append((k, th[o:o + co]))
        o += co
    hw, hb = th[o:o + 16], th[o + 16]
    F = torch.nn.functional

    def block(v, a):
        for q in (a, a + 1):
            v = F.gelu(F.conv2d(v, layers[q][0], layers[q][1], padding=1), approximate="tanh")
        return v

    v = torch.tensor(x.astype(np.float64)).permute(2, 0, 1)[None]
    e0 = block(v, 0)
    e1 = block(F.avg_pool2d(e0, 2), 2)
    e2 = block(F.avg_pool2d(e1, 2), 4)
    d = block(F.avg_pool2d(e2, 2), 6)
    for skip, a in ((e2, 8), (e1, 10), (e0, 12)):
        d = block(torch.cat([F.interpolate(d, scale_factor=2, mode="nearest"), skip], 1), a)
    out = torch.einsum("chw,c->hw", d[0], hw) + hb
    mm = torch.tensor(m.astype(np.float64))
    diff = (out - torch.tensor(t.astype(np.float64))) * mm
    loss = (diff * diff).sum() / mm.sum()
    loss.backward()
    return dict(out=out.detach(), loss=float(loss), grads=th.grad, weights=None)


def _exact_bin(case, seed):
    r, s, ty, aspect = _bin_inputs(case, seed)
    nx, nz, nt = case["nx"], case["nz"], case["ntype"]
    i = torch.floor(r / (aspect / nx) + 0.5).long()
    k = torch.floor(s / (1.0 / nz) + 0.5).long()
    key = (ty.long() * (nz + 1) + k) * (nx + 1) + i
    n = torch.bincount(key, minlength=(nt + 1) * (nz + 1) * (nx + 1)).reshape(nt + 1, nz + 1, nx + 1)
    tot = n.sum(0)
    C = torch.where(tot > 0, n[1:].double() / tot.clamp(min=1).double(), torch.zeros((), dtype=torch.float64, device=n.device))
    ix = torch.arange(-2, nx + 3, device=n.device).abs()
    ix = torch.where(ix > nx, 2 * nx - ix, ix)
    kx = torch.arange(-2, nz + 3, device=n.device).abs()
    kx = torch.where(kx > nz, 2 * nz - kx, kx)
    full = C[:, kx][:, :, ix].clone()
    # the corners beside the walls are filled before their column's mirror
    # is: they keep what a plane of zeros holds
    for kk in (1, nz + 3):
        for ii in (0, nx + 4):
            full[:, kk, ii] = 0.0
    return dict(count=None, nempty=None, C=full)


def exact(case, seed):
    if case["kind"] == "net":
        return _exact_net(case, seed) if case["H"] * case["W"] <= 40000 else None
    if case["kind"] == "bin":
        return _exact_bin(case, seed)
    # what a solve returns is the iterate at which its stop test passes: it is
    # `tol` away from the discrete solution, not a rounding away
    return None
