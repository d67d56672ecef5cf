"""The blocked visits of the FP64 reference form (k_visit_ref: several sweeps
per launch, the correction in registers) against one sweep per launch
(k_sweep, TC_TB=0): the same operations in the same order, so the same bits,
at the sizes where the regions end -- a level of one region with and without
idle columns, one cell more than a region, ragged tiles, spacings that are
no powers of two, more sweeps than a launch takes."""
import numpy as np
import pytest

from tracer_code_amd import Solver, config, ic

pytestmark = pytest.mark.gpu


def solve(monkeypatch, tb, nx, nz, **ov):
    monkeypatch.setenv("TC_TB", tb)
    cfg = dict(config.PRESETS["cfg0"], nx=nx, nz=nz, aspect=nx / nz, tpc=2, max_cycles=3, **ov)
    params = config.make_params(**cfg)
    cfg.update(nx=params.nx, nz=params.nz)
    T, r, s, ty = ic.workload(cfg, seed=5)
    print(f"[visit] {params.nx}x{params.nz}, {params.grids} levels, Nmulti {params.Nmulti}, TC_TB={tb}", flush=True)
    SF = np.random.default_rng(1).uniform(-1.0, 1.0, (params.nz + 5, params.nx + 5))   # walls included
    with Solver(params, len(r)) as g:
        g.initialize(T, r, s, ty, SF=SF)
        try:
            g.multigrid()
        except Exception:
            pass   # three cycles need not converge: the residual and the next step's fields show the iterates
        st = g.stats()
        res = st.residual_last, st.res_ref_last, list(st.sweeps_exec), list(st.residuals_exec)
        return res, g.get("SF"), g.get("RHS")


@pytest.mark.parametrize("nx,nz,ov", [
    (16, 16, {}), (32, 32, {}), (34, 32, {}), (64, 32, {}), (64, 36, {}), (128, 64, dict(Nmulti=7)),
    (96, 96, {}), (152, 104, dict(Nmulti=5)), (100, 60, dict(Nmulti=97)), (20, 84, dict(Vbc=1)),
    (256, 256, dict(Nmulti=9)), (512, 320, dict(Nmulti=6)), (128, 128, dict(fixes=1, tolerance=1e-3, Nmulti=30)),
    (608, 352, dict(Nmulti=13, fixes=1, tolerance=1e-2, ivis=0)),
])
def test_blocked_visits_same_bits(monkeypatch, nx, nz, ov):
    a, sfa, ra = solve(monkeypatch, "0", nx, nz, **ov)
    b, sfb, rb = solve(monkeypatch, "1", nx, nz, **ov)
    assert a == b and a[0] > 0.0
    assert np.array_equal(sfa, sfb) and np.array_equal(ra, rb)


@pytest.mark.parametrize("nx,nz", [(32, 32), (152, 104), (512, 320)])
@pytest.mark.parametrize("seq", [
    [1, 2, 3, 2, 3, 2], [2, 1, 2, 3], [1, 3, 2], [1, 2, 3, 1, 2], [1, 2, 2, 3, 2, 1], [1, 2, 3],
], ids=lambda s: "".join(map(str, s)))
def test_schedules_same_bits(monkeypatch, nx, nz, seq):
    """Schedules other than the presets': they skip or repeat levels, start
    below level 1, or end on a level from which the next cycle's first visit is
    more than one level away."""
    monkeypatch.setattr(config, "cycle_sequence", lambda grids, cycle="W": seq)
    a, sfa, ra = solve(monkeypatch, "0", nx, nz, Nmulti=7, grids=3)
    b, sfb, rb = solve(monkeypatch, "1", nx, nz, Nmulti=7, grids=3)
    assert a == b and a[0] > 0.0
    assert np.array_equal(sfa, sfb) and np.array_equal(ra, rb)


@pytest.mark.parametrize("mode", ["mixed", "dc64"])
@pytest.mark.parametrize("nx,nz,ov", [
    (32, 32, {}), (66, 34, dict(Nmulti=9)), (128, 32, dict(Nmulti=8)), (152, 104, dict(Nmulti=16)),
    (100, 60, dict(Nmulti=97)), (192, 64, dict(Vbc=1, Nmulti=10)), (512, 320, dict(Nmulti=8)),
    (256, 256, dict(Nmulti=12)),
])
def test_defect_correction_visits_reach_the_same_solution(monkeypatch, mode, nx, nz, ov):
    """k_visit13 against one sweep per launch: another rounding of the
    corrections only, so both solves stop at the tolerance, within a cycle of
    each other, and SF agrees to what a relative residual of 1e-11 leaves
    (FP64 corrections, 1e-9 relative to the largest value) or of 1e-9 (FP32
    ones, 1e-6)."""
    tol = 1e-9 if mode == "mixed" else 1e-11
    cfg = dict(config.PRESETS["cfg0"], nx=nx, nz=nz, aspect=nx / nz, tpc=2, tolerance=tol, fixes=1, **ov)
    params = config.make_params(**cfg)
    cfg.update(nx=params.nx, nz=params.nz)
    T, r, s, ty = ic.workload(cfg, seed=5)
    print(f"[visit13] {mode} {params.nx}x{params.nz}, {params.grids} levels, Nmulti {params.Nmulti}", flush=True)
    got = []
    for tb in ("0", "1"):
        monkeypatch.setenv("TC_TB", tb)
        with Solver(params, len(r)) as g:
            g.initialize(T, r, s, ty)
            g.set_mode(mode)
            q, resid, ref = g.multigrid()
            assert resid <= tol * ref
            got.append((q, g.get("SF")))
    assert abs(got[0][0] - got[1][0]) <= 1
    assert np.max(np.abs(got[0][1] - got[1][1])) <= (1e-6 if mode == "mixed" else 1e-9) * np.max(np.abs(got[0][1]))


@pytest.mark.parametrize("mode", ["mixed", "dc64"])
@pytest.mark.parametrize("nx,nz", [(32, 32), (152, 104), (256, 128)])
def test_other_tables_stay_blocked(monkeypatch, mode, nx, nz):
    """Finite-difference tables other than the second-order ones: the
    defect-correction visits still run several sweeps per launch, and solve the
    same equation as one sweep per launch does (to the bars above)."""
    tol = 1e-9 if mode == "mixed" else 1e-11
    cfg = dict(config.PRESETS["cfg0"], nx=nx, nz=nz, aspect=nx / nz, tpc=2, tolerance=tol, fixes=1, Nmulti=20)
    params = config.make_params(**cfg)
    cfg.update(nx=params.nx, nz=params.nz)
    for t, f in ((params.D1, 1.01), (params.D2, 0.99), (params.D3, 1.02), (params.D4, 0.98)):
        for j in range(5):
            t[j] *= f
    T, r, s, ty = ic.workload(cfg, seed=5)
    got = []
    for tb in ("0", "1"):
        monkeypatch.setenv("TC_TB", tb)
        print(f"[other tables] {mode} {params.nx}x{params.nz}, {params.grids} levels, TC_TB={tb}", flush=True)
        with Solver(params, len(r)) as g:
            g.initialize(T, r, s, ty)
            g.set_mode(mode)
            g.set_profiling(True)
            q, resid, ref = g.multigrid()
            assert resid <= tol * ref
            got.append((q, g.get("SF"), g.kernel_timing()[1], g.stats().sweeps_exec[0]))
    assert abs(got[0][0] - got[1][0]) <= 1
    assert np.max(np.abs(got[0][1] - got[1][1])) <= (1e-6 if mode == "mixed" else 1e-9) * np.max(np.abs(got[0][1]))
    assert got[0][2] == got[0][3] and 4 * got[1][2] <= got[1][3]   # launches and sweeps of level 1
