"""The coarse factorisation and inverse by blocks (k_lu_panels, k_inv_blocks)
against the oracle's banded LU: two-level solves whose coarse matrix ends on
and around the edges of the 16-column blocks, of the one-row-per-lane panel
(bandwidth 48), and of the widest band that the kernels take (72; above it the
general kernels).  Both coarse forms, the inverse and the substitution with the
factors, reproduce the oracle's solve to the bar of the full hierarchy's
(the same cycles, 1e-10 relative)."""
import numpy as np
import pytest

import oracle
from conftest import load_oracle_state, rel_err
from tracer_code_amd import Solver, config, ic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nxc,nzc", [
    (4, 4), (7, 7), (14, 4), (9, 6), (10, 23), (10, 24), (8, 35), (8, 36), (40, 7), (24, 8),
], ids=lambda v: str(v))
def test_two_level_solve_matches_the_oracle(monkeypatch, nxc, nzc):
    cfg = dict(config.PRESETS["cfg0"], nx=2 * nxc, nz=2 * nzc, aspect=nxc / nzc, tpc=4, grids=2)
    params = config.make_params(**cfg)
    cfg.update(nx=params.nx, nz=params.nz)
    assert (params.nx, params.nz, params.grids) == (2 * nxc, 2 * nzc, 2)
    T, r, s, ty = ic.workload(cfg, seed=3)
    o = load_oracle_state(params, T, r, s, ty)
    assert o.multigrid() == 0
    for lu in ("0", "1"):
        monkeypatch.setenv("TC_COARSE_LU", lu)
        print(f"[coarse] {nxc}x{nzc}, substitution {lu}", flush=True)
        with Solver(params, len(r)) as g:
            g.initialize(T, r, s, ty)
            q, resid, ref = g.multigrid()
            assert q == int(o.scalar(oracle.ORS_Q))
            assert rel_err(g.get("SF"), o.plane(oracle.OR_SF)) <= 1e-10
