"""The per-type fields and the tracer arrays across the boundary: what
tc_put_field took comes back from tc_get_field, in the type-fastest layout, for
every number of types and at row lengths that are no multiple of a block or
a chunk; and positions in the caller's order, sorted or not."""
import numpy as np
import pytest

from tracer_code_amd import Solver, config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz,nt", [(16, 16, 1), (36, 52, 2), (252, 64, 3), (260, 20, 4), (640, 320, 4)])
def test_fields_round_trip(nx, nz, nt):
    ones = (1.0,) * nt
    params = config.make_params(nx=nx, nz=nz, aspect=nx / nz, grids=6 if nx > 300 else 2, ntype=nt, RaC=ones, visC=ones,
                                delta_visC=(2.0,) * nt, conduct_factor=ones, Htype=ones)
    print(f"[boundary] {params.nx}x{params.nz}, {nt} types", flush=True)
    rng = np.random.default_rng(nx + nt)
    shape = (params.nz + 5, params.nx + 5)
    n = 70001
    with Solver(params, n) as g:
        for name in ("Cnew", "Cvis", "Cbuoy"):
            a = rng.random(shape + (nt,))
            g.put(name, a)
            assert np.array_equal(g.get(name), a)
        for name, sh in (("count_type", shape + (nt + 1,)), ("nempty", shape)):
            a = rng.integers(0, 1 << 30, sh).astype(np.int32)
            g.put(name, a)
            assert np.array_equal(g.get(name), a)
        a = rng.random(shape)
        g.put("T1", a)
        assert np.array_equal(g.get("T1"), a)
        r = rng.uniform(1e-6, params.aspect - 1e-6, n)
        s = rng.uniform(1e-6, 1.0 - 1e-6, n)
        ty = rng.integers(0, nt + 1, n).astype(np.int32)
        g.put_tracers(r, s, ty)
        for sort in (False, True):
            if sort:
                g.sort_tracers()
            x, z = g.get_tracers("x")
            assert np.array_equal(x, r) and np.array_equal(z, s) and np.array_equal(g.get_tracer_types(), ty)
