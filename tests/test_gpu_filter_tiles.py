"""The C filter's tiles (k_filter_multi) against one launch per iteration, on
fields that the tracers do not give: random ratios, values beyond [0,1] (the
clamp), a NaN, and infinities and values whose quotients overflow, at the heights and widths where a tile ends -- heights that
one tile holds (4 to 16 rows), the smallest height with tiles, a last tile
that overlaps the one before it, one column or row more than a tile, and
every tile height.  Same iterates, stop and bits."""
import numpy as np
import pytest

from tracer_code_amd import Solver, config

pytestmark = pytest.mark.gpu


# the larger grids take tiles of 11, 16 and 21 rows (on 256 CUs), the smaller
# ones of 8; spacings that are powers of two at 512 and 1024 rows
@pytest.mark.parametrize("kind", ["ratio", "beyond", "nan", "huge"])
@pytest.mark.parametrize("nx,nz", [(12, 4), (52, 6), (10, 16), (24, 16), (104, 10),
                                   (300, 14), (16, 18), (54, 20), (56, 38), (108, 50), (110, 26), (160, 96), (212, 130),
                                   (1952, 192), (1024, 512), (1952, 288), (544, 1024), (1920, 992), (2048, 1024)])
def test_filter_tiles_same_bits(nx, nz, kind):
    params = config.make_params(nx=nx, nz=max(nz, 8), aspect=nx / nz, grids=2 if nx * nz < 50000 else 6, ivis=2,
                                visC=(1.0 / 30.0,), delta_visC=(1.5,))
    params.nz = nz   # (make_params keeps 4 cells on the coarsest level, the library 2)
    print(f"[filter tiles] {params.nx}x{params.nz} {kind}", flush=True)
    assert params.nx == nx
    rng = np.random.default_rng(nx * 7 + nz)
    C = rng.integers(0, 21, (nz + 5, nx + 5, 1)) / 20.0
    if kind == "beyond":
        C[rng.random(C.shape) < 0.1] = 1.5
        C[rng.random(C.shape) < 0.1] = -0.25
    if kind == "nan":
        C[nz // 2, nx // 2] = np.nan
    if kind == "huge":
        C[1, nx // 3], C[nz // 2, 2], C[nz - 1, nx // 2], C[nz // 2, nx - 1] = np.inf, -np.inf, 1e307, -1e307
    out = []
    with Solver(params, 0) as g:
        for blocking in (False, True):
            g.set_filter_blocking(blocking)
            g.put("Cnew", C)
            n0 = g.stats().c_iters
            n = g.smoother_time()
            out.append((g.get("Cvis"), n, g.stats().c_iters - n0))
    assert out[0][1] == out[1][1] and out[0][2] == out[1][2] and out[0][2] > 4
    assert np.array_equal(out[0][0], out[1][0], equal_nan=True)


@pytest.mark.parametrize("nx,nz", [(24, 16), (64, 32), (108, 50), (256, 128)])
def test_other_table_same_bits(nx, nz):
    """A second-derivative table that is not (1, -2, 1), on spacings that are
    powers of two and not."""
    params = config.make_params(nx=nx, nz=nz, aspect=nx / nz, grids=2, ivis=2, visC=(1.0 / 30.0,), delta_visC=(1.5,))
    params.D2[1], params.D2[2], params.D2[3] = 0.96, -1.93, 0.98
    print(f"[filter tiles] {params.nx}x{params.nz} other table", flush=True)
    C = np.random.default_rng(nx).integers(0, 21, (nz + 5, nx + 5, 1)) / 20.0
    out = []
    with Solver(params, 0) as g:
        for blocking in (False, True):
            g.set_filter_blocking(blocking)
            g.put("Cnew", C)
            n0 = g.stats().c_iters
            n = g.smoother_time()
            out.append((g.get("Cvis"), n, g.stats().c_iters - n0))
    assert out[0][1:] == out[1][1:] and out[0][2] > 4
    assert np.array_equal(out[0][0], out[1][0])
