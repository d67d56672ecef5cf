"""The counting kernel and the composition ghosts against numpy, value for
value: tracer counts around the 256 and 512 tracers of a workgroup's halves,
one and many workgroups, tracers node by node, cell by cell, in no order (the
workgroup's table of counters overflows) and all on one node, spacings that
are powers of two and not, the smallest grid."""
import ctypes

import numpy as np
import pytest

from test_zz_no_alloc import _Hip
from tracer_code_amd import _abi

pytestmark = pytest.mark.gpu


def expected(nx, nz, aspect, nt, r, s, ty, C):
    """composition.f90:704-776 and 792-803, the latter in its order."""
    i = np.floor(r / (aspect / nx) + 0.5).astype(int) + 2
    k = np.floor(s / (1.0 / nz) + 0.5).astype(int) + 2
    cnt = np.zeros((nt + 1, nz + 5, nx + 5), dtype=np.int32)
    np.add.at(cnt, (ty, k, i), 1)
    for d in (1, 2):
        cnt[:, 2:-2, 2 - d] = cnt[:, 2:-2, 2 + d]
        cnt[:, 2:-2, nx + 2 + d] = cnt[:, 2:-2, nx + 2 - d]
        cnt[:, 2 - d, 2:-2] = cnt[:, 2 + d, 2:-2]
        cnt[:, nz + 2 + d, 2:-2] = cnt[:, nz + 2 - d, 2:-2]
    tot = cnt.sum(0)
    C = C.copy()
    some = np.zeros(tot.shape, dtype=bool)
    some[2:-2, 2:-2] = tot[2:-2, 2:-2] > 0
    for t in range(nt):
        C[t][some] = cnt[t + 1][some] / tot[some]
        c = C[t]
        for d in (1, 2):
            c[2:-2, 2 - d] = c[2:-2, 2 + d]
            c[2:-2, nx + 2 + d] = c[2:-2, nx + 2 - d]
            c[2 - d, :] = c[2 + d, :]
            c[nz + 2 + d, :] = c[nz + 2 - d, :]
    return cnt, tot, C


@pytest.mark.parametrize("nx,nz,nt", [(2, 2, 1), (32, 16, 2), (300, 200, 2)])
@pytest.mark.parametrize("order", ["nodes", "cells", "none", "one"])
@pytest.mark.parametrize("n", [1, 255, 257, 511, 513, (1 << 20) + 1])
def test_counts(nx, nz, nt, order, n):
    rng = np.random.default_rng(n % 1000 + nx)
    aspect = nx / nz if nx != 300 else 1.7
    dr, ds = aspect / nx, 1.0 / nz
    node = np.arange(n) * ((nx + 1) * (nz + 1)) // n
    i, k = node // (nz + 1), node % (nz + 1)
    if order == "nodes":
        r, s = (i + rng.random(n) - 0.5) * dr, (k + rng.random(n) - 0.5) * ds
    elif order == "cells":
        r, s = (i + rng.random(n)) * dr, (k + rng.random(n)) * ds
    elif order == "none":
        r, s = rng.random(n) * aspect, rng.random(n)
    else:
        r, s = np.full(n, 0.9 * dr), np.full(n, 0.9 * ds)
    r, s = np.clip(r, 1e-6 * dr, aspect - 1e-6 * dr), np.clip(s, 1e-6 * ds, 1 - 1e-6 * ds)
    ty = rng.integers(0, nt + 1, n).astype(np.int32) if order != "one" else np.full(n, nt, dtype=np.int32)
    C = rng.random((nt, nz + 5, nx + 5))
    print(f"[bin] {nx}x{nz} {order} n={n}", flush=True)
    hip = _Hip()
    cnt0, ne0 = np.full((nt + 1, nz + 5, nx + 5), 7, dtype=np.int32), np.full((nz + 5, nx + 5), 9, dtype=np.int32)
    R, S, TY, CNT, NE, CN = (hip.put(a) for a in (r, s, ty, cnt0, ne0, C))
    assert _abi.load_library().tc_bin_tracers_noalloc(nx, nz, ctypes.c_double(aspect), nt, 1, R, S, TY,
                                                      ctypes.c_int64(n), CNT, NE, CN, None) == 0
    got = hip.get(CNT, cnt0), hip.get(NE, ne0), hip.get(CN, C)
    hip.free()
    cnt, tot, Cx = expected(nx, nz, aspect, nt, r, s, ty, C)
    assert np.array_equal(got[0], cnt) and np.array_equal(got[1], tot) and np.array_equal(got[2], Cx)
