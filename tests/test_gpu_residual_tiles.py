"""The tiled residual on device arrays (cism_compute_residual_vector_3d_noalloc) at the edges
of its 64-node tiles: a ragged last tile with an odd number of coefficients, one level, tiles
without an active node, more tiles than workgroups, and blocks that start 8 bytes off a 16-byte
boundary (8-byte loads).  The residual bit for bit against the row products summed in the same
order by numpy; the norms to 1e-13 relative (sums of at most 3e5 squares in another order)."""
import ctypes as C

import numpy as np
import pytest

from cism_amd import gpu as G
from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu


def reference(nx, ny, nz, periodic, av, A, bu, bv, u, v):
    lo = 2 if periodic else 1
    own = np.zeros((nx - 1, ny - 1), bool)
    own[lo:nx - 2, lo:ny - 2] = True
    own &= av != 0
    up, vp = (np.pad(a, 1) for a in (u, v))
    su, sv = np.zeros(u.shape), np.zeros(u.shape)
    for m in range(27):
        sl = tuple(slice(o, o + n) for o, n in zip((m // 9, m % 3, m // 3 % 3), u.shape))
        su = (su + A[0][m] * up[sl]) + A[1][m] * vp[sl]
        sv = (sv + A[2][m] * up[sl]) + A[3][m] * vp[sl]
    return np.where(own, su - bu, 0.0), np.where(own, sv - bv, 0.0), own


@pytest.mark.parametrize("nx,ny,nz,periodic,active,off", [
    (8, 8, 1, 1, 1.0, 0),       # 49 nodes: one tile, short
    (8, 8, 1, 1, 1.0, 1),
    (12, 10, 3, 0, 0.7, 0),     # 297 nodes: last tile of 41, an odd count of coefficients
    (12, 10, 3, 0, 0.7, 1),
    (36, 35, 10, 1, 0.05, 0),   # most tiles without an active node
    (160, 140, 5, 1, 0.9, 1),   # more tiles than the 1024 workgroups
])
def test_residual_tiles(nx, ny, nz, periodic, active, off):
    rng = np.random.default_rng(nx + off)
    s3, s2 = (nz, nx - 1, ny - 1), (nx - 1, ny - 1)
    A = [np.asfortranarray(rng.standard_normal((27,) + s3)) for _ in range(4)]
    bu, bv, u, v = (np.asfortranarray(rng.standard_normal(s3)) for _ in range(4))
    av = np.asfortranarray((rng.random(s2) < active).astype(np.int32))
    hip, L = Hip(), G.lib()
    f = L.cism_compute_residual_vector_3d_noalloc
    f.argtypes = [C.c_int] * 5 + [C.c_void_p] * 13
    shift = np.zeros(off)
    blocks = [hip.put(np.concatenate((shift, a.ravel(order="F")))).value + 8 * off for a in A]
    vecs = [hip.put(a) for a in (bu, bv, u, v)]
    nn = u.size
    ru, rv, norms = (hip.put(np.full(n, np.nan)) for n in (nn, nn, 2))
    assert f(nx, ny, nz, periodic, 0, None, hip.put(av), *blocks, *vecs, ru, rv, norms) == 0
    got = [hip.get(p, nn).reshape(s3, order="F") for p in (ru, rv)]
    L2, L2r = hip.get(norms, 2)
    hip.free()
    wu, wv, own = reference(nx, ny, nz, periodic, av, A, bu, bv, u, v)
    assert np.array_equal(got[0], wu) and np.array_equal(got[1], wv)
    w2 = np.sqrt((wu ** 2).sum() + (wv ** 2).sum())
    b2 = np.sqrt(((bu ** 2 + bv ** 2) * own).sum())
    assert abs(L2 - w2) <= 1e-13 * w2 and abs(L2r - w2 / b2) <= 1e-13 * w2 / b2


@pytest.mark.parametrize("nx,ny,nz", [
    (304, 264, 1),     # one level: the middle nine slots alone
    (160, 140, 5),     # 1726 tiles, all but a few without a row, more than one pass of the workgroups
    (12, 9, 150),      # a tile inside a column
])
def test_few_rows_far_apart(nx, ny, nz):
    """the first and the last owned column alone, blocks that hold NaN where no row reads"""
    rng = np.random.default_rng(nz)
    s3, s2 = (nz, nx - 1, ny - 1), (nx - 1, ny - 1)
    A = [np.asfortranarray(rng.standard_normal((27,) + s3)) for _ in range(4)]
    bu, bv, u, v = (np.asfortranarray(rng.standard_normal(s3)) for _ in range(4))
    av = np.zeros(s2, np.int32, order="F")
    av[2, 2] = av[nx - 3, ny - 3] = 1
    hip, L = Hip(), G.lib()
    f = L.cism_compute_residual_vector_3d_noalloc
    f.argtypes = [C.c_int] * 5 + [C.c_void_p] * 13
    wu, wv, own = reference(nx, ny, nz, 1, av, A, bu, bv, u, v)
    for a in A:
        a[:9, 0] = np.nan          # the level above the surface and the one below the bed
        a[18:, nz - 1] = np.nan
        a[:, :, av == 0] = np.nan
    dev = [hip.put(a) for a in (*A, bu, bv, u, v)]
    nn = u.size
    ru, rv, norms = (hip.put(np.full(n, np.nan)) for n in (nn, nn, 2))
    assert f(nx, ny, nz, 1, 0, None, hip.put(av), *dev, ru, rv, norms) == 0
    got = [hip.get(p, nn).reshape(s3, order="F") for p in (ru, rv)]
    L2 = hip.get(norms, 2)[0]
    hip.free()
    assert own.sum() == 2
    assert np.array_equal(got[0], wu) and np.array_equal(got[1], wv)
    w2 = np.sqrt((wu ** 2).sum() + (wv ** 2).sum())
    assert abs(L2 - w2) <= 1e-13 * w2
