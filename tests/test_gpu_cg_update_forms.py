"""The Chron-Gear update where its form changes: column factors in registers or in memory (past
24 levels, and past 12 where the scalars come from a workgroup of their own), and scalars formed
by the update itself or, from more than 2048 workgroups on, read from memory: 64 columns a
workgroup with the column preconditioner, 256 nodes with the diagonal or on one level.

The large grids are a small periodic system tiled 8 x 8: its iterates are the small system's,
tiled, and its dot products the small ones 64 times, so the oracle runs the small system alone.
Only the order of the global sums differs: 1e-11, as in test_gpu_cg_reductions."""
from types import SimpleNamespace

import numpy as np
import pytest

import oracle as O
from cism_amd import configs, gpu as G

pytestmark = pytest.mark.gpu


def periodic_system(n, nz, rng):
    """blocks as (n, n, nz, 27) [j, i, k, slot] of a symmetric, diagonally dominant operator on
    n x n columns, a tenth of them inactive (no row, no column); right-hand sides; the mask"""
    av = rng.random((n, n)) > 0.1
    A = [np.zeros((n, n, nz, 27)) for _ in range(4)]
    for m in range(13):
        iA, jA, kA = m % 3 - 1, m // 3 % 3 - 1, m // 9 - 1
        on = av & np.roll(av, (-jA, -iA), (0, 1))
        c = [0.25 * rng.standard_normal((n, n, nz)) * on[..., None] for _ in range(4)]
        if m == 4:                       # the node below: the columns' own coupling
            c[0] -= 2.0 * av[..., None]
            c[3] -= 2.0 * av[..., None]
        for b, t in ((0, 0), (1, 2), (2, 1), (3, 3)):
            if kA:
                c[b][..., 0] = 0.0
            A[b][..., m] = c[b]
            A[t][..., 26 - m] = np.roll(c[b], (jA, iA, kA), (0, 1, 2))
    for b in (0, 3):
        A[b][..., 13] = (10.0 + rng.random((n, n, nz))) * av[..., None]
    A[1][..., 13] = 0.1 * rng.standard_normal((n, n, nz)) * av[..., None]
    A[2][..., 13] = A[1][..., 13]
    rhs = [rng.standard_normal((n, n, nz)) * av[..., None] for _ in range(2)]
    return A, rhs, av.astype(np.int32)


def tiled(n, tiles, arrays):
    """the staggered arrays of tiles x tiles copies, halo included, in the Fortran layouts"""
    idx = (np.arange(n * tiles + 3) - 2) % n
    return [np.ascontiguousarray(a[idx][:, idx]).T for a in arrays]


@pytest.mark.parametrize("n,tiles,nz,precond", [
    (24, 1, 24, 2), (24, 1, 25, 2), (9, 1, 48, 2),   # the update's own scalars, both factor forms
    (46, 8, 12, 2), (46, 8, 13, 2), (46, 8, 25, 2),  # 371 x 371 columns: 2151 workgroups
    (46, 8, 4, 1),                                   # 550,564 nodes: 2151 workgroups
    (92, 8, 1, 2), (92, 8, 1, 1),                    # 739 x 739 columns: 2134 workgroups
])
def test_update_forms(n, tiles, nz, precond):
    rng = np.random.default_rng(n + nz)
    A, rhs, av = periodic_system(n, nz, rng)
    print(f"[cg update] {n}x{n}x{nz} tiled {tiles} precond {precond}", flush=True)
    got = {}
    for t in (1, tiles):
        a = tiled(n, t, A)
        bu, bv = tiled(n, t, rhs)
        mask, = tiled(n, t, [av])
        xu, xv = np.zeros_like(bu), np.zeros_like(bv)
        nx = n * t + 4
        if t == 1:
            p = SimpleNamespace(nx=nx, ny=nx, nz=nz, periodic=True, active_vertex=mask)
            ou, ov = xu.copy(order="F"), xv.copy(order="F")
            st, _, nit_o = O.pcg(p, a, bu, bv, ou, ov, precond, maxiters=8, tolerance=1e-30)
            assert st == 0 and nit_o == 8
        with G.Context(nx, nx, nz) as ctx:
            ctx.set_linear_solver(8, 1e-30)
            _, nit = ctx.pcg_solver_chrongear_3d(mask, *a, bu, bv, xu, xv, precond)
        assert nit == 8
        got[t] = [x[:, 2:n * t + 2, 2:n * t + 2] for x in (xu, xv)]
    want = [x[:, 2:n + 2, 2:n + 2] for x in (ou, ov)]
    for t in got:
        for g, w in zip(got[t], want):
            w = np.tile(w, (1, t, t))
            err = np.linalg.norm(g - w) / np.linalg.norm(w)
            print(f"  {t}: rel L2 diff {err:.2e}")
            assert err < 1e-11


@pytest.mark.parametrize("n", [40, 364])   # 29 and 2105 workgroups of 64 columns
def test_timed_update_leaves_solves_alone(n):
    """the timing of the FP32 update, in the form that the grid's solves run, between two solves"""
    p = configs.grf_sheet(ewn=n, nsn=n, nz=3, seed=2)
    print(f"[cg update] timing {n}x{n}x3", flush=True)
    with G.Context.for_problem(p) as ctx:
        lu, lv = ctx.loads(p)
        solve = lambda: ctx.velo_higher_solve_3d(p, lu, lv, precision=1, maxiter_nonlinear=2)   # noqa: E731
        first = solve()
        assert ctx.time_kernel(4, 3) > 0.0
        again = solve()
    assert first["fp32_matvecs"] == again["fp32_matvecs"] > 0
    assert np.array_equal(first["uvel"], again["uvel"]) and np.array_equal(first["vvel"], again["vvel"])
