"""The solver's NaN signal: an all-zero matrix gives alpha = 0 / 0, an error in the reference
(pcg:460-463, 1505-1512) and in the oracle.  It reaches the host with a convergence check, every
fifth iteration, or, when the iterations end between two checks, at the end of the solve; a
context solves as before after it."""
from types import SimpleNamespace

import numpy as np
import pytest

import oracle as O
from cism_amd import gpu as G
from helpers import rel_l2
from test_gpu_cg_update_forms import periodic_system, tiled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("its", [3, 5, 7])    # before the first check, at it, after it
@pytest.mark.parametrize("chrongear,precond", [(True, 0), (True, 1), (True, 2), (False, 0), (False, 1), (False, 2)])
@pytest.mark.parametrize("n,nz", [(12, 4), (12, 1), (740, 1)])   # own scalars; from memory (2157 workgroups)
def test_zero_matrix(n, nz, chrongear, precond, its):
    nx = n + 4
    zero = np.zeros((27, nz, nx - 1, nx - 1), order="F")
    b = np.ones((nz, nx - 1, nx - 1), order="F")
    av = np.ones((nx - 1, nx - 1), np.int32, order="F")
    print(f"[nan] {n}x{n}x{nz} chrongear {chrongear} precond {precond} its {its}", flush=True)
    if n < 100:
        p = SimpleNamespace(nx=nx, ny=nx, nz=nz, periodic=True, active_vertex=av)
        ou, ov = np.zeros_like(b), np.zeros_like(b)
        assert O.pcg(p, [zero] * 4, b, b, ou, ov, precond, chrongear=chrongear, maxiters=its)[0] != 0
    with G.Context(nx, nx, nz) as ctx:
        ctx.set_linear_solver(its, 1e-8)
        f = ctx.pcg_solver_chrongear_3d if chrongear else ctx.pcg_solver_standard_3d
        x = [np.zeros_like(b) for _ in range(2)]
        with pytest.raises(G.CismError, match="NaN"):
            f(av, zero, zero, zero, zero, b, b, *x, precond)
        if n < 100:
            A, rhs, mask = periodic_system(n, nz, np.random.default_rng(n))
            A = tiled(n, 1, A)
            (bu, bv), (mask,) = tiled(n, 1, rhs), tiled(n, 1, [mask])
            p.active_vertex = mask
            ou, ov, xu, xv = (np.zeros_like(bu) for _ in range(4))
            st, _, nit_o = O.pcg(p, A, bu, bv, ou, ov, precond, chrongear=chrongear, maxiters=its)
            assert st == 0 and f(mask, *A, bu, bv, xu, xv, precond)[1] == nit_o
            s = np.s_[:, 2:n + 2, 2:n + 2]
            assert rel_l2(np.stack((xu[s], xv[s])), np.stack((ou[s], ov[s]))) < 1e-11
