"""The standard PCG's matvec forms the new direction in LDS windows: three per block up to 258
levels, nine beyond, the first 1024 entries loaded ahead (three windows of 41 levels fit, of 42
do not).  Both sides of each line, one level, blocks that end inside a column and grids of less
than one block, against the oracle from the same start: only the order of the global sums
differs, so four iterates agree to rounding (1e-11), as twelve do in test_gpu_cg_reductions."""
import numpy as np
import pytest

import oracle as O
from cism_amd import configs, gpu as G
from helpers import assembled_system, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("ewn, nsn, nz", [(4, 5, 2), (30, 31, 2), (13, 9, 41), (9, 13, 42), (7, 6, 258), (6, 7, 259)])
def test_windows(ewn, nsn, nz, periodic):
    p = configs.grf_sheet(ewn=ewn, nsn=nsn, nz=nz, seed=9, periodic=periodic)
    A, bu, bv, u, v, _ = assembled_system(p, seed=5)
    print(f"[windows] {ewn}x{nsn}x{nz} periodic {periodic}", flush=True)
    ou, ov, gu, gv = (a.copy(order="F") for a in (u, v, u, v))
    st, _, nit_o = O.pcg(p, A, bu, bv, ou, ov, 1, chrongear=False, maxiters=4)
    assert st == 0
    with G.Context.for_problem(p) as ctx:
        ctx.set_linear_solver(4, 1e-8)
        _, nit_g = ctx.pcg_solver_standard_3d(p.active_vertex, *A, bu, bv, gu, gv, 1)
    assert nit_g == nit_o
    x_o, x_g = (np.concatenate([a.ravel(), b.ravel()]) for a, b in ((ou, ov), (gu, gv)))
    print(f"  rel L2 diff {rel_l2(x_g, x_o):.2e}")
    assert rel_l2(x_g, x_o) < 1e-11
