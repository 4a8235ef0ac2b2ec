"""The depth solvers' element kernel, four lanes a cell with the layers in LDS, at its extremes:
two and 64 levels, a ragged last workgroup.  Four Picard iterations against the oracle at the
bound of test_gpu_depth (both run the same iterations; 1e-8)."""
import numpy as np
import pytest

import oracle as O
from cism_amd import configs, gpu as G
from helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("approx", [3, 4])
@pytest.mark.parametrize("ewn,nsn,nz", [(13, 11, 2), (13, 11, 64)])   # 255 cells: 3 workgroups and 63 cells
def test_layers(ewn, nsn, nz, approx):
    p = configs.grf_sheet(ewn=ewn, nsn=nsn, nz=nz, seed=4)
    lu, lv = O.loads(p)
    print(f"[depth] {ewn}x{nsn}x{nz} approx={approx}", flush=True)
    ro = O.picard_depth(p, lu, lv, approx, maxiter=4)
    with G.Context.for_problem_2d(p) as ctx:
        rg = ctx.velo_higher_solve_depth(p, lu, lv, approx, maxiter_nonlinear=4)
    assert rg["picard_iters"] == ro["picard_iters"]
    for k in ("uvel", "vvel", "uvel_2d", "vvel_2d", "efvs"):
        assert np.abs(ro[k]).max() > 0
        assert rel_l2(rg[k], ro[k]) < 1e-8, k
