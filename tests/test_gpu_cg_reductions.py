"""The dot products that the PCG kernels add for themselves, at the sizes where their form
changes: one record a group (up to 64 node blocks), up to eight (512), more (a launch of its
own, from 513 on), and updates of more than 2048 workgroups, whose scalars come from one
workgroup.  A dozen iterations from the same start against the oracle, as in
test_gpu_parity.test_pcg_short: only the order of the global sums differs, so the iterates agree
to rounding (1e-11).  Twelve iterations end between two convergence checks, eleven leave a
standard PCG's halo as it is."""
import numpy as np
import pytest

import oracle as O
from cism_amd import configs, gpu as G
from helpers import assembled_system, rel_l2

pytestmark = pytest.mark.gpu

SIZES = {                                # nodes nz (ewn + 3) (nsn + 3) in blocks of 256
    "64_blocks": (61, 61, 4),
    "65_blocks": (62, 61, 4),
    "512_blocks": (125, 125, 8),
    "513_blocks": (190, 167, 4),
    "516_blocks": (126, 125, 8),
    "1041_update_blocks": (254, 256, 2),
    "2105_update_blocks": (364, 364, 2),
}


@pytest.fixture(scope="module", params=list(SIZES))
def system(request):
    ewn, nsn, nz = SIZES[request.param]
    p = configs.grf_sheet(ewn=ewn, nsn=nsn, nz=nz, seed=8)
    blocks = -(-nz * (ewn + 3) * (nsn + 3) // 256)
    columns = -(-(ewn + 3) * (nsn + 3) // 64)
    assert str(columns if "update" in request.param else blocks) == request.param.split("_")[0]
    return (p,) + assembled_system(p, seed=5)[:5]


@pytest.mark.parametrize("chrongear,precond,its", [(True, 2, 12), (True, 1, 12), (False, 1, 12), (False, 0, 11),
                                                   (False, 2, 11)])
def test_iterates_match_oracle(system, chrongear, precond, its):
    p, A, bu, bv, u, v = system
    print(f"[cg] {p.ewn}x{p.nsn}x{p.nz} chrongear {chrongear} precond {precond}", flush=True)
    ou, ov, gu, gv = (a.copy(order="F") for a in (u, v, u, v))
    st, _, nit_o = O.pcg(p, A, bu, bv, ou, ov, precond, chrongear=chrongear, maxiters=its)
    assert st == 0
    with G.Context.for_problem(p) as ctx:
        ctx.set_linear_solver(its, 1e-8)
        f = ctx.pcg_solver_chrongear_3d if chrongear else ctx.pcg_solver_standard_3d
        _, nit_g = f(p.active_vertex, *A, bu, bv, gu, gv, precond)
    assert nit_g == nit_o
    x_o, x_g = (np.concatenate([a.ravel(), b.ravel()]) for a, b in ((ou, ov), (gu, gv)))
    assert rel_l2(x_g, x_o) < 1e-11
