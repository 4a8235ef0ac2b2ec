"""The V-cycle's coarse end in one workgroup (coarse.hip, k_cg_tail) against the numpy
restatement, at the hierarchies where its lanes and levels run out: 64 parents (every lane a
child) over a level that is itself smoothed, 40 parents (a level past the dense limit, ragged
both ways), a chain of aggregates one wide, and a level of more than 64 under which it starts.
FP32 against FP64: the bound of the correction's own test."""
import numpy as np
import pytest

from cism_amd import configs, gpu as G
from helpers import assembled_system, rel_l2
from test_gpu_coarse import Restated

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name, sizes", [
    ("full", [1024, 64, 4]),
    ("ragged", [551, 40, 4]),
    ("chain", [750, 63, 16]),
    ("above", [1156, 81, 9]),
])
def test_coarse_end(name, sizes):
    p = {"full": lambda: configs.grf_sheet(ewn=128, nsn=128, nz=3, seed=21),
         "ragged": lambda: configs.grf_sheet(ewn=112, nsn=75, nz=3, seed=22, periodic=False),
         "chain": lambda: configs.grf_sheet(ewn=12, nsn=1000, nz=3, seed=23),
         "above": lambda: configs.grf_sheet(ewn=136, nsn=135, nz=3, seed=24)}[name]()
    A = assembled_system(p, seed=5)[0]
    R = Restated(p, A)
    assert [l[0] * l[1] for l in R.levels] == sizes
    rng = np.random.default_rng(3)
    ru, rv = (np.asfortranarray(rng.standard_normal((p.nz, p.nx - 1, p.ny - 1))) for _ in range(2))
    z = R.correction(np.stack([ru[R.act], rv[R.act]], axis=1).ravel())
    print(f"[coarse end] {name} {sizes}", flush=True)
    with G.Context.for_problem(p) as ctx:
        assert ctx.coarse_build(p.active_vertex, p.umask_dirichlet, p.vmask_dirichlet, *A) == len(sizes)
        zu, zv = ctx.coarse_correction(ru, rv)
    err = rel_l2(np.stack([zu[R.act], zv[R.act]], axis=1).ravel(), z)
    print(f"  rel L2 diff {err:.2e}")
    assert err < 1e-4
