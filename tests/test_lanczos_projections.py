"""Block Lanczos with blocks of one vector, of fewer than a projection tile's
four columns, and of sizes that leave partial tiles, on a row count of a whole
chunk and a part of one: each finds the largest eigenvalue of the dense
compliance operator. With a Ritz residual of 1e-9 the eigenvalue's own error is
of its square; the solves' 1e-11 and the device's FP64 sums leave 1e-7 as the
bound that the block size 8 is held to as well."""
import numpy as np
import pytest

from problems import bits_of
from test_worst_case import _dense_top, _problem


@pytest.mark.gpu
@pytest.mark.parametrize("k", [1, 3, 5, 6])
def test_block_sizes_reach_the_dense_eigenvalue(k):
    import robtop_amd as rt
    a, H, fixed, rho, rhop, load, nrm, f0 = prob = _problem()
    print(f"[lanczos projections] k {k}, {int(load.sum())} load nodes", flush=True)
    g = rt.HierarchyGrid.genFromMesh(bits_of(a), 32)
    g.set_material(1e6, 0.4, 3.0)
    g.set_support(fixed)
    g.set_density(rho)
    g.update_stencil()
    g.set_load_nodes(load.astype(np.uint8), None)
    lam, ftop = _dense_top(prob, None, g.get_rhop())
    c, st = g.block_lanczos(k=k, max_blocks=60, tol=1e-9, solve_tol=1e-11, mode=rt.RT_SOLVE_FP64, seed=3)
    assert abs(c - lam) / lam < 1e-7, (c, lam, st)
    assert abs(abs(g.get_force().T.reshape(-1) @ ftop) - 1) < 1e-6
    g.close()
