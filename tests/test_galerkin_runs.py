"""The x2 Galerkin product (16 parent elements of a row at a time) against P^T A P
with scipy: rows of fewer parents than a run, of whole runs, and of a run and a part
of one, with holes and inactive elements at the boundary. Both sides are FP64 sums of
a few hundred products per entry; 1e-12 of the largest entry bounds their rounding."""
import numpy as np
import pytest
import scipy.sparse as sp

from robtop_amd.workloads import cube_bits, cube_side

pytestmark = pytest.mark.gpu


def matrix(g):
    """level matrix over all box nodes, from the stencils"""
    nx, ny, nz = (int(v) for v in g.nodes)
    st = g.getStencil()
    _, act = g.masks()
    v = np.nonzero(act)[0]
    x, y, z = v % nx, v // nx % ny, v // (nx * ny)
    rows, cols, vals = [], [], []
    for nb in range(27):
        jx, jy, jz = x + nb % 3 - 1, y + nb // 3 % 3 - 1, z + nb // 9 - 1
        ok = (jx >= 0) & (jx < nx) & (jy >= 0) & (jy < ny) & (jz >= 0) & (jz < nz)
        j = jx + nx * (jy + ny * jz)
        for r in range(3):
            for c in range(3):
                rows.append(3 * v[ok] + r)
                cols.append(3 * j[ok] + c)
                vals.append(st[nb, 3 * r + c, v[ok]])
    n = 3 * nx * ny * nz
    return sp.csr_matrix((np.concatenate(vals), (np.concatenate(rows), np.concatenate(cols))), (n, n))


def interpolation(nc):
    """trilinear, coarse nodes (nx, ny, nz) to twice the resolution, three components"""
    def line(n):
        m = sp.lil_matrix((2 * (n - 1) + 1, n))
        for i in range(2 * (n - 1) + 1):
            m[i, i // 2] = 1.0 if i % 2 == 0 else 0.5
            if i % 2:
                m[i, i // 2 + 1] = 0.5
        return m
    p = sp.kron(sp.kron(line(nc[2]), line(nc[1])), line(nc[0]))
    return sp.kron(p, sp.identity(3)).tocsr()


@pytest.mark.parametrize("size,hole", [((256, 24, 24), False), ((136, 48, 40), True), ((40, 24, 72), True),
                                       ((200, 20, 36), True)])
def test_second_coarse_level_is_the_galerkin_product(size, hole):
    import robtop_amd as rt
    print(f"[galerkin] {size}", flush=True)
    ex, ey, ez = size
    a = np.zeros((cube_side(*size),) * 3, bool)
    a[:ex, :ey, :ez] = True
    if hole:
        a[ex // 3:ex // 2, ey // 3:, :ez // 2] = False
    hg = rt.HierarchyGrid.genFromMesh(cube_bits(a), a.shape[0])
    hg.set_material(1e6, 0.4, 3.0)
    nx, ny, nz = hg[0].nodes
    eact, vact = hg[0].masks()
    fixed = np.zeros((nz, ny, nx), bool)
    fixed[:, :, 0] = True
    hg.set_support(fixed.reshape(-1) & vact)
    hg.set_density((np.random.default_rng(ex).uniform(0.1, 1.0, eact.size) * eact).astype(np.float32))
    hg.set_precision(64)
    hg.update_stencil()
    n1, n2 = [tuple(int(v) for v in hg[k].nodes) for k in (1, 2)]
    assert all(a == 2 * (b - 1) + 1 for a, b in zip(n1, n2))
    P = interpolation(n2)
    want = P.T @ matrix(hg[1]) @ P
    got = matrix(hg[2])
    _, act = hg[2].masks()
    keep = sp.diags(np.repeat(act, 3).astype(float))
    d = keep @ (want - got) @ keep
    assert abs(d).max() <= 1e-12 * abs(got).max()
    hg.close()
