"""Cluster labels on rows longer than one wave's 64-element segment, on rows
that end inside one, and on densities sparse and dense enough that runs start
and end at every place of a segment: the number of floating clusters equals that
of scipy.ndimage.label's 6-connected components that touch no support."""
import numpy as np
import pytest
from scipy.ndimage import label

import robtop_amd as rt
from robtop_amd.workloads import cube_bits, cube_side

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ex,ey,ez,p", [(63, 9, 7, 0.4), (64, 8, 8, 0.25), (65, 7, 9, 0.6), (130, 11, 5, 0.35),
                                        (200, 3, 13, 0.5), (9, 40, 33, 0.3), (9, 9, 70, 0.75)])
def test_labels_of_split_rows(ex, ey, ez, p):
    print(f"[island rows] {ex}x{ey}x{ez} p {p}", flush=True)
    R = cube_side(ex, ey, ez)
    a = np.zeros((R, R, R), bool)
    a[:ex, :ey, :ez] = True
    hg = rt.HierarchyGrid.genFromMesh(cube_bits(a), R)
    hg.set_material(1e6, 0.4, 3.0)
    nx, ny, nz = hg[0].nodes
    eact, vact = hg[0].masks()
    fixed = np.zeros((nz, ny, nx), bool)
    fixed[:, :, 0] = True
    hg.set_support(fixed.reshape(-1) & vact)
    box = eact.reshape(nz - 1, ny - 1, nx - 1)
    stiff = (np.random.default_rng(ex + ey).random(box.shape) < p) & box
    hg.set_density((np.where(stiff, 1.0, 1e-3) * box).reshape(-1).astype(np.float32))
    hg.update_stencil()
    lab, n = label(stiff)
    held = set(np.unique(lab[:, :, 0]))
    sizes = np.bincount(lab.ravel(), minlength=n + 1)
    for min_size in (1, 2, 9, 400):
        hg.set_island_deflation(0.5, min_size)
        want = sum(1 for c in range(1, n + 1) if c not in held and sizes[c] >= min_size)
        assert want < 4096
        assert hg.num_islands() == want, min_size
    hg.close()
