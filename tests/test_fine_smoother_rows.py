"""The finest smoother's row kernel (one thread per even / odd pair of a row)
against the tiled smoother, which computes each node by itself: the same bits,
at the row lengths where the row kernel's workgroups differ: rows of one node
more than whole waves with and without enough rows to give the node left over
to the last pair's thread, several rows to a workgroup, rows of part of a wave;
and where the pair kernel takes over, rows of five waves in FP64 and rows longer
than a workgroup; with holes and with supports inside the solid, so that
neighbour checks run."""
import numpy as np
import pytest

from robtop_amd.workloads import cube_bits, cube_side

SHAPES = [
    (128, 96, 96),      # 65 pairs, 2,401 rows a launch: the 65th node goes with the last pair
    (128, 32, 32),      # 65 pairs, few rows: two waves a row
    (80, 112, 112),     # 41 pairs, three rows a workgroup
    (56, 24, 40),       # 29 pairs, one wave a row
    (384, 64, 64),      # 193 pairs: in FP32 the 193rd node goes with the last pair, in FP64 it has a wave
]
LONG = [
    (640, 16, 16),      # 321 pairs, six waves
    (544, 16, 16),      # 273 pairs, five waves: the pair kernel in FP64
    (1024, 8, 8),       # 513 pairs: the pair kernel
]


def problem(ex, ey, ez, seed):
    import robtop_amd as rt
    R = cube_side(ex, ey, ez)
    a = np.zeros((R, R, R), bool)
    a[:ex, :ey, :ez] = True
    a[ex // 3:ex // 3 + 3, ey // 2:, :ez // 2] = False
    a[ex - 1, :, ez // 4] = False
    hg = rt.HierarchyGrid.genFromMesh(cube_bits(a), R)
    hg.set_material(1e6, 0.4, 3.0)
    nx, ny, nz = hg[0].nodes
    _, vact = hg[0].masks()
    rng = np.random.default_rng(seed)
    fixed = np.zeros((nz, ny, nx), bool)
    fixed[:, :, 0] = True
    fixed[nz // 2, ny // 2, 5:9] = True
    fixed[1, 1, nx - 2:] = True
    fixed = fixed.reshape(-1) & vact
    hg.set_support(fixed)
    eact, _ = hg[0].masks()
    hg.set_density((rng.uniform(0.1, 1.0, eact.size) * eact).astype(np.float32))
    f = rng.standard_normal((3, vact.size)) * (vact & ~fixed)
    u = rng.standard_normal((3, vact.size)) * vact
    return hg, f, u


def check_sweeps(hg, f, u, bits):
    hg.set_precision(bits)
    out = {}
    for kind in (0, 1):
        hg.set_fine_smoother(kind)
        g = hg[0]
        g.setForce(f)
        g.setDisplacement(u)
        g.gs_relax(1)
        fwd = g.getDisplacement()
        g.gs_relax(2, reverse=True)
        out[kind] = (fwd, g.getDisplacement())
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
    assert not np.array_equal(out[0][0], u)


def check_cycles(hg, f):
    """Zero supports, zero start and reverse sweeps: the FP64 PCG's iterates."""
    import robtop_amd as rt
    out = []
    for kind in (0, 1):
        hg.set_fine_smoother(kind)
        hg.set_displacement(np.zeros_like(f))
        hg.solve(tol=0.0, maxit=3, mode=rt.RT_SOLVE_FP64, pre=2, post=2)
        out.append(hg.get_displacement())
    assert np.array_equal(out[0], out[1])


def check_rz(hg, f):
    """r.z summed by the last sweep of each cycle against the separate pass over r and z that goes with the tiled
    smoother, through the first step length: the same terms in another order (1e-9: 4 M products summed in FP64). The
    next ones see FP32 vectors that may differ in their last places."""
    import robtop_amd as rt
    out = []
    for kind in (0, 1):
        hg.set_fine_smoother(kind)
        hg.set_displacement(np.zeros_like(f))
        hg.solve(tol=0.0, maxit=4, mode=rt.RT_SOLVE_RELIABLE, pre=2, post=2)
        out.append(hg.cg_coefficients())
    (a0, b0), (a1, b1) = out
    assert len(a0) == len(a1) == 4 and abs(a0[0] - a1[0]) <= 1e-9 * a1[0]
    assert np.allclose(a0, a1, rtol=1e-4, atol=0) and np.allclose(b0[:3], b1[:3], rtol=1e-4, atol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("bits", [32, 64])
def test_sweeps_equal_the_tiled_smoother(shape, bits):
    print(f"[rows] sweeps {shape} {bits}", flush=True)
    hg, f, u = problem(*shape, 1)
    check_sweeps(hg, f, u, bits)
    hg.close()


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_preconditioner_sweeps_equal_the_tiled_smoother(shape):
    print(f"[rows] cycles {shape}", flush=True)
    hg, f, _ = problem(*shape, 2)
    hg.set_force(f)
    hg.update_stencil()
    check_cycles(hg, f)
    check_rz(hg, f)
    hg.close()


@pytest.mark.gpu
@pytest.mark.parametrize("shape", LONG)
def test_long_rows_equal_the_tiled_smoother(shape):
    hg, f, u = problem(*shape, 1)
    for bits in (32, 64):
        print(f"[rows] sweeps {shape} {bits}", flush=True)
        check_sweeps(hg, f, u, bits)
    print(f"[rows] cycles {shape}", flush=True)
    hg.set_force(f)
    hg.update_stencil()
    check_cycles(hg, f)
    check_rz(hg, f)
    hg.close()


@pytest.mark.gpu
@pytest.mark.parametrize("shorter,longer,sizes", [((384, 64, 64), (448, 64, 64), (64,)),
                                                  ((640, 64, 64), (700, 64, 64), (32, 64))])
def test_a_shorter_row_takes_no_longer(shorter, longer, sizes):
    """Rows of one pair more than three or five whole waves: the workgroup shape must not cost more than rows that are
    longer still (a tenth for the timings' spread)."""
    import robtop_amd as rt
    from robtop_amd.workloads import box_bits
    print(f"[rows] sweep times {shorter} {longer}", flush=True)
    t = {}
    for s in (shorter, longer):
        R = cube_side(*s)
        hg = rt.HierarchyGrid.genFromMesh(box_bits(R, *s), R)
        hg.set_material(1e6, 0.4, 3.0)
        hg.init_rho(0.4)
        nx, ny, nz = hg[0].nodes
        fixed = np.zeros((nz, ny, nx), bool)
        fixed[:, :, 0] = True
        hg.set_support(fixed.reshape(-1) & hg[0].masks()[1])
        hg.update_stencil()
        for bits in sizes:
            hg.time_fine_sweep(bits, 20)
            t[s, bits] = min(hg.time_fine_sweep(bits, 20) for _ in range(5))
        hg.close()
    print({k: round(1e3 * v, 1) for k, v in t.items()}, flush=True)
    for bits in sizes:
        assert t[shorter, bits] <= 1.1 * t[longer, bits], bits
