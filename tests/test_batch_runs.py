"""Batched solves whose vectors stop at different times, so that the launches go
over several runs of live vectors: a zero load (never live) in the middle, loads
that take different numbers of iterations around it. Each displacement and
iteration count is, bit for bit, that of the load solved as a batch of one, on
rows of one, two and part of a wave, on rows whose last node goes with the last pair in
the batch and by itself alone, on a box deeper than one plane block and on rows longer
than a workgroup."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(128, 24, 40), (128, 32, 40), (90, 41, 37), (12, 12, 100), (63, 9, 7)])
def test_runs_of_live_vectors(size):
    check_runs(size, 1e-7, 1000)


def test_runs_on_long_rows():
    """513 pairs a row, whose sweeps the pair kernel makes; a slender beam, stopped after 40 iterations."""
    check_runs((1024, 8, 8), 1e-3, 40)


def check_runs(size, tol, maxit):
    from bench import build_problem
    print(f"[batch runs] {size}", flush=True)
    hg, bits, R, fixed, f, rho = build_problem(*size, 1)
    hg.update_stencil()
    _, vact = hg[0].masks()
    free = (vact & ~fixed.astype(bool))[None]
    rng = np.random.default_rng(4)
    F = np.stack([f, rng.standard_normal(f.shape) * free, np.zeros_like(f), free * np.ones_like(f),
                  rng.standard_normal(f.shape) * free * (rng.random(f.shape) < 0.01), np.zeros_like(f), -2 * f])
    U, it, rel = hg.solve_batch(F, tol=tol, maxit=maxit)
    assert it[2] == 0 and it[5] == 0 and not U[2].any() and not U[5].any()
    print(f"[batch runs] iterations {it.tolist()}", flush=True)
    for b in range(len(F)):
        U1, it1, rel1 = hg.solve_batch(F[b:b + 1], tol=tol, maxit=maxit)
        assert it1[0] == it[b], b
        assert np.array_equal(U1[0], U[b]), b
    hg.close()
