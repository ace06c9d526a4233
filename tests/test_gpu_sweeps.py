"""The pass solver (AGSI solves run there) against the default solve of the
same problem.  In-tile sweeps: odd and even numbers of them, tiles of one wave
and of several, with and without shifts of the neighbour values.  Stencils
stored on the way, after an eighth of the tiles' number of visits.

Bar: both stop at changes below atol + rtol |u| = 1e-6 (FP32) or 1e-12 (FP64)
of values of order 1, and a value inherits what its upwind neighbours left
unannounced, tile after tile: with at most 40 tiles along a path, 1e-4 and
1e-10 of max u; identical finite masks.
"""
import numpy as np
import pytest

from gpu_helpers import log
from test_gpu_region import _solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,dims,shape_i,options", [
    ('Isotropic2', (61, 50), (8, 8), {}),
    ('Isotropic2', (61, 50), (16, 16), {'walls': True}),
    ('Riemann2', (40, 33), (8, 16), {'fp64': True}),
    ('Riemann2', (40, 33), (16, 16), {'periodic': (True, False)}),
    ('Rander2', (33, 47), (8, 8), {}),
    ('Rander2', (33, 47), (16, 16), {'fp64': True}),
    ('Riemann3', (13, 18, 9), (4, 4, 4), {}),
    ('Riemann3', (13, 18, 9), (8, 8, 4), {}),
    ('Isotropic3', (13, 18, 9), (4, 4, 8), {'walls': True, 'fp64': True}),
])
@pytest.mark.parametrize("niter_i", [1, 2, 5])
def test_sweeps_match_default_solve(model, dims, shape_i, options, niter_i):
    log(f"sweeps {model} {dims} {shape_i} {options} niter_i {niter_i}")
    a = _solve(model, dims, 'AGSI', traits={'shape_i': shape_i, 'niter_i': niter_i}, **options)
    b = _solve(model, dims, 'FIM', **options)
    u, v = (x['values'].cpu().numpy().astype(np.float64) for x in (a, b))
    fin = np.isfinite(v)
    assert np.array_equal(fin, np.isfinite(u))
    err = np.max(np.abs(u - v)[fin]) / np.max(np.abs(v[fin]))
    log(f"  rel diff {err:.2e}")
    assert err <= (1e-10 if options.get('fp64') else 1e-4)


@pytest.mark.parametrize("model,dims,options", [
    ('Riemann2', (9, 5), {}),      # four tiles: stored after the first visit
    ('Riemann2', (150, 97), {'walls': True, 'periodic': (False, True)}),
    ('Riemann2', (64, 130), {'fp64': True, 'walls': True}),
    ('Riemann3', (21, 30, 17), {'walls': True}),
    ('Riemann3', (16, 22, 12), {'fp64': True, 'periodic': (True, False, True)}),
])
@pytest.mark.parametrize("solver", ['AGSI', 'global_iteration'])
def test_stored_stencils_match_rebuilt_ones(model, dims, options, solver):
    """Without passes queued ahead, stencils are rebuilt at every visit."""
    log(f"stored stencils {model} {dims} {solver} {options}")
    a = _solve(model, dims, solver, **options)
    b = _solve(model, dims, solver, hipGraph=False, **options)
    u, v = (x['values'].cpu().numpy().astype(np.float64) for x in (a, b))
    fin = np.isfinite(v)
    assert np.array_equal(fin, np.isfinite(u))
    err = np.max(np.abs(u - v)[fin]) / np.max(np.abs(v[fin]))
    log(f"  rel diff {err:.2e}")
    assert err <= (1e-10 if options.get('fp64') else 1e-4)
