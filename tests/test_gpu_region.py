"""The one-launch solve (region_kernels.hpp), which FIM solves of grids that
fit the device's LDS take, against the pass solver on the same inputs: AGSI
solves run there, with the same scheme and tolerances.  Sizes sit on the edges
of tiles and boxes, and dimensions, types, walls and periodic axes select each
form of the set-up.

Bar: both stop at changes below atol + rtol |u| = 1e-6 (FP32) or 1e-12 (FP64)
of values of order 1, and a value inherits what its upwind neighbours left
unannounced, tile after tile: with at most 40 tiles along a path, 1e-4 and
1e-10 of max u; identical finite masks.
"""
import numpy as np
import pytest

from adaptivegriddiscretizations_amd import Eikonal, Metrics, workloads
from gpu_helpers import log

pytestmark = pytest.mark.gpu


def _metric(rng, d, dims):
    a = rng.normal(size=(d, d) + dims).astype(np.float32) * 0.4
    return np.einsum('ij...,kj...->ik...', a, a) + np.eye(d, dtype=np.float32).reshape((d, d) + (1,) * d)


def _solve(model, dims, solver, seed=1, fp64=False, walls=False, periodic=None, nseeds=2, **extra):
    rng = np.random.default_rng(seed)
    d = len(dims)
    h = Eikonal.dictIn({'model': model, 'exportValues': True, 'verbosity': 0, 'solver': solver, **extra})
    h.SetRect([[0, n / 16.] for n in dims], dims=list(dims))
    cells = np.stack([rng.integers(0, n, nseeds) for n in dims], 1)
    h['seeds'] = ((cells + 0.5) / 16.).astype(np.float32)
    h['seedValues'] = -0.1 * np.arange(nseeds)
    if model[:-1] == 'Diagonal':
        h['metric'] = Metrics.Diagonal(rng.uniform(0.5, 2, (d,) + dims).astype(np.float32))
    elif model[:-1] == 'Riemann':
        h['metric'] = Metrics.Riemann(_metric(rng, d, dims))
    elif model[:-1] == 'Rander':
        h['metric'] = Metrics.Rander(_metric(rng, d, dims), rng.uniform(-.3, .3, (d,) + dims).astype(np.float32))
    h['cost'] = rng.uniform(0.7, 1.3, dims).astype(np.float32)
    if walls:
        w = rng.random(dims) < 0.2
        w[tuple(cells.T)] = False
        h['walls'] = w
    if periodic:
        h['periodic'] = periodic
    tol = 1e-12 if fp64 else 1e-6
    h['atol'] = h['rtol'] = tol
    if fp64:
        h['values_float64'] = True
    return h.Run()


@pytest.mark.parametrize("model,dims,options", [
    ('Isotropic2', (1, 1), {'nseeds': 1}),
    ('Isotropic2', (8, 33), {}),
    ('Isotropic2', (250, 129), {'walls': True}),
    ('Diagonal2', (65, 31), {'periodic': (True, False)}),
    ('Riemann2', (97, 40), {'fp64': True}),
    ('Riemann2', (63, 64), {'fp64': True, 'walls': True, 'periodic': (True, True)}),
    ('Riemann2', (45, 70), {'fp64': True}),
    ('Rander2', (100, 31), {'fp64': True}),
    ('Rander2', (33, 32), {'fp64': True, 'walls': True}),
    ('Isotropic3', (17, 9, 70), {'walls': True}),
    ('Isotropic3', (8, 8, 16), {'fp64': True}),
    ('Diagonal3', (5, 31, 20), {'periodic': (False, True, True)}),
    ('Riemann3', (37, 21, 30), {}),
    ('Riemann3', (12, 13, 20), {'fp64': True, 'periodic': (True, False, False)}),
    ('Rander3', (20, 18, 13), {}),
])
def test_one_launch_solve_matches_pass_solver(model, dims, options):
    log(f"one-launch solve {model} {dims} {options}")
    a = _solve(model, dims, 'FIM', **options)
    b = _solve(model, dims, 'AGSI', **options)
    u, v = (x['values'].cpu().numpy().astype(np.float64) for x in (a, b))
    assert a['stats']['eikonal']['converged'] == 1
    fin = np.isfinite(v)
    assert np.array_equal(fin, np.isfinite(u))
    err = np.max(np.abs(u - v)[fin]) / max(np.max(np.abs(v[fin])), 0.1)
    log(f"  rel diff {err:.2e}")
    assert err <= (1e-10 if options.get('fp64') else 1e-4)


@pytest.mark.parametrize("model", ['TTI2', 'ReedsShepp2', 'ReedsSheppForward2', 'Elastica2', 'Dubins2'])
def test_one_launch_stored_schemes_match_pass_solver(model):
    log(f"one-launch solve {model}")
    wl = workloads.tti_tilted(n=45, d=2) if model == 'TTI2' else workloads.curvature2(model, n=20, ntheta=18)
    u, v = (wl.dict_in(exportValues=True, solver=s, atol=1e-6, rtol=1e-6).Run()['values'].cpu().numpy()
            for s in ('FIM', 'AGSI'))
    fin = np.isfinite(v)
    assert np.array_equal(fin, np.isfinite(u))
    # (the far, barely reachable states of the forward models lose FP32 digits
    # in either order: 4e-4 of them at most, as in the tests of those models)
    err = np.max(np.abs(u - v)[fin]) / np.max(v[fin])
    log(f"  rel diff {err:.2e}")
    assert err <= 4e-4


def test_a_bounded_number_of_passes_is_counted_in_passes():
    """nitermax_o below its default selects the pass solver: the bound is on passes."""
    with pytest.raises(ValueError, match="convergence"):
        _solve('Riemann3', (37, 21, 30), 'FIM', nitermax_o=3, check_interval=1)


def test_solve_continues_from_given_values():
    a = _solve('Riemann3', (37, 21, 30), 'FIM')
    u = a['values'].cpu().numpy()
    b = _solve('Riemann3', (37, 21, 30), 'FIM', values=(u + 0.3).astype(np.float32), warmStartAllTiles=True)
    assert np.max(np.abs(b['values'].cpu().numpy() - u)) <= 1e-4 * np.max(np.abs(u))


@pytest.mark.parametrize("model,fp64", [('Isotropic2', False), ('Riemann2', True)])
def test_nan_seed_stays_and_blocks_as_in_the_pass_solver(model, fp64):
    """A seed of value NaN keeps it, and a cell that reads it is not updated."""
    rng = np.random.default_rng(4)
    dims = (40, 33)
    out = {}
    for solver in ('FIM', 'AGSI'):
        h = Eikonal.dictIn({'model': model, 'exportValues': True, 'verbosity': 0, 'solver': solver})
        h.SetRect([[0, n / 16.] for n in dims], dims=list(dims))
        h['seeds'] = ((np.array([[4, 5], [30, 20]]) + 0.5) / 16.).astype(np.float32)
        h['seedValues'] = np.array([0., np.nan])
        if model == 'Riemann2':
            h['metric'] = Metrics.Riemann(_metric(np.random.default_rng(5), 2, dims))
        h['cost'] = np.ones(dims, np.float32)
        if fp64:
            h['values_float64'] = True
        out[solver] = h.Run()['values'].cpu().numpy()
    u, v = out['FIM'], out['AGSI']
    assert np.isnan(u[30, 20]) and np.isnan(v[30, 20])
    assert np.array_equal(np.isnan(u), np.isnan(v)) and np.array_equal(np.isinf(u), np.isinf(v))
