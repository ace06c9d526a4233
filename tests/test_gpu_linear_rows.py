"""Linear systems over made-up flow graphs, whose rows are of any length: none,
fewer than the entries held in registers, more than those ranked there; sources
inside and outside the tile; the same source twice.  Against the substitution
in 64 bits.

Bar: a value is a sum of up to 200 positive terms along chains of at most 40
cells, each rounded once: 40 * 200 * 2^-24 = 5e-4 of it in FP32 at the very
worst, and 1e-12 in FP64; the iterations stop at atol = 0, rtol = 0, that is
when nothing changes.
"""
import numpy as np
import pytest
import torch

from adaptivegriddiscretizations_amd import FiniteDifferences as FD
from adaptivegriddiscretizations_amd import _lib
from adaptivegriddiscretizations_amd.Eikonal._device import ptr
from gpu_helpers import log

pytestmark = pytest.mark.gpu


def _graph(rng, shape, tile, nsym, hubs):
    """Upwind neighbours of lower row number (first axis) within reach of the
    next tile; with hubs, all of a row's cells that can do so choose one of a few."""
    so = FD.round_up_ratio(np.array(shape), np.array(tile))
    N = int(np.prod(so) * np.prod(tile))
    fw = np.zeros((nsym, N))
    fi = np.full((nsym, N), np.iinfo(np.int32).max, np.int32)
    order = []
    for x in np.ndindex(*shape):
        n = int(FD.tiled_index(np.array(x), tile, so))
        order.append(n)
        for k in range(nsym):
            if x[0] == 0 or rng.random() < 0.2:
                continue
            y = [x[0] - int(rng.integers(1, min(x[0], 3) + 1))]
            for c in range(1, len(shape)):  # (the tile of x: marks go to face neighbours)
                lo, hi = x[c] // tile[c] * tile[c], min(x[c] // tile[c] * tile[c] + tile[c], shape[c])
                y.append(min(lo + 3, hi - 1) if hubs else int(rng.integers(lo, hi)))
            fi[k, n] = FD.tiled_index(np.array(y), tile, so)
            fw[k, n] = rng.uniform(0.02, 0.1) if hubs else rng.uniform(0.1, 1.)
    return fw, fi, np.array(order)


@pytest.mark.parametrize("shape,tile", [((40, 21), (8, 8)), ((33, 30), (16, 16)), ((14, 9, 13), (4, 4, 4)),
                                        ((11, 9, 13), (8, 8, 4))])
@pytest.mark.parametrize("hubs", [False, True])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("forward", [False, True])
def test_linear_system_matches_substitution(shape, tile, hubs, dtype, forward):
    rng = np.random.default_rng(2)
    d = len(shape)
    nsym = {2: 3, 3: 6}[d]  # of Riemann
    fw, fi, order = _graph(rng, shape, tile, nsym, hubs)
    fw = fw.astype(dtype).astype(np.float64)
    N = fw.shape[1]
    wsum = (0.5 + fw.sum(0)).astype(dtype)
    rhs = rng.uniform(0.5, 1.5, N).astype(dtype)
    u = np.full(N, np.inf, dtype)
    u[order] = 1.
    ref = rhs.astype(np.float64)
    edge = fi != np.iinfo(np.int32).max
    indeg = np.bincount(fi[edge], minlength=N)
    log(f"linear rows {shape} {tile} hubs {hubs} {np.dtype(dtype).name}: longest row {indeg.max()}")
    assert not hubs or indeg.max() > 16
    if forward:
        for n in order:
            ref[n] = (ref[n] + sum(fw[k, n] * ref[fi[k, n]] for k in range(nsym) if edge[k, n])) / wsum[n]
    else:
        for n in order[::-1]:
            ref[n] /= wsum[n]
            for k in range(nsym):
                if edge[k, n]:
                    ref[fi[k, n]] += fw[k, n] * ref[n]
    desc = _lib.EikonalDesc()
    desc.model, desc.ndim = _lib.RIEMANN, d
    desc.scalar = int(dtype == np.float64)
    for k in range(3):
        desc.shape[k], desc.shape_i[k] = (shape[k], tile[k]) if k < d else (1, 1)
    desc.niter_i, desc.nitermax_o, desc.check_interval, desc.use_graph = 8, 2000, 8, 1
    g = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda()
         for k, v in dict(u=u, fw=fw.astype(dtype), fi=fi, wsum=wsum, rhs=rhs).items()}
    sol = torch.empty(N, dtype=g['u'].dtype, device='cuda')
    fn = _lib.lib.agd_eikonal_forward_ad if forward else _lib.lib.agd_eikonal_adjoint
    stats = _lib.EikonalStats()
    _lib.check(fn(desc, ptr(g['u']), ptr(g['fw']), ptr(g['fi']), ptr(g['wsum']), 1, ptr(g['rhs']), ptr(sol), 0., 0.,
                  stats, torch.cuda.current_stream().cuda_stream))
    assert stats.converged
    got = sol.cpu().numpy()[order]
    err = np.max(np.abs(got - ref[order]) / ref[order])
    log(f"  rel err {err:.2e}")
    assert err <= (5e-4 if dtype == np.float32 else 1e-12)
