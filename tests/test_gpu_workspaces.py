"""Workspaces kept between calls: handles alive at the same time never share
one, a kept one serves grids of other sizes and other entry points, and
releasing them gives the memory back without harm to later calls."""
import gc

import numpy as np
import pytest

from adaptivegriddiscretizations_amd import _lib, workloads
from gpu_helpers import log, oracle_problem, rel_err, run_gpu

pytestmark = pytest.mark.gpu


def _prepare(wl, **extra):
    from adaptivegriddiscretizations_amd.Eikonal import HFM_GPU
    iface = HFM_GPU.Interface(wl.dict_in(**extra))
    iface.SetKernelTraits()
    iface.SetGeometry()
    iface.SetArgs()
    return iface


def test_workspaces_are_reused_and_released(O):
    sizes = (40, 90, 24)
    refs = {}
    for n in sizes:
        P, _ = oracle_problem(O, workloads.riemann2_aniso(n=n, seed=n, sigma=4., amax=5.))
        refs[n] = P.solve_fm()
    for solver in ('FIM', 'AGSI'):
        for n in sizes:
            log(f"reuse {n}^2 {solver}")
            wl = workloads.riemann2_aniso(n=n, seed=n, sigma=4., amax=5.)
            u, _ = run_gpu(wl, solver=solver, sensitivity=np.ones(wl.dims + (1,), np.float32))
            assert rel_err(u, refs[n]) <= 1e-4
    gc.collect()
    assert _lib.release_workspaces() > 0
    assert _lib.release_workspaces() == 0
    u, _ = run_gpu(workloads.riemann2_aniso(n=40, seed=40, sigma=4., amax=5.))
    assert rel_err(u, refs[40]) <= 1e-4


def test_handles_alive_at_once_do_not_share(O):
    """Six handles (more than are kept), solved in turn and again in reverse:
    each reaches its own problem's answer both times."""
    import torch
    its = [_prepare(workloads.isotropic2_bumps(n=32 + 9 * i, seed=i)) for i in range(6)]
    handles = [_lib.Solver(it.stream, it._desc()) for it in its]
    refs = []
    for i in range(6):
        P, _ = oracle_problem(O, workloads.isotropic2_bumps(n=32 + 9 * i, seed=i))
        refs.append(P.solve_fm())
    for order in (range(6), reversed(range(6))):
        for i in order:
            its[i].values_t.fill_(float('inf'))
            its[i]._values = None
            _lib.check(handles[i].solve(its[i]._desc(), its[i]._io(), _lib.EikonalStats()))
            torch.cuda.synchronize()
            assert rel_err(its[i].values.cpu().numpy().astype(np.float64), refs[i]) <= 1e-4
    for h in handles:
        h.close()


def test_failed_call_leaves_later_ones_alone(O):
    wl = workloads.riemann2_aniso(n=60, seed=3, sigma=4., amax=5.)
    with pytest.raises(ValueError, match="convergence"):
        run_gpu(wl, nitermax_o=2)
    P, _ = oracle_problem(O, wl)
    u, _ = run_gpu(wl)
    assert rel_err(u, P.solve_fm()) <= 1e-4
