"""Layout kernels for every form of their index arithmetic (tiles of powers of
two that fill waves or not, other tiles) against the numpy restatement of the
tiled layout: moves are exact, the geometry is computed in double and rounded
once."""
import numpy as np
import pytest

from adaptivegriddiscretizations_amd import FiniteDifferences as fd
from adaptivegriddiscretizations_amd import _lib
from gpu_helpers import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,tile", [
    ((7,), (4,)), ((9, 17), (8, 8)), ((33, 16), (16, 16)), ((5, 13), (4, 8)), ((10, 11), (3, 5)),
    ((9, 6, 7), (4, 4, 4)), ((8, 17, 5), (8, 8, 4)), ((6, 7, 8), (2, 3, 4)), ((1, 1, 1), (4, 4, 8))])
@pytest.mark.parametrize("dtype", [np.uint8, np.float32, np.float64])
def test_expand_and_squeeze(shape, tile, dtype):
    import torch
    log(f"layout {shape} in {tile} {np.dtype(dtype).name}")
    rng = np.random.default_rng(0)
    src = rng.integers(0, 200, (2,) + shape).astype(dtype)
    so = fd.round_up_ratio(shape, tile)
    size = int(np.prod(so) * np.prod(tile))
    ref = np.full((2, size), 7, dtype)
    idx = fd.tiled_index(np.stack(np.meshgrid(*map(np.arange, shape), indexing='ij'), -1), tile, so)
    for c in range(2):
        ref[c][idx] = src[c]
    a = torch.from_numpy(src).cuda()
    t = torch.empty((2, size), dtype=a.dtype, device='cuda')
    back = torch.empty_like(a)
    n, es = len(shape), np.dtype(dtype).itemsize
    L = _lib.lib
    _lib.check(L.agd_block_expand(n, _lib.i64(shape), _lib.i32(tile), 2, es, a.data_ptr(), 1, t.data_ptr(), 7., None))
    _lib.check(L.agd_block_squeeze(n, _lib.i64(shape), _lib.i32(tile), 2, es, t.data_ptr(), back.data_ptr(), None))
    torch.cuda.synchronize()
    assert np.array_equal(t.cpu().numpy(), ref)
    assert np.array_equal(back.cpu().numpy(), src)


@pytest.mark.parametrize("shape,tile", [((9, 17), (8, 8)), ((5, 6), (4, 4)), ((7, 7), (3, 5)), ((5, 9, 6), (4, 4, 4))])
@pytest.mark.parametrize("const", [False, True])
def test_riemann_geometry(shape, tile, const):
    import torch
    d = len(shape)
    log(f"geometry {shape} in {tile} constant {const}")
    rng = np.random.default_rng(1)
    a = rng.normal(size=(() if const else shape) + (d, d))
    m = np.moveaxis(a @ np.swapaxes(a, -1, -2) + 0.3 * np.eye(d), (-2, -1), (0, 1)).astype(np.float32)
    h = np.array([0.1, 0.25, 0.3])[:d]
    D = np.linalg.inv(np.moveaxis(m.astype(np.float64), (0, 1), (-2, -1)) * h[:, None] * h)
    low = np.stack([np.broadcast_to(D[..., i, j], shape) for i in range(d) for j in range(i + 1)])
    so = fd.round_up_ratio(shape, tile)
    size = int(np.prod(so) * np.prod(tile))
    idx = fd.tiled_index(np.stack(np.meshgrid(*map(np.arange, shape), indexing='ij'), -1), tile, so)
    import ctypes
    m_d = torch.from_numpy(np.ascontiguousarray(m)).cuda()
    g = torch.empty((len(low), size), dtype=torch.float32, device='cuda')
    _lib.check(_lib.lib.agd_prepare_geometry(
        _lib.RIEMANN, d, _lib.i64(shape), _lib.i32(tile), _lib.F32, (ctypes.c_double * 3)(*h, *[1.] * (3 - d)),
        m_d.data_ptr(), None, 0 if const else 1, g.data_ptr(), None))
    torch.cuda.synchronize()
    g = g.cpu().numpy()
    # cofactors in double: relative error below cond(m) 1e-15 < 1e-9, then one rounding to FP32
    assert np.max(np.abs(g[:, idx] - low) / np.abs(D).max()) <= 2 ** -23
    pad = np.ones(size, bool)
    pad[idx] = False
    assert np.all(np.isinf(g[:, pad]))


@pytest.mark.parametrize("tile", [(4, 4, 4), (3, 4, 5)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_spread_fields(tile, dtype):
    """A constant, a plane, a line and a full field, spread and rounded exactly."""
    import ctypes
    import torch
    shape = (5, 9, 6)
    log(f"spread {shape} in {tile} {np.dtype(dtype).name}")
    rng = np.random.default_rng(2)
    parts = [rng.normal(size=s) for s in ((1, 1, 1), (5, 9, 1), (1, 1, 6), shape)]
    so = fd.round_up_ratio(shape, tile)
    size = int(np.prod(so) * np.prod(tile))
    idx = fd.tiled_index(np.stack(np.meshgrid(*map(np.arange, shape), indexing='ij'), -1), tile, so)
    ref = np.full((4, size), -1, dtype)
    for c, p in enumerate(parts):
        ref[c][idx] = np.broadcast_to(p, shape).astype(dtype)
    src = torch.from_numpy(np.concatenate([p.reshape(-1) for p in parts])).cuda()
    offset = np.concatenate([[0], np.cumsum([p.size for p in parts])])[:4].tolist()
    stride = sum([[s // 8 if n > 1 else 0 for s, n in zip(p.strides, p.shape)] for p in parts], [])
    out = torch.empty((4, size), dtype=torch.float32 if dtype == np.float32 else torch.float64, device='cuda')
    _lib.check(_lib.lib.agd_spread_fields(
        3, _lib.i64(shape), _lib.i32(tile), 4, _lib.F32 if dtype == np.float32 else _lib.F64, src.data_ptr(),
        (ctypes.c_int64 * 4)(*offset), (ctypes.c_int64 * 12)(*stride), out.data_ptr(), -1., None))
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), ref)
