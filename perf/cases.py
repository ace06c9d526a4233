"""The eikonal work that a user has this package do, as timed cases.

A case is one problem (or one batch of problems) with its inputs on the GPU,
solved through the public entry points: dictIn.Run(), autograd.eikonal_values
with its backward pass, or a prepared batch.Batch.  The listed cases span the
package's own benchmark and test configurations, from grids where a call is
mostly latency to the largest benchmark grids; draw() spreads over the same
ranges.  exact() solves the same discrete scheme in 64 bits with plain torch.

The second-order scheme is not among the cases: the limit of its decreasing
iteration depends on the schedule.  Geodesics are not either: their number of
points does.
"""
import math

import numpy as np
import torch

from adaptivegriddiscretizations_amd import Metrics
from adaptivegriddiscretizations_amd.Eikonal import autograd, batch, dictIn

XI = 0.3          # cost of rotation of the curvature-penalised models
EPS2 = 0.1 ** 2   # their relaxation (the solver's default eps = 0.1)
HEXAGONAL = (15., 4., 10., 3.)  # TTI material: c11, c13, c33, c44


def _case(name, model, n0, n1, n2=0, job='solve', seeds=1, flow=False, sens=False, walls=False, fp64=False):
    return {'name': name, 'job': job, 'model': model, 'n0': n0, 'n1': n1, 'n2': n2, 'seeds': seeds,
            'flow': flow, 'sens': sens, 'walls': walls, 'fp64': fp64}


def listed():
    return [
        # the smallest calls (interactive use, unit problems): latency and launches
        _case('isotropic2 61x48', 'Isotropic2', 61, 48),
        # the 2D benchmark image size, with the flow that path extraction reads
        _case('isotropic2 512 flow', 'Isotropic2', 512, 512, flow=True),
        # an image-sized anisotropic metric in FP64 arithmetic
        _case('riemann2 389x257 fp64', 'Riemann2', 389, 257, fp64=True),
        # the large 2D benchmark: 4 seeds, values and flow
        _case('riemann2 2000 flow', 'Riemann2', 2000, 2000, seeds=4, flow=True),
        # reverse differentiation of a drift model (2D navigation)
        _case('rander2 501x403 sensitivity', 'Rander2', 501, 403, seeds=2, sens=True),
        # motion planning around obstacles in a volume
        _case('isotropic3 121x77x95 walls', 'Isotropic3', 121, 77, 95, walls=True),
        # the 3D benchmark grid
        _case('riemann3 200', 'Riemann3', 200, 200, 200),
        # inversion: values and the gradient of a receiver loss, by autograd
        _case('riemann3 97x101x89 gradient', 'Riemann3', 97, 101, 89, job='gradient'),
        # seismic travel times in a tilted medium
        _case('tti2 301x263', 'TTI2', 301, 263),
        # vehicle planning: (x, y, theta) grids
        _case('reedssheppforward2 96x80x64', 'ReedsSheppForward2', 96, 80, 64),
        _case('elastica2 64x56x48', 'Elastica2', 64, 56, 48),
        # a prepared batch of many images, sides 64 to 1024, solved again and again
        _case('isotropic2 batch of 32', 'Isotropic2', 64, 1024, job='batch', seeds=32),
    ]


def draw(rng):
    def side(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(['isotropic2', 'riemann2', 'riemann2', 'rander2', 'isotropic3', 'riemann3', 'riemann3',
                       'gradient', 'tti', 'reedssheppforward2', 'elastica2', 'batch'])
    if kind == 'isotropic2':
        c = _case('', 'Isotropic2', side(48, 1024), side(48, 1024), seeds=rng.randint(1, 8), flow=rng.random() < .5)
    elif kind == 'riemann2':
        fp64 = rng.random() < .3
        top = 600 if fp64 else 2000
        c = _case('', 'Riemann2', side(100, top), side(100, top), seeds=rng.randint(1, 4), fp64=fp64,
                  flow=not fp64 and rng.random() < .5)
    elif kind == 'rander2':
        c = _case('', 'Rander2', side(100, 600), side(100, 600), seeds=rng.randint(1, 3), sens=rng.random() < .7)
    elif kind == 'isotropic3':
        c = _case('', 'Isotropic3', side(40, 150), side(40, 150), side(40, 150), walls=rng.random() < .7)
    elif kind == 'riemann3':
        c = _case('', 'Riemann3', side(40, 200), side(40, 200), side(40, 200), seeds=rng.randint(1, 3))
    elif kind == 'gradient':
        c = _case('', 'Riemann3', side(40, 110), side(40, 110), side(40, 110), job='gradient')
    elif kind == 'tti':
        c = _case('', 'TTI2', side(64, 320), side(64, 320)) if rng.random() < .6 else \
            _case('', 'TTI3', side(24, 48), side(24, 48), side(24, 48))
    elif kind == 'reedssheppforward2':
        c = _case('', 'ReedsSheppForward2', side(48, 112), side(48, 112), side(32, 72))
    elif kind == 'elastica2':
        c = _case('', 'Elastica2', side(32, 64), side(32, 64), side(32, 48))
    else:
        top = side(256, 1024)
        c = _case('', 'Isotropic2', 64, top, job='batch', seeds=rng.randint(8, 32))
    del c['name']
    return c


def _shape(case):
    return (case['n0'], case['n1']) + ((case['n2'],) if case['n2'] else ())


def _curvature(case):
    return case['model'] in ('ReedsSheppForward2', 'Elastica2')


# ------------------------------------------------------------------ inputs
def _smooth(gen, shape, sigma, lo, hi, normal=False):
    """Periodic Gaussian filtering of noise; mapped onto [lo, hi] unless normal."""
    dev = torch.device('cuda')
    f = (torch.randn if normal else torch.rand)(shape, generator=gen, device=dev)
    damp = torch.ones((), device=dev)
    for k, n in enumerate(shape):
        q = torch.fft.fftfreq(n, device=dev)
        s = min(sigma, n / 8.)
        damp = damp * torch.exp(-2. * (math.pi * s * q) ** 2).reshape((-1,) + (1,) * (len(shape) - 1 - k))
    f = torch.fft.ifftn(torch.fft.fftn(f) * damp).real
    if normal:
        return f
    f = (f - f.min()) / (f.max() - f.min())
    return lo + (hi - lo) * f


def _bumps(rng, shape):
    """Cost 1 + 0.5 tanh(sum of 32 Gaussian bumps) on [-1, 1]^2."""
    dev = torch.device('cuda')
    centres = torch.tensor(rng.uniform(-1, 1, (32, 2)), device=dev)
    widths = torch.tensor(rng.uniform(0.05, 0.2, 32), device=dev)
    amps = torch.tensor(rng.normal(size=32), device=dev)
    part = []
    for k in range(2):
        x = -1 + (torch.arange(shape[k], device=dev, dtype=torch.float64) + 0.5) * (2. / shape[k])
        part.append(torch.exp(-(x - centres[:, k:k + 1]) ** 2 / (2 * widths[:, None] ** 2)))
    g = (amps[:, None] * part[0]).T @ part[1]
    return (1 + 0.5 * torch.tanh(g)).float()


def _rotation3(q):
    r, i, j, k = q
    return torch.stack([torch.stack([1 - 2 * (j * j + k * k), 2 * (i * j - k * r), 2 * (i * k + j * r)]),
                        torch.stack([2 * (i * j + k * r), 1 - 2 * (i * i + k * k), 2 * (j * k - i * r)]),
                        torch.stack([2 * (i * k - j * r), 2 * (j * k + i * r), 1 - 2 * (i * i + j * j)])])


def _metric2(gen, shape):
    """R^T diag(1, a^2) R, smooth angle and log a in [0, ln 10]."""
    th = _smooth(gen, shape, 20., 0., math.pi)
    a2 = torch.exp(2 * _smooth(gen, shape, 20., 0., math.log(10.)))
    c, s = torch.cos(th), torch.sin(th)
    off = (a2 - 1) * s * c
    return torch.stack([torch.stack([c * c + a2 * s * s, off]), torch.stack([off, s * s + a2 * c * c])]).contiguous()


def _metric3(gen, shape):
    """Q diag(l) Q^T, smooth quaternion field, log l in [0, ln 5]."""
    q = torch.stack([_smooth(gen, shape, 10., 0, 0, normal=True) for _ in range(4)])
    rot = _rotation3(q / q.norm(dim=0))
    lam = torch.stack([torch.exp(_smooth(gen, shape, 10., 0., math.log(5.))) for _ in range(3)])
    m = torch.empty((3, 3) + tuple(shape), device='cuda')
    for i in range(3):
        for j in range(i + 1):
            m[i, j] = m[j, i] = (rot[i] * lam * rot[j]).sum(0)
    return m


def _problem(case, seed):
    """The fields of a case, on the GPU (float32), its seed cells and its box."""
    shape, model, d = _shape(case), case['model'], len(_shape(case))
    gen = torch.Generator(device='cuda').manual_seed(seed)
    rng = np.random.default_rng(seed)
    p = {'model': model, 'shape': shape, 'cells': np.stack([rng.integers(0, n, case['seeds']) for n in shape], 1)}
    if d == 2 or not _curvature(case):
        p['sides'] = [[-1, 1]] * d
        p['h'] = np.float32(2.) / np.asarray(shape, np.float32)
    if model == 'Isotropic2':
        p['cost'] = _bumps(rng, shape)
    elif model == 'Isotropic3':
        p['cost'] = _smooth(gen, shape, 8., 0.5, 1.5)
    elif model == 'Riemann2':
        p['metric'] = _metric2(gen, shape)
    elif model == 'Riemann3':
        p['metric'] = _metric3(gen, shape)
    elif model == 'Rander2':
        p['metric'] = _metric2(gen, shape)
        p['drift'] = torch.stack([_smooth(gen, shape, 20., -0.4, 0.4) for _ in range(2)])
    elif model.startswith('TTI'):
        th = _smooth(gen, shape, max(shape) / 16., -0.6, 0.6)
        if d == 2:
            c, s = torch.cos(th), torch.sin(th)
            p['rot'] = torch.stack([torch.stack([c, -s]), torch.stack([s, c])]).contiguous()
        else:
            phi = _smooth(gen, shape, max(shape) / 16., 0., 2 * math.pi)
            q = torch.stack([torch.cos(th / 2), torch.sin(th / 2) * torch.cos(phi),
                             torch.sin(th / 2) * torch.sin(phi), torch.zeros_like(th)])
            p['rot'] = _rotation3(q).contiguous()
    else:
        h = np.float32(2.) / np.float32(shape[0])
        p['sides'] = [[-1, 1], [-float(h) * shape[1] / 2, float(h) * shape[1] / 2]]
        p['h'] = np.array([h, h, 2 * np.pi / shape[2]], np.float32)
        p['cost'] = _bumps(rng, shape[:2])
    if case['walls']:
        walls = _smooth(gen, shape, 3., 0., 1.) > 0.6
        for c in p['cells']:
            walls[tuple(slice(max(0, int(x) - 3), int(x) + 4) for x in c)] = False
        p['walls'] = walls.to(torch.uint8)
    if case['sens'] or case['job'] == 'gradient':
        # a smooth misfit residual, respectively receivers on the faces
        p['weight'] = _smooth(gen, shape, 4., -1., 1.) if case['sens'] else torch.zeros(shape, device='cuda')
        if case['job'] == 'gradient':
            at = np.stack([rng.integers(0, n, 64) for n in shape], 1)
            axis = rng.integers(0, d, 64)
            at[np.arange(64), axis] = rng.integers(0, 2, 64) * (np.asarray(shape)[axis] - 1)
            p['weight'][tuple(torch.as_tensor(at[:, k], device='cuda') for k in range(d))] = 1.
            p['cost'] = _smooth(gen, shape, 10., 0.7, 1.3)
    return p


def _box(p):
    """Lower corner of the physical box (the angle axis starts half a cell below 0)."""
    lo = [s[0] for s in p['sides']]
    if len(lo) < len(p['shape']):
        lo.append(-p['h'][2] / 2)
    return np.array(lo, np.float64)


def _dict_in(p, case):
    points = _box(p) + (p['cells'] + 0.5) * p['h'].astype(np.float64)
    d = {'model': p['model'], 'seeds': points.astype(np.float32), 'exportValues': 1, 'verbosity': 0}
    if 'drift' in p:
        d['metric'] = Metrics.Rander(p['metric'], p['drift'])
    elif 'metric' in p:
        d['metric'] = Metrics.Riemann(p['metric'])
    elif 'rot' in p:
        c11, c13, c33, c44 = HEXAGONAL
        dim = len(p['shape'])
        base = Metrics.Seismic.TTI.from_hexagonal(c11, None, c13, c33, c44, vdim=dim)
        d['metric'] = Metrics.Seismic.TTI(base.linear, base.quadratic, vdim=dim, inverse_transformation=p['rot'])
    if 'cost' in p and case['job'] != 'gradient':
        d['cost'] = p['cost']
    if 'walls' in p:
        d['walls'] = p['walls']
    if case['flow']:
        d['exportGeodesicFlow'] = True
    if case['sens']:
        d['sensitivity'] = p['weight'].unsqueeze(-1)
    if case['fp64']:
        d['multiprecision'] = True
    if _curvature(case):
        d['xi'] = XI
    hfm = dictIn(d)
    if _curvature(case):
        hfm.SetRect(p['sides'], dimx=p['shape'][0])
        hfm.nTheta = p['shape'][2]
    else:
        hfm.SetRect(p['sides'], dims=list(p['shape']))
    if tuple(hfm.shape) != tuple(p['shape']):
        raise ValueError(f"grid {hfm.shape} instead of {p['shape']}")
    return hfm


def _batch_shapes(case):
    """Sides of the problems of a batch, uniform in n0..n1."""
    rng = np.random.default_rng(case['seeds'])
    return [tuple(int(v) for v in rng.integers(case['n0'], case['n1'] + 1, 2)) for _ in range(case['seeds'])]


def _batch_members(case, seed):
    """The problems of a batch, 1 to 8 seeds each."""
    rng = np.random.default_rng(seed)
    out = []
    for n0, n1 in _batch_shapes(case):
        member = _case('', 'Isotropic2', n0, n1, seeds=int(rng.integers(1, 9)))
        out.append((member, _problem(member, int(rng.integers(1 << 30)))))
    return out


# ------------------------------------------------------------------ the calls
def prepare(case, seed):
    if case['job'] == 'batch':
        return {'batch': batch.Batch([_dict_in(p, m) for m, p in _batch_members(case, seed)])}
    p = _problem(case, seed)
    state = {'hfm': _dict_in(p, case)}
    if case['job'] == 'gradient':
        state['cost'] = p['cost'].clone().requires_grad_(True)
        state['weight'] = p['weight']
    return state


def run(state):
    if 'batch' in state:
        b = state['batch']
        b.solve()
        return [b.values(i) for i in range(len(b.ifaces))]
    if 'cost' in state:
        state['cost'].grad = None
        values = autograd.eikonal_values(state['hfm'], state['cost'])
        (values * state['weight']).sum().backward()
        return {'values': values.detach(), 'gradient': state['cost'].grad}
    out = state['hfm'].Run()
    return {k: out[k] for k in ('values', 'flow', 'costSensitivity', 'seedValueSensitivity') if k in out}


def work(case):
    """Each input field read once, each output written once; the operations of
    one upwind update a cell (neighbour choice, sorting, quadratic)."""
    if case['job'] == 'batch':
        cells = sum(n0 * n1 for n0, n1 in _batch_shapes(case))
        return {'bytes': 8. * cells, 'flops': 20. * cells}
    shape = _shape(case)
    d, cells = len(shape), float(np.prod(shape))
    sym = d * (d + 1) // 2
    words = {'Isotropic': 1, 'Riemann': d * d, 'Rander': d * d + d, 'TTI': d * d}.get(case['model'][:-1], 0)
    words += 1 + (d if case['flow'] else 0) + (2 if case['sens'] else 0) + (3 if case['job'] == 'gradient' else 0)
    slots = {'Isotropic': d, 'TTI': 7 * sym, 'ReedsSheppForward': 7, 'Elastica': 30}.get(case['model'][:-1], sym)
    return {'bytes': 4. * words * cells + (cells if case['walls'] else 0.), 'flops': 10. * slots * cells}


# ------------------------------------------------------------------ 64 bits
def _quad(x, m, y):
    return sum(x[i] * m[i][j] * y[j] for i in range(len(x)) for j in range(len(y)))


def _selling(m):
    """Selling decomposition of the matrices m[i][j]: weights (K, N), offsets (K, d, N)."""
    d, like = len(m), m[0][0]
    b = [[torch.full_like(like, float(i == c)) for c in range(d)] for i in range(d)]
    b.append([torch.full_like(like, -1.) for _ in range(d)])
    phases = [(0, 1, 2), (1, 2, 0), (2, 0, 1)] if d == 2 else \
        [(0, 1, 2, 3), (0, 2, 1, 3), (0, 3, 1, 2), (1, 2, 0, 3), (1, 3, 0, 2), (2, 3, 0, 1)]
    for _ in range(34):
        moved = False
        for i, j, *rest in phases:
            acute = _quad(b[i], m, b[j]) > 0
            if not bool(acute.any()):
                continue
            moved = True
            for c in range(d):
                if d == 2:
                    b[rest[0]][c] = torch.where(acute, b[i][c] - b[j][c], b[rest[0]][c])
                else:
                    for r in rest:
                        b[r][c] = torch.where(acute, b[r][c] + b[i][c], b[r][c])
                b[i][c] = torch.where(acute, -b[i][c], b[i][c])
        if not moved:
            break
    w = torch.stack([(-_quad(b[i], m, b[j])).clamp(min=0) for i, j, *_ in phases])
    e = []
    for _, _, *rest in phases:
        if d == 2:
            x = b[rest[0]]
            e.append(torch.stack([-x[1], x[0]]))
        else:
            x, y = b[rest[0]], b[rest[1]]
            e.append(torch.stack([x[1] * y[2] - x[2] * y[1], x[2] * y[0] - x[0] * y[2], x[0] * y[1] - x[1] * y[0]]))
    return w, torch.stack(e).to(torch.int32)


def _inverse(m):
    """Inverse of symmetric matrices m[i][j] by cofactors."""
    if len(m) == 2:
        det = m[0][0] * m[1][1] - m[0][1] * m[0][1]
        return [[m[1][1] / det, -m[0][1] / det], [-m[0][1] / det, m[0][0] / det]]

    def minor(i, j):
        r, c = [k for k in range(3) if k != i], [k for k in range(3) if k != j]
        return (-1) ** (i + j) * (m[r[0]][c[0]] * m[r[1]][c[1]] - m[r[0]][c[1]] * m[r[1]][c[0]])
    det = sum(m[0][j] * minor(0, j) for j in range(3))
    return [[minor(j, i) / det for j in range(3)] for i in range(3)]


def _tangents(l, q):
    """The 7 tangent ellipses of the TTI dual ball l.x + x.q.x / 2 = 1 and whether the scheme is their min."""
    def roots(a, b, c):
        s = math.sqrt(b * b - a * c)
        return sorted([(-b + s) / c, (-b - s) / c] if abs(c) > abs(a) else [a / (-b + s), a / (-b - s)])

    def above(a, b, c, bound):
        lo, hi = roots(a, b, c)
        return lo if lo >= bound else hi

    def ratio(x, y):
        g = l[0] + q[0] * x + q[1] * y, l[1] + q[1] * x + q[2] * y
        s = x * g[0] + y * g[1]
        return g[0] / s, g[1] / s
    a, b = above(-2., l[0], q[0], 0.), above(-2., l[1], q[2], 0.)
    lp, lm = (l[0] + l[1]) / 2, (l[0] - l[1]) / 2
    qpp, qpm, qmm = (q[0] + 2 * q[1] + q[2]) / 4, (q[0] - q[2]) / 4, (q[0] - 2 * q[1] + q[2]) / 4
    out = [ratio(a, 0.)]
    for i in range(1, 6):
        v = (1 - i / 6) * a - i / 6 * b
        u = above(-2 + 2 * lm * v + qmm * v * v, lp + qpm * v, qpp, abs(v))
        out.append(ratio((u + v) / 2, (u - v) / 2))
    out.append(ratio(0., b))
    return out, out[0][0] * out[6][1] - out[0][1] * out[6][0] > 0


def _forward(v, m):
    """Selling decomposition of m kept near the direction v, its offsets turned against v."""
    w, e = _selling(m)
    f = e.double()
    ve = (torch.stack(v) * f).sum(1)
    near = ve * ve >= sum(x * x for x in v) * (f * f).sum(1) * (2. / 3.)
    return torch.where(near, w, 0.), torch.where((near & (ve > 0))[:, None], -e, e)


def _scheme(p):
    """Sub-schemes [(weights, offsets, shifts or None, forward slots)], whether
    their min is taken, and the right-hand side, in grid units."""
    shape, model, d = p['shape'], p['model'], len(p['shape'])
    n = int(np.prod(shape))
    h = [float(x) for x in p['h']]
    one = torch.ones(n, dtype=torch.float64, device='cuda')
    cost = p['cost'].double() if 'cost' in p else torch.ones(shape, dtype=torch.float64, device='cuda')
    if model.startswith('Isotropic'):
        e = torch.eye(d, dtype=torch.int32, device='cuda')[:, :, None].expand(d, d, n)
        return [(torch.stack([one / x ** 2 for x in h]), e, None, 0)], True, cost.reshape(-1)
    if model[:-1] in ('Riemann', 'Rander'):
        m = p['metric'].double().reshape(d, d, n)
        w, e = _selling(_inverse([[m[i, j] * (h[i] * h[j]) for j in range(d)] for i in range(d)]))
        shift = None
        if 'drift' in p:
            drift = p['drift'].double().reshape(d, n)
            shift = sum(drift[i] * h[i] * e[:, i].double() for i in range(d))
        return [(w, e, shift, 0)], True, cost.reshape(-1)
    if model.startswith('TTI'):
        c11, c13, c33, c44 = HEXAGONAL
        mixed = c13 ** 2 - c11 * c33 + 2 * c13 * c44
        lin = [float(np.float32(x)) for x in (c11 + c44, c33 + c44)]
        quad = [float(np.float32(x)) for x in (-2 * c11 * c44, mixed, -2 * c33 * c44)]
        diags, is_min = _tangents(lin, quad)
        rot = p['rot'].double().reshape(d, d, n)
        a = torch.linalg.inv(torch.stack([rot[:, j] * h[j] for j in range(d)], 1).permute(2, 0, 1)).permute(2, 1, 0)
        d0 = [[sum(a[k, i] * a[k, j] for k in range(d - 1)) for j in range(d)] for i in range(d)]
        d1 = [[a[d - 1, i] * a[d - 1, j] for j in range(d)] for i in range(d)]
        subs = []
        for x, y in diags:
            w, e = _selling([[x * d0[i][j] + y * d1[i][j] for j in range(d)] for i in range(d)])
            subs.append((w, e, None, 0))
        return subs, is_min, cost.reshape(-1)
    ixi = h[0] / (h[2] * XI)
    theta = torch.arange(shape[2], device='cuda', dtype=torch.float64) * (2 * math.pi / shape[2])
    theta = theta.repeat(n // shape[2])
    ct, st = torch.cos(theta), torch.sin(theta)

    def along(v):
        vv = sum(x * x for x in v)
        return _forward(v, [[v[i] * v[j] * (1 - EPS2) + (EPS2 * vv if i == j else 0.) for j in range(3)]
                            for i in range(3)])
    rhs = (cost[:, :, None] * h[0]).expand(shape).reshape(-1)
    if model == 'ReedsSheppForward2':
        w, e = along([ct, st, 0 * ct])
        turn = torch.zeros_like(e[:1])
        turn[0, 2] = -1
        return [(torch.cat([one[None] * ixi ** 2, w]), torch.cat([turn, e]), None, 6)], True, rhs
    parts = []
    for k in range(5):  # Fejer's rule on [0, pi] with the weight sin, 5 nodes (9 and 6 decimals, as tabulated)
        phi = math.pi * (k + 0.5) / 5
        wf = round(2 / 5 * (1 - 2 * sum(math.cos(2 * j * phi) / (4 * j * j - 1) for j in (1, 2))), 6)
        cp, sp = round(math.cos(phi), 9), round(math.sin(phi), 9)
        w, e = along([sp * ct, sp * st, cp * ixi * one])
        parts.append((w * wf, e))
    return [(torch.cat([w for w, _ in parts]), torch.cat([e for _, e in parts]), None, 30)], True, rhs


def _neighbours(e, shape, wrap):
    """Index of x + e for each offset, N where it leaves the grid."""
    n = int(np.prod(shape))
    at = torch.arange(n, device='cuda')
    out, inside, stride = torch.zeros_like(e[:, 0], dtype=torch.int64), torch.ones_like(e[:, 0], dtype=torch.bool), n
    for k, s in enumerate(shape):
        stride //= s
        y = (at // stride) % s + e[:, k]
        if wrap[k]:
            y = y % s
        inside &= (y >= 0) & (y < s)
        out += y * stride
    return torch.where(inside, out, n)


def _sorted(v, w):
    if len(v) > 6:
        v, o = v.sort(0)
        return v, w.gather(0, o)
    v, w = list(v), list(w)
    for p in range(len(v)):
        for i in range(p % 2, len(v) - 1, 2):
            keep = v[i] <= v[i + 1]
            v[i], v[i + 1] = torch.minimum(v[i], v[i + 1]), torch.maximum(v[i], v[i + 1])
            w[i], w[i + 1] = torch.where(keep, w[i], w[i + 1]), torch.where(keep, w[i + 1], w[i])
    return torch.stack(v), torch.stack(w)


def _upwind(u, sub, near):
    """Values and side (True: x + e) of the smaller neighbour of each offset."""
    w, _, shift, nfwd = sub
    plus, minus = u[near[0]], u[near[1]]
    if shift is not None:
        plus, minus = plus - shift, minus + shift
    if nfwd:
        minus[len(w) - nfwd:] = math.inf
    side = plus < minus
    v = torch.where(side, plus, minus)
    return (torch.where(w > 0, v, math.inf) if nfwd else v), side


def _update(v, w, rhs):
    """Solution of sum w (u - v)_+^2 = rhs^2."""
    v, w = _sorted(v, w)
    t = torch.where(v == math.inf, math.inf, v - v[:1])
    a, b, c = w.cumsum(0), (w * t).cumsum(0), (w * t * t).cumsum(0) - rhs * rhs
    k = ((a[:-1] * t[1:] - 2 * b[:-1]) * t[1:] + c[:-1] <= 0).to(torch.int64).cumprod(0).sum(0, keepdim=True)
    a, b, c = a.gather(0, k)[0], b.gather(0, k)[0], c.gather(0, k)[0]
    u = v[0] + (b + torch.sqrt((b * b - a * c).clamp(min=0))) / a
    return torch.where((v[0] == math.inf) | (a == 0), math.inf, u)


def _fixed_point(subs, near, is_min, rhs, fixed, start):
    """Decreasing Jacobi iteration from +inf to the fixed point of the scheme."""
    u = torch.cat([start, torch.full((1,), math.inf, dtype=torch.float64, device='cuda')])
    for it in range(20000):
        best = None
        for sub, nb in zip(subs, near):
            x = _update(_upwind(u, sub, nb)[0], sub[0], rhs)
            best = x if best is None else (torch.minimum if is_min else torch.maximum)(best, x)
        new = torch.where(fixed, u[:-1], torch.minimum(best, u[:-1]))
        if it % 16 == 15 and not bool((new < u[:-1] * (1 - 1e-13)).any()):
            break
        u[:-1] = new
    return u


def _exact(p, case):
    shape, d = p['shape'], len(p['shape'])
    n = int(np.prod(shape))
    subs, is_min, rhs = _scheme(p)
    wrap = [_curvature(case) and k == 2 for k in range(d)]
    near = [(_neighbours(s[1], shape, wrap), _neighbours(-s[1], shape, wrap)) for s in subs]
    seeds = torch.as_tensor(np.unique(np.ravel_multi_index(tuple(p['cells'].T), shape)), device='cuda')
    start = torch.full((n,), math.inf, dtype=torch.float64, device='cuda')
    fixed = torch.zeros(n, dtype=torch.bool, device='cuda')
    if 'walls' in p:
        fixed |= p['walls'].reshape(-1) != 0
    fixed[seeds] = True
    start[seeds] = 0.
    u = _fixed_point(subs, near, is_min, rhs, fixed, start)
    out = {'values': u[:-1].reshape(shape)}
    if not (case['flow'] or case['sens'] or case['job'] == 'gradient'):
        return out
    v, side = _upwind(u, subs[0], near[0])
    live = ~fixed & (u[:-1] < math.inf)
    fw = torch.where(live & (v < u[:-1]), subs[0][0] * (u[:-1] - v), 0.)
    signed = torch.where(side, fw, -fw)
    vec = torch.stack([(signed * subs[0][1][:, k]).sum(0) for k in range(d)])
    h = torch.tensor([float(x) for x in p['h']], dtype=torch.float64, device='cuda')[:, None]
    if case['flow']:
        out['flow'] = (-h * vec).reshape((d,) + tuple(shape))
        return out
    # adjoint of the linearised scheme: (D - W)^T lambda = s
    total = fw.sum(0)
    diag = torch.where(total == 0, 1., total)
    to = torch.where(fw > 0, torch.where(side, near[0][0], near[0][1]), n).reshape(-1)
    s = p['weight'].double().reshape(-1)
    lam = torch.zeros_like(s)
    for it in range(20000):
        new = torch.zeros(n + 1, dtype=torch.float64, device='cuda').index_add_(0, to, (fw * lam).reshape(-1))
        new = (new[:-1] + s) / diag
        if it % 16 == 15 and bool(((new - lam).abs() <= 1e-13 * new.abs().max()).all()):
            break
        lam = new
    if case['job'] == 'gradient':
        grad = lam * rhs
        grad[seeds] = 0.
        out['gradient'] = grad.reshape(shape)
        return out
    first = torch.as_tensor(np.ravel_multi_index(tuple(p['cells'].T), shape), device='cuda')
    out['seedValueSensitivity'] = lam[first].reshape(-1, 1)
    lam = lam.clone()
    lam[seeds] = 0.
    if 'drift' in p:  # sensitivities of a drift model are divided by the metric norm of the flow
        m, drift = p['metric'].double().reshape(d, d, n), p['drift'].double().reshape(d, n)
        back = -vec * h
        norm = torch.sqrt(sum(back[i] * m[i, j] * back[j] for i in range(d) for j in range(d))) + (drift * back).sum(0)
        lam = lam / torch.where(fixed, 1., norm)
    out['costSensitivity'] = lam.reshape(tuple(shape) + (1,))
    return out


def exact(case, seed):
    if case['job'] == 'batch':
        return [_exact(p, m)['values'] for m, p in _batch_members(case, seed)]
    return _exact(_problem(case, seed), case)
