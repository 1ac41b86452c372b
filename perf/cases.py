"""The work that users have this library do, as cases that can be timed and compared.

A case is one call, or one short job, through the Python binding of the C ABI
(scadyn_amd/native.py):

  bar      one wavelength bar, host mesh in, T-matrix out (tmat_solve): operator set-up
           included, as scadyn's per-bar driver calls it
  requests several bars through the request loop (Server), waited for in order
  columns  T-matrix columns of a kept operator (Operator.tmatrix_cols)
  solve    right-hand sides of a caller against a kept operator (Operator.solve)
  matvec   the bare operator product of a caller's own iteration (Operator.matvec)
  project  T = mat^H X on device buffers (Operator.project_noalloc)

Meshes are this package's seeded cube-split bodies: the sphere, and the Gaussian random
ellipsoid (axes 1:0.8:0.6), whose grids are ragged.  The seed moves the inner vertices
(jitter), so that another seed is another mesh with the same number of tets, and it shifts
the permittivity a little; right-hand sides are standard normal.  Materials, size
parameters, expansion orders and solver settings are those of the benchmark's workloads
(scadyn_amd/workloads.py) and of the tests.
"""
import math

import numpy as np
import torch

from scadyn_amd import meshgen, native
from scadyn_amd.workloads import A_RADIUS

ITER = {False: 12, True: 30}  # iterations of one system at these size parameters, FP64 (1e-5) and mixed (1e-9)


def listed():
    return [
        # the smallest bar of the tests: launches, allocations and host set-up
        dict(name='bar-192-fp64', kind='bar', body='sphere', cells=4, ka=2.0, eps=2.5, loss=0.01, nmax=1, mixed=False),
        # a small irregular particle of a size-distribution sweep, mixed precision
        dict(name='bar-4686-mixed', kind='bar', body='ellipsoid', cells=16, ka=2.0, eps=2.0, loss=0.1, nmax=6,
             mixed=True),
        # the 43,248-tet sphere workload, the reference's GMRES settings
        dict(name='bar-43248-fp64', kind='bar', body='sphere', cells=24, ka=2.0, eps=2.5, loss=0.01, nmax=5,
             mixed=False),
        # a mid-size irregular particle at a larger size parameter, mixed precision
        dict(name='bar-24708-mixed', kind='bar', body='ellipsoid', cells=28, ka=4.0, eps=1.8, loss=0.05, nmax=5,
             mixed=True),
        # a few small requests that arrive together at the request loop
        dict(name='requests-3x2k-mixed', kind='requests', body='ellipsoid', cells=12, ka=2.0, eps=2.2, loss=0.1,
             nmax=4, mixed=True, count=3),
        # one product of a caller's own solver: latency
        dict(name='matvec-1680x1', kind='matvec', body='sphere', cells=8, ka=2.0, eps=2.5, loss=0.01, nrhs=1),
        # a narrow, odd batch on a ragged grid
        dict(name='matvec-24708x7', kind='matvec', body='ellipsoid', cells=28, ka=4.0, eps=3.0, loss=0.1, nrhs=7),
        # a full batch
        dict(name='matvec-43248x64', kind='matvec', body='sphere', cells=24, ka=2.0, eps=2.5, loss=0.01, nrhs=64),
        # a caller's few right-hand sides, FP64
        dict(name='solve-5472x3-fp64', kind='solve', body='sphere', cells=12, ka=2.0, eps=2.5, loss=0.01, nrhs=3,
             mixed=False),
        # columns of a larger particle on a kept operator, FP64: matvec and Krylov at full batch
        dict(name='columns-72204x48-fp64', kind='columns', body='ellipsoid', cells=40, ka=2.0, eps=2.5, loss=0.1,
             nmax=6, ncols=48, mixed=False),
        # the same in mixed precision on a mesh large enough for the binary16 Krylov basis, as the benchmark's sphere
        dict(name='columns-369390x64-mixed', kind='columns', body='sphere', cells=49, ka=3.0, eps=2.0, loss=0.02,
             nmax=7, ncols=64, mixed=True),
        # the projection of a 43,248-tet bar at nmax 12
        dict(name='project-129744x336x336', kind='project', rows=129744, na=336, nx=336),
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['bar', 'bar', 'requests', 'matvec', 'solve', 'columns', 'columns', 'project'])
    if kind == 'project':
        return dict(kind=kind, rows=_between(rng, 500, 129744), na=_between(rng, 6, 336), nx=_between(rng, 1, 336))
    body = rng.choice(['sphere', 'ellipsoid'])
    top = {'bar': 26, 'requests': 13, 'matvec': 28, 'solve': 24, 'columns': 34}[kind]
    case = dict(kind=kind, body=body, cells=_between(rng, 6 if body == 'sphere' else 9, top),
                ka=round(rng.uniform(1.0, 3.0), 3), eps=round(rng.uniform(1.5, 2.5), 3),
                loss=round(rng.uniform(0.0, 0.2), 3))
    if kind == 'matvec':
        case.update(nrhs=_between(rng, 1, 64))
        return case
    case.update(mixed=rng.random() < 0.5)
    if kind == 'solve':
        case.update(nrhs=_between(rng, 1, 48))
    elif kind == 'columns':
        nmax = rng.randint(2, 7)
        case.update(nmax=nmax, ncols=min(2 * nmax * (nmax + 2), _between(rng, 1, 64)))
        if case['mixed'] and rng.random() < 0.5:
            case.update(basis=2)
    else:
        case.update(nmax=rng.randint(1, 5))
        if kind == 'requests':
            case.update(count=rng.randint(2, 4))
    return case


def _tets(case):
    """Tets of the case's mesh: 6 per lattice cell inside the body (about 0.52 of the
    sphere's cells and 0.19 of the ellipsoid's)."""
    return 6.0 * (0.52 if case['body'] == 'sphere' else 0.19) * case['cells'] ** 3


_radius = {}


def _mesh(case, seed):
    """(coord, etopol, param, k) of a case; the seed moves the inner vertices and the permittivity."""
    if case['body'] == 'sphere':
        c, e = meshgen.sphere(case['cells'], seed=seed)
    else:
        if not _radius:
            fn = meshgen.gaussian_ellipsoid_radius(seed=0)
            t, p = np.meshgrid(np.linspace(0, np.pi, 91), np.linspace(-np.pi, np.pi, 181))
            _radius['fn'], _radius['extent'] = fn, 1.02 * float(fn(t, p).max())
        c, e = meshgen.star_body(_radius['fn'], case['cells'], _radius['extent'], seed=seed)
    v = meshgen.tet_volumes(c, e).sum()
    c = c * (A_RADIUS / (3.0 * v / 4.0 / math.pi) ** (1.0 / 3.0))
    rng = np.random.default_rng(seed)
    eps = complex(case['eps'], case['loss']) + 0.01 * rng.random()
    return c, e, np.full(e.shape[0], eps), case['ka'] / A_RADIUS


def _opts(case):
    o = dict(precision=native.PREC_MIXED if case.get('mixed') else native.PREC_FP64)
    if case.get('mixed'):
        o.update(tol=1e-4, restart=20)
    if case.get('basis'):
        o.update(basis=case['basis'])
    return o


def _normal(seed, *shape):
    rng = np.random.default_rng(seed + 1)
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


def _device():
    return 'cuda' if torch.cuda.is_available() else 'cpu'


def _buffers(case, seed):
    gen = torch.Generator(device=_device()).manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, dtype=torch.complex128, device=_device(), generator=gen)
    return normal(case['rows'], case['na']), normal(case['rows'], case['nx'])


def prepare(case, seed):
    kind = case['kind']
    s = dict(case=case)
    if kind == 'project':
        small = dict(body='sphere', cells=4, ka=2.0, eps=2.5, loss=0.01)
        s['op'] = native.Operator(*_mesh(small, seed))
        s['mat'], s['X'] = _buffers(case, seed)
        s['T'] = torch.empty(case['na'], case['nx'], dtype=torch.complex128, device=_device())
        return s
    if kind == 'bar':
        s['mesh'] = _mesh(case, seed)
        return s
    if kind == 'requests':
        # the bars of one particle size, each a mesh of its own
        s['meshes'] = [_mesh(case, seed + 1000 * (q + 1)) for q in range(case['count'])]
        s['server'] = native.Server()
        return s
    mesh = _mesh(case, seed)
    s['op'] = native.Operator(*mesh, **_opts(case))
    n = 3 * mesh[1].shape[0]
    if kind in ('matvec', 'solve'):
        s['x'] = _normal(seed, case['nrhs'], n)
    else:
        total = 2 * case['nmax'] * (case['nmax'] + 2)
        s['cols'] = np.random.default_rng(seed).permutation(total)[:case['ncols']]
    return s


def run(s):
    case = s['case']
    kind = case['kind']
    if kind == 'bar':
        return native.tmat_solve(*s['mesh'], case['nmax'], **_opts(case))
    if kind == 'requests':
        ids = [s['server'].submit(*m, case['nmax'], **_opts(case)) for m in s['meshes']]
        return [s['server'].wait(i)[:2] for i in ids]
    if kind == 'columns':
        return s['op'].tmatrix_cols(case['nmax'], s['cols'])
    if kind == 'solve':
        return s['op'].solve(s['x'])
    if kind == 'matvec':
        return s['op'].matvec(s['x'])
    s['op'].project_noalloc(case['rows'], case['na'], case['nx'], s['mat'].data_ptr(), s['X'].data_ptr(),
                            s['T'].data_ptr())
    return s['T']


def work(case):
    """Counted per pass.  N tets, P ~ 80 N near-zone blocks (about 160 near tets each, every
    pair stored once); a product with the operator is 8 (9 x 2 P) flops near, 4 x 2 x 27 x 8 N
    for both grid projections and 4 transforms of the padded grid there and back.  A set-up
    evaluates 1,360 kernel values (about 40 flops) per block."""
    if case['kind'] == 'project':
        r, a, x = case['rows'], case['na'], case['nx']
        return {'bytes': 16.0 * (r * a + r * x + a * x), 'flops': 8.0 * r * a * x}
    N = _tets(case)
    P = 80.0 * N
    grid = 8.0 * N  # padded grid points of a body that fills its box
    product = 144.0 * P + 1728.0 * N + 2 * 4 * 5 * grid * math.log2(max(grid, 2.0))
    if case['kind'] == 'matvec':
        return {'bytes': 16.0 * 6 * N * case['nrhs'] + 72.0 * P + 1728.0 * N, 'flops': product * case['nrhs']}
    n, it = 3 * N, ITER[bool(case['mixed'])]
    solve = it * product + 16.0 * it * it * n  # flops of one system
    if case['kind'] == 'solve':
        return {'bytes': 32.0 * n * case['nrhs'] + 72.0 * P + 1728.0 * N, 'flops': solve * case['nrhs']}
    full = 2 * case['nmax'] * (case['nmax'] + 2)
    if case['kind'] == 'columns':
        m = case['ncols']
        return {'bytes': 72.0 * P + 1728.0 * N + 16.0 * full * m, 'flops': (solve + 8.0 * full * n) * m}
    q = case.get('count', 1)
    return {'bytes': q * (16.0 * N + 8.0 * n + 16.0 * full * full),
            'flops': q * (full * (solve + 8.0 * full * n) + 40.0 * 1360 * P)}


# ---- the same in plain torch, 64 bits --------------------------------------------------
# The precorrected-FFT operator written out: grid, tet -> cube map, 3 x 3 x 3 projections, the
# near-zone blocks with the singularity subtracted (24-point tet, 7-point triangle rules; kept
# in complex64, as the method stores them), and the convolution with torch.fft.

_TET24 = [(3.561913862225449e-01, 2.146028712591517e-01, 6.653791709694644e-03),
          (8.779781243961660e-01, 4.067395853461134e-02, 1.679535175886776e-03),
          (3.298632957317306e-02, 3.223378901422757e-01, 9.226196923942399e-03)]
_TET24_EDGE = (2.696723314583159e-01, 6.366100187501753e-02, 6.030056647916491e-01, 8.035714285714282e-03)


def _tables(dev):
    """Tet rule (24 x 3, weights) and triangle rule (7 x 2, weights), reference-element weights."""
    p, w = [], []
    for a, b, wt in _TET24:
        for q in range(4):
            v = [b] * 4
            v[q] = a
            p.append(v[1:])
            w.append(wt)
    g, h, i, wt = _TET24_EDGE
    for x in range(4):
        for y in range(4):
            if x != y:
                v = [h] * 4
                v[x], v[y] = g, i
                p.append(v[1:])
                w.append(wt)
    tri = [(1 / 3, 1 / 3, 0.1125)]
    for a, b, wt in ((0.0597158717897698, 0.470142064105115, 0.0661970763942531),
                     (0.797426985353087, 0.101286507323456, 0.0629695902724136)):
        tri += [(a, b, wt), (b, b, wt), (b, a, wt)]
    tri = torch.tensor(tri, dtype=torch.float64, device=dev)
    return (torch.tensor(p, dtype=torch.float64, device=dev), torch.tensor(w, dtype=torch.float64, device=dev),
            tri[:, :2].contiguous(), tri[:, 2].contiguous())


def _green(R, k):
    return torch.polar(1.0 / (4 * math.pi * R), k * R)


def _smooth(R, k):
    """exp(ikR)/(4 pi R) without its 1/R and R terms; the limit ik/(4 pi) at R = 0."""
    near = R < 1e-10 * R.max()
    Rs = torch.where(near, torch.ones_like(R), R)
    v = _green(Rs, k) - (1.0 / Rs - 0.5 * k * k * Rs) / (4 * math.pi)
    return torch.where(near, torch.complex(torch.zeros_like(R), torch.full_like(R, k / (4 * math.pi))), v)


def _triangle(p, n, r):
    """Integrals of 1/R and R over flat triangles (Wilton et al. 1984): p (..., 3, 3), n (..., 3), r (..., 3)."""
    w0 = ((r - p[..., 0, :]) * n).sum(-1)
    a0 = w0.abs()
    k1, k2 = 0.0, 0.0
    for l in range(3):
        p1, p2 = p[..., (l + 1) % 3, :], p[..., (l + 2) % 3, :]
        s = p2 - p1
        length = s.norm(dim=-1)
        s = s / length[..., None]
        m = torch.linalg.cross(s, n)
        t0, sm = ((p1 - r) * m).sum(-1), ((p1 - r) * s).sum(-1)
        sp, Rp, Rm = sm + length, (r - p2).norm(dim=-1), (p1 - r).norm(dim=-1)
        R2 = t0 * t0 + w0 * w0
        beta = torch.where(a0 > 1e-10, torch.atan(t0 * sp / (R2 + a0 * Rp)) - torch.atan(t0 * sm / (R2 + a0 * Rm)),
                           torch.zeros_like(a0))
        I = torch.where(Rm + sm > Rp - sp, torch.log(((Rp + sp) / (Rm + sm)).abs()),
                        torch.log(((Rm - sm) / (Rp - sp)).abs()))
        k1 = k1 - a0 * beta + t0 * I
        k2 = k2 + t0 * 0.5 * (sp * Rp - sm * Rm + R2 * I)
    return k1, (w0 * w0 * k1 + k2) / 3.0


_FACES = [(1, 2, 3), (0, 3, 2), (0, 1, 3), (0, 2, 1)]


class _Plain:
    """The operator of one mesh."""

    def __init__(self, coord, etopol, param, k):
        dev = _device()
        t = torch.as_tensor(coord, device=dev)[torch.as_tensor(etopol.astype(np.int64), device=dev)]  # (N, 4, 3)
        self.N, self.k, self.dev = t.shape[0], k, dev
        self.vol = ((t[:, 3] - t[:, 0]) * torch.linalg.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0])).sum(-1).abs() / 6
        lo, hi = torch.as_tensor(coord.min(0), device=dev), coord.max(0)
        delta = 0.9 * (float(self.vol.sum()) / self.N) ** float(np.float32(1.0) / np.float32(3.0))
        dims = []
        for c in range(3):
            n = math.ceil((hi[c] - float(lo[c])) / delta) + 1
            dims.append(n + (n + 1) % 2 + 1)
        self.dims, self.delta = dims, delta
        cube = torch.floor((t.mean(1) - lo) / (2 * delta)).long()
        off = torch.tensor([(j % 3, j // 3 % 3, j // 9) for j in range(27)], device=dev)
        nodes = 2 * cube[:, None, :] + off
        self.nodes = nodes[..., 0] + dims[0] * (nodes[..., 1] + dims[1] * nodes[..., 2])  # (N, 27)
        # projection: match the fields on the 98 surface points of a 5 x 5 x 5 lattice
        lat = torch.tensor([(x, y, z) for z in range(5) for y in range(5) for x in range(5)
                            if max(abs(x - 2), abs(y - 2), abs(z - 2)) == 2], dtype=torch.float64, device=dev) / 2 - 1
        test = 2 * (2 * delta) * lat + delta
        W = _green((test[:, None, :] - delta * off.double()[None]).norm(dim=-1), k)
        U, s, Vh = torch.linalg.svd(W, full_matrices=False)
        inv = torch.where(s > 1e-6, 1.0 / s, torch.zeros_like(s))
        WW = (Vh.mH * inv) @ U.mH
        corner = lo + 2 * delta * cube
        self.S = torch.empty(self.N, 27, 4, dtype=torch.complex128, device=dev)
        for a in range(0, self.N, 8192):
            q = t[a:a + 8192]
            pt = test[None] + corner[a:a + 8192, None, :]
            Q = [_green((pt - q.mean(1)[:, None]).norm(dim=-1), k) * self.vol[a:a + 8192, None]]
            grad = torch.zeros(q.shape[0], 98, 3, dtype=torch.complex128, device=dev)
            for f in _FACES:
                p = q[:, list(f)]
                area = 0.5 * torch.linalg.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0])  # outward, length = area
                grad += _green((pt - p.mean(1)[:, None]).norm(dim=-1), k)[..., None] * area[:, None, :]
            Q = torch.cat([Q[0][..., None], grad], dim=-1)
            self.S[a:a + 8192] = torch.matmul(WW, Q) / self.vol[a:a + 8192, None, None].sqrt()
        self._near(t, cube, torch.as_tensor(param, device=dev))
        # circulant kernel on the doubled grid
        L = [2 * n for n in dims]
        ax = [torch.minimum(torch.arange(l, device=dev), l - torch.arange(l, device=dev)).double() * delta for l in L]
        R = (ax[2][:, None, None] ** 2 + ax[1][None, :, None] ** 2 + ax[0][None, None, :] ** 2).sqrt()
        R[0, 0, 0] = 1.0
        G = _green(R, k)
        G[0, 0, 0] = 0
        self.FG = torch.fft.fftn(G)

    def _near(self, t, cube, param):
        k, dev = self.k, self.dev
        nc = [(n - 2) // 2 for n in self.dims]
        cid = cube[:, 0] + nc[0] * (cube[:, 1] + nc[1] * cube[:, 2])
        order = torch.argsort(cid, stable=True)
        start = torch.searchsorted(cid[order], torch.arange(nc[0] * nc[1] * nc[2] + 1, device=dev))
        T, B, O = [], [], []
        every = torch.arange(self.N, device=dev)
        for o in range(27):
            d = torch.tensor((o % 3 - 1, o // 3 % 3 - 1, o // 9 - 1), device=dev)
            c = cube + d
            ok = ((c >= 0) & (c < torch.tensor(nc, device=dev))).all(-1)
            q = (c[:, 0] + nc[0] * (c[:, 1] + nc[1] * c[:, 2]))[ok]
            cnt = start[q + 1] - start[q]
            row = torch.repeat_interleave(every[ok], cnt)
            first = torch.repeat_interleave(start[q] - (torch.cumsum(cnt, 0) - cnt), cnt)
            col = order[first + torch.arange(row.numel(), device=dev)]
            keep = col >= row
            T.append(row[keep])
            B.append(col[keep])
            O.append(torch.full((int(keep.sum()),), o, device=dev))
        self.T, self.B, O = torch.cat(T), torch.cat(B), torch.cat(O)
        P = self.T.numel()
        j = torch.arange(27, device=dev)
        jj = torch.stack((j % 3, j // 3 % 3, j // 9), -1)
        oo = 2 * (jj - 1)
        R = self.delta * (jj[None, :, None] - jj[None, None, :] - oo[:, None, None]).double().norm(dim=-1)
        Gt = torch.where(R == 0, torch.zeros_like(R, dtype=torch.complex128), _green(torch.where(R == 0, 1.0, R), k))
        tp, tw, sp, sw = _tables(dev)
        bary = torch.cat((1 - tp.sum(1, keepdim=True), tp), 1)                   # (24, 4)
        quad = torch.einsum('qa,nac->nqc', bary, t)                              # (N, 24, 3)
        face = t[:, torch.tensor(_FACES, device=dev)]                            # (N, 4, 3, 3)
        nrm = torch.linalg.cross(face[:, :, 1] - face[:, :, 0], face[:, :, 2] - face[:, :, 0])
        twice = nrm.norm(dim=-1)                                                 # 2 x area
        nrm = nrm / twice[..., None]
        tb = torch.cat((1 - sp.sum(1, keepdim=True), sp), 1)
        surf = torch.einsum('qa,nfac->nfqc', tb, face)                           # (N, 4, 7, 3)
        blocks = torch.empty(P, 3, 3, dtype=torch.complex64, device=dev)
        four = 4 * math.pi
        for a in range(0, P, 16384):
            T, B, o = self.T[a:a + 16384], self.B[a:a + 16384], O[a:a + 16384]
            vT, vB = self.vol[T], self.vol[B]
            # both volumes
            v = (_smooth((quad[T][:, :, None] - quad[B][:, None]).norm(dim=-1), k) * tw).sum(-1) * (6 * vB)[:, None]
            for f in range(4):
                K1, K2 = _triangle(face[B, f][:, None], nrm[B, f][:, None], quad[T])
                h = (nrm[B, f][:, None] * (face[B, f, 0][:, None] - quad[T])).sum(-1)
                v = v + (h * K1 * 0.5 - 0.5 * k * k * h * K2 * 0.25) / four
            vv = (v * tw).sum(-1) * 6 * vT
            # both surfaces
            dd = torch.zeros(T.numel(), 3, 3, dtype=torch.complex128, device=dev)
            for f in range(4):
                s = _smooth((surf[T][:, :, :, None] - surf[B, f][:, None, None]).norm(dim=-1), k)
                s = (s * sw).sum(-1) * twice[B, f][:, None, None]
                K1, K2 = _triangle(face[B, f][:, None, None], nrm[B, f][:, None, None], surf[T])
                s = ((s + (K1 - 0.5 * k * k * K2) / four) * sw).sum(-1) * twice[T]    # (p, 4)
                dd += (s[..., None] * nrm[T]).sum(1)[..., None] * nrm[B, f][:, None]
            # what the grid already gives
            far = torch.matmul(self.S[T].mT, torch.matmul(Gt[o], self.S[B])) * (vT * vB).sqrt()[:, None, None]
            eye = torch.eye(3, device=dev)
            z = -k * k * ((vv - far[:, 0, 0])[:, None, None] * eye) + (dd - far[:, 1:, 1:])
            z = z / (vT * vB).sqrt()[:, None, None]
            z = z + torch.where(T == B, 1.0 / (param[T] - 1.0), torch.zeros_like(param[T]))[:, None, None] * eye
            blocks[a:a + 16384] = z.to(torch.complex64)
        self.blocks = blocks

    def __call__(self, x):
        """A x for one vector (3 N,)."""
        x = x.reshape(self.N, 3)
        nx, ny, nz = self.dims
        src = torch.cat((self.S[..., :1] * x[:, None], (self.S[..., 1:] * x[:, None]).sum(-1, keepdim=True)), -1)
        grid = torch.zeros(nx * ny * nz, 4, dtype=torch.complex128, device=self.dev)
        grid.index_add_(0, self.nodes.reshape(-1), src.reshape(-1, 4))
        out = torch.empty_like(grid)
        for c in range(4):
            F = torch.fft.fftn(grid[:, c].reshape(nz, ny, nx), s=(2 * nz, 2 * ny, 2 * nx)) * self.FG
            out[:, c] = torch.fft.ifftn(F)[:nz, :ny, :nx].reshape(-1)
        g = out[self.nodes]
        y = (self.S[..., 1:] * g[..., 3:]).sum(1) - self.k ** 2 * (self.S[..., :1] * g[..., :3]).sum(1)
        for a in range(0, self.T.numel(), 1 << 20):
            T, B, A = self.T[a:a + (1 << 20)], self.B[a:a + (1 << 20)], self.blocks[a:a + (1 << 20)].to(torch.complex128)
            y.index_add_(0, T, (A * x[B][:, None, :]).sum(-1))
            two = T != B
            y.index_add_(0, B[two], (A[two] * x[T[two]][:, :, None]).sum(1))
        return y.reshape(-1)


def exact(case, seed):
    """Products and projections in 64 bits.  A solve ends at its tolerance, far above 64 bits,
    and its own reference would be a dense or iterated solve of the operator that the matvec
    cases already hold: no value here for it."""
    if case['kind'] == 'project':
        mat, X = _buffers(case, seed)
        return torch.matmul(mat.mH.contiguous(), X)
    if case['kind'] != 'matvec':
        return None
    op = _Plain(*_mesh(case, seed))
    x = torch.as_tensor(_normal(seed, case['nrhs'], 3 * op.N), device=op.dev)
    return torch.stack([op(v) for v in x]).cpu().numpy()
