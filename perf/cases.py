"""
What a user of this framework has it do, as measurable cases.

Five paths, each through the public entry points a fitting or rendering program
calls:

- ``views``     clip transform, rasterize, interpolate, antialias over one or
                more views of a mesh; with ``grad`` an L2 fitting step that
                returns the gradients of the vertices and attributes, with
                ``graph`` that step replayed from a captured HIP graph;
- ``textured``  a fitting step that rasterizes with screen-space derivatives,
                interpolates uv and its texel footprint, samples a texture and
                antialiases;
- ``layers``    depth-peeled layers composited front to back, antialiased,
                recomputed in the backward pass;
- ``uneven``    meshes of different sizes, each at its own resolution, as one
                packed batch, forward and backward;
- ``session``   a scene of several objects through the deferred session.

Meshes are the noisy icospheres of the repository's benchmark and tests; the
cameras look at the origin from Fibonacci directions at distance 3.2.

``exact`` evaluates the same paths in 64 bits with plain torch: visibility by
the documented conventions (4 sub-pixel bits, top-left rule, smallest float32
z/w, ties to the smaller triangle), every value and gradient in float64 from the
float32 clip-space buffer.
"""
import functools
import math

import torch

from diffrp_amd import batch, deferred, layered, nvdr, texture
from diffrp_amd.camera import PerspectiveCamera, clip_space
from diffrp_amd.geometry import fibonacci_directions, icosphere
from diffrp_amd.loss import l2_loss

_DIST = 3.2  # camera distance


# ----------------------------------------------------------------------------
# the cases
# ----------------------------------------------------------------------------
def _views(name, views, subdiv, height, width, channels, noise=0.01, grad=True, graph=False, prepared=False):
    return {'name': name, 'path': 'views', 'views': views, 'subdiv': subdiv, 'height': height, 'width': width,
            'channels': channels, 'noise': noise, 'grad': grad, 'graph': graph, 'prepared': prepared}


def listed():
    return [
        # a preview or a tool's redraw: one small view of the README-size mesh, no gradient
        _views('preview', 1, 3, 256, 256, 3, noise=0.0, grad=False),
        # one optimisation step on one large view, called eagerly as diffrp does
        _views('view_step', 1, 6, 1024, 1024, 8),
        # the same loop of a program that captured its step in a HIP graph
        _views('view_step_graph', 1, 5, 512, 512, 4, graph=True),
        # the benchmark's step: 64 views of the 82k-triangle mesh
        _views('views_step', 64, 6, 512, 512, 8, prepared=True),
        # normals and uv (5 channels) at a photograph's odd crop
        _views('ragged_step', 3, 6, 733, 1019, 5),
        # a whole G-buffer (position, normal, colour, uv, tangent) fitted at once
        _views('gbuffer_step', 8, 6, 512, 512, 16),
        # rendering a turntable of a dense mesh, no gradient
        _views('turntable', 24, 7, 361, 641, 3, grad=False),
        # texture fitting with the texel footprint (mip selection, density terms)
        {'name': 'textured_step', 'path': 'textured', 'views': 4, 'subdiv': 5, 'height': 768, 'width': 768,
         'noise': 0.01, 'texture': 1024},
        # a transparent object: three layers of vertex RGBA
        {'name': 'layers_step', 'path': 'layers', 'subdiv': 7, 'height': 720, 'width': 1280, 'channels': 4,
         'layers': 3, 'noise': 0.005},
        # the large one: 5.2M triangles, 4 layers, 16 channels at 2048 x 2048
        {'name': 'layers_large', 'path': 'layers', 'subdiv': 9, 'height': 2048, 'width': 2048, 'channels': 16,
         'layers': 4, 'noise': 0.005},
        # many crumpled meshes of different sizes and resolutions as one batch
        {'name': 'uneven_step', 'path': 'uneven', 'meshes': 16, 'subdiv_min': 3, 'subdiv_max': 7, 'res_min': 200,
         'res_max': 1100, 'channels': 4, 'noise': 0.02, 'mix': 3},
        # several objects through the session: normals, albedo, depth, antialiased
        {'name': 'session', 'path': 'session', 'objects': 3, 'subdiv': 5, 'height': 512, 'width': 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_size(rng, most, lo=200, hi=2048):
    """A height and a width with at most ``most`` pixels."""
    h = _log_int(rng, lo, min(hi, most // lo))
    return h, max(lo, min(_log_int(rng, max(lo, h // 2), min(hi, 2 * h)), most // h))


def draw(rng):
    path = rng.choice(['views', 'views', 'views', 'textured', 'layers', 'uneven', 'session'])
    if path == 'views':
        views = _log_int(rng, 1, 64)
        subdiv = rng.randint(3, 7 if views <= 16 else 6)
        h, w = _draw_size(rng, (1 << 24) // views)
        case = _views('', views, subdiv, h, w, rng.choice([1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 14, 16]),
                      noise=round(rng.uniform(0.0, 0.01), 4), grad=rng.random() < 0.75,
                      prepared=rng.random() < 0.3)
        case['graph'] = case['grad'] and views <= 8 and rng.random() < 0.3
    elif path == 'textured':
        views = _log_int(rng, 1, 16)
        h, w = _draw_size(rng, (1 << 22) // views)
        case = {'path': path, 'views': views, 'subdiv': rng.randint(3, 6), 'height': h, 'width': w,
                'noise': round(rng.uniform(0.0, 0.01), 4), 'texture': rng.choice([256, 512, 1024, 2048])}
    elif path == 'layers':
        h, w = _draw_size(rng, 1 << 22)
        case = {'path': path, 'subdiv': rng.randint(4, 8), 'height': h, 'width': w,
                'channels': rng.choice([4, 5, 6, 8, 12, 16]), 'layers': rng.randint(2, 4), 'noise': 0.005}
    elif path == 'uneven':
        top = rng.randint(5, 7)
        case = {'path': path, 'meshes': rng.randint(3, 24), 'subdiv_min': 3, 'subdiv_max': top, 'res_min': 150,
                'res_max': rng.randint(400, 1200), 'channels': rng.choice([1, 3, 4, 8]), 'noise': 0.02,
                'mix': rng.randrange(1 << 16)}
    else:
        h, w = _draw_size(rng, 1 << 20)
        case = {'path': path, 'objects': rng.randint(1, 6), 'subdiv': rng.randint(3, 6), 'height': h, 'width': w}
    case.pop('name', None)
    return case


# ----------------------------------------------------------------------------
# inputs
# ----------------------------------------------------------------------------
@functools.lru_cache(maxsize=16)
def _sphere(subdiv):
    v, f = icosphere(subdiv, 0.8)
    return torch.from_numpy(v).float(), torch.from_numpy(f).int()


def _gen(seed):
    return torch.Generator(device='cuda').manual_seed(seed)


def _mesh(subdiv, noise, gen):
    v, f = _sphere(subdiv)
    v = v.cuda()
    return v + noise * torch.randn(v.shape, generator=gen, device='cuda'), f.cuda()


def _view_projection(views, h, w):
    out = []
    for d in fibonacci_directions(views):
        cam = PerspectiveCamera.looking_at_origin_from(d * _DIST, h=h, w=w)
        out.append(cam.P('cpu') @ cam.V('cpu'))
    return torch.stack(out).cuda()


def _uneven_items(case):
    """(subdivision, height, width) of each mesh: sizes fixed by the case, spread over its ranges."""
    g = torch.Generator().manual_seed(case['mix'])
    n = case['meshes']
    sub = torch.randint(case['subdiv_min'], case['subdiv_max'] + 1, (n,), generator=g).tolist()
    lo, hi = math.log(case['res_min']), math.log(case['res_max'])
    side = torch.exp(lo + (hi - lo) * torch.rand(n, 2, generator=g)).int().tolist()
    return [(s, h, w) for s, (h, w) in zip(sub, side)]


def _inputs(case, seed):
    """The random inputs of a case, on the GPU, as a dict."""
    g = _gen(seed)
    path = case['path']
    if path == 'session':
        objs = []
        for i in range(case['objects']):
            v, f = _mesh(case['subdiv'], 0.01, g)
            a = 2.0 * math.pi * i / case['objects']
            m = torch.eye(4)
            m[0, 0] = m[1, 1] = m[2, 2] = 0.6
            m[0, 3], m[2, 3] = 0.35 * math.cos(a), 0.35 * math.sin(a)
            objs.append((v, f, m.cuda(), torch.rand(v.shape[0], 4, generator=g, device='cuda')))
        return {'objects': objs}
    if path == 'uneven':
        pos, tri, res = [], [], []
        items = _uneven_items(case)
        dirs = fibonacci_directions(len(items))
        for (s, h, w), d in zip(items, dirs):
            v, f = _mesh(s, case['noise'], g)
            cam = PerspectiveCamera.looking_at_origin_from(d * _DIST, h=h, w=w)
            pos.append(clip_space(v, (cam.P('cpu') @ cam.V('cpu')).cuda()))
            tri.append(f)
            res.append((h, w))
        n_pix = sum(h * w for h, w in res)
        return {'pos': torch.cat(pos), 'tri': tri, 'n_verts': [p.shape[0] for p in pos], 'res': res,
                'attr': torch.rand(sum(p.shape[0] for p in pos), case['channels'], generator=g, device='cuda'),
                'target': torch.rand(n_pix, case['channels'], generator=g, device='cuda')}
    h, w = case['height'], case['width']
    v, f = _mesh(case['subdiv'], case['noise'], g)
    d = {'verts': v, 'tri': f, 'VP': _view_projection(case.get('views', 1), h, w)}
    if path == 'layers':
        d['VP'] = d['VP'][0]
        d['attr'] = torch.rand(v.shape[0], case['channels'], generator=g, device='cuda')
        d['target'] = torch.rand(1, h, w, 3, generator=g, device='cuda')
    elif path == 'textured':
        n = torch.nn.functional.normalize(v, dim=-1)  # a cylindrical unwrap
        d['attr'] = torch.stack([torch.atan2(n[:, 0], n[:, 2]) / (2 * math.pi) + 0.5, n[:, 1] * 0.5 + 0.5], -1)
        d['texture'] = torch.rand(case['texture'], case['texture'], 3, generator=g, device='cuda')
        d['target'] = torch.rand(case['views'], h, w, 3, generator=g, device='cuda')
        d['density'] = 0.001 * torch.rand(case['views'], h, w, 4, generator=g, device='cuda')
    else:
        d['attr'] = torch.rand(v.shape[0], case['channels'], generator=g, device='cuda')
        if case['grad']:
            d['target'] = torch.rand(case['views'], h, w, case['channels'], generator=g, device='cuda')
    return d


# ----------------------------------------------------------------------------
# the passes
# ----------------------------------------------------------------------------
def _shade(g, rast):
    """Straight-alpha RGBA of a layer from its first four attributes."""
    return g[..., :4]


def _views_pass(s):
    pos = clip_space(s['verts'], s['VP'])
    rast, _ = nvdr.rasterize(s['ctx'], pos, s['tri'], s['res'], grad_db=False)
    col, _ = nvdr.interpolate(s['attr'], rast, s['tri'])
    img = nvdr.antialias(col, rast, pos, s['tri'], topology_hash=s.get('topology'))
    if 'target' not in s:
        return {'image': img, 'rast': rast}
    loss = l2_loss(img, s['target'])
    gv, ga = torch.autograd.grad(loss, [s['verts'], s['attr']])
    return {'loss': loss.detach(), 'image': img.detach(), 'verts': gv, 'attr': ga}


def _textured_pass(s):
    pos = clip_space(s['verts'], s['VP'])
    rast, db = nvdr.rasterize(s['ctx'], pos, s['tri'], s['res'])
    uv, uv_da = nvdr.interpolate(s['attr'], rast, s['tri'], rast_db=db, diff_attrs='all')
    rgb = texture.sample2d(s['texture'], uv, wrap='reflection') * (rast[..., 3:] > 0)
    img = nvdr.antialias(rgb, rast, pos, s['tri'])
    loss = l2_loss(img, s['target']) + l2_loss(uv_da, s['density'])
    gv, ga, gt = torch.autograd.grad(loss, [s['verts'], s['attr'], s['texture']])
    return {'loss': loss.detach(), 'image': img.detach(), 'uv_da': uv_da.detach(), 'verts': gv, 'attr': ga,
            'texture': gt}


def _layers_pass(s):
    pos = clip_space(s['verts'], s['VP'])
    img = layered.render_layers(s['ctx'], pos, s['tri'], s['attr'], s['res'], s['layers'], _shade)
    loss = l2_loss(img, s['target'])
    gv, ga = torch.autograd.grad(loss, [s['verts'], s['attr']])
    return {'loss': loss.detach(), 'image': img.detach(), 'verts': gv, 'attr': ga}


def _uneven_pass(s):
    ub = s['batch']
    rast, boxes = ub.rasterize(s['pos'])
    col = ub.interpolate(s['attr'], rast, boxes)
    img = ub.antialias(col, rast, s['pos'])
    loss = l2_loss(img, s['target'])
    gp, ga = torch.autograd.grad(loss, [s['pos'], s['attr']])
    return {'loss': loss.detach(), 'image': img.detach(), 'pos': gp, 'attr': ga}


def _session_pass(s):
    rp = deferred.SurfaceDeferredRenderSession(s['scene'], s['camera'], ctx=s['ctx'])
    return {'albedo': rp.nvdr_antialias(rp.albedo()), 'normal': rp.false_color_camera_space_normal(),
            'depth': rp.depth()}


_PASS = {'views': _views_pass, 'textured': _textured_pass, 'layers': _layers_pass, 'uneven': _uneven_pass,
         'session': _session_pass}


def prepare(case, seed):
    s = _inputs(case, seed)
    path = case['path']
    s['path'] = path
    s['ctx'] = nvdr.RasterizeCudaContext(torch.device('cuda:0'), prepare_antialias=case.get('prepared', False))
    if path == 'session':
        scene = deferred.Scene()
        for v, f, m, c in s['objects']:
            scene.add_mesh_object(deferred.MeshObject(deferred.DefaultMaterial(), v, f,
                                                      normals=torch.nn.functional.normalize(v, dim=-1), M=m, color=c))
        s['scene'] = scene
        s['camera'] = PerspectiveCamera(h=case['height'], w=case['width'])
        return s
    if path == 'uneven':
        s['batch'] = batch.UnevenBatch(s['ctx'], s['tri'], s['n_verts'], s['res'])
        s['pos'].requires_grad_(True)
        s['attr'].requires_grad_(True)
        return s
    s['res'] = (case['height'], case['width'])
    s['layers'] = case.get('layers')
    if case.get('prepared'):
        s['topology'] = nvdr.antialias_construct_topology_hash(s['tri'])
    if path != 'views' or case['grad']:
        for k in ('verts', 'attr', 'texture'):
            if k in s:
                s[k].requires_grad_(True)
    if case.get('graph'):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                _views_pass(s)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            s['outputs'] = _views_pass(s)
        s['graph'] = graph
    return s


def run(state):
    if 'graph' in state:
        state['graph'].replay()
        return state['outputs']
    return _PASS[state['path']](state)


def work(case):
    """Bytes of the entry points' inputs and outputs, each once, and the operations on them."""
    path = case['path']
    if path == 'uneven':
        items = _uneven_items(case)
    else:
        items = [(case['subdiv'], case['height'], case['width'])] * case.get('views', case.get('objects', 1))
        if path == 'session':
            items = items[:1]
    C = {'textured': 2, 'session': 4}.get(path) or case['channels']
    layers = case.get('layers', 1)
    grad = path != 'session' and case.get('grad', True)
    nbytes = flops = 0
    for s, h, w in items:
        V, F, N = 10 * 4 ** s + 2, 20 * 4 ** s, h * w
        if path == 'session':
            V, F = V * case['objects'], F * case['objects']
        out = 3 if path in ('textured', 'layers') else C  # colour channels
        # rasterize, interpolate: per layer; antialias, loss: once
        nbytes += layers * ((32 + 4 * C) * N + (28 + 4 * C) * V + 24 * F) + (16 + 8 * out) * N + 16 * V + 12 * F
        flops += layers * (60 + 6 * C) * N + 10 * out * N + 40 * V
        if path == 'textured':
            nbytes += (16 + 16 + 8 + 12) * N
        if path == 'session':
            nbytes += 4 * (16 + 2 * 4) * N
        if grad:
            nbytes += layers * ((48 + 4 * C) * N + (32 + 8 * C) * V + 24 * F) + (16 + 20 * out) * N + 48 * V
            flops += layers * (250 + 16 * C) * N + 20 * out * N + 60 * V
            if path == 'textured':
                nbytes += (16 + 16 + 8 + 8 + 12) * N
    if path == 'textured':
        nbytes += (2 if grad else 1) * 12 * case['texture'] ** 2
    return {'bytes': nbytes, 'flops': flops}


# ----------------------------------------------------------------------------
# the same in 64 bits, plain torch
# ----------------------------------------------------------------------------
_NONE = torch.iinfo(torch.int64).max  # the depth key of an empty pixel


def _fma32(a, b, c):
    """float32 a * b + c rounded once."""
    return (a.double() * b.double() + c.double()).float()


def _clip64(verts, VP):
    """Clip positions [n, V, 4]: the float32 buffer's values, gradients through the product in 64 bits."""
    VP = VP.reshape(-1, 4, 4)
    x, y, z = (verts.detach().float()[:, k] for k in range(3))
    rows = []
    for i in range(4):
        m = VP[:, i, :, None]  # [n, 4, 1]
        rows.append(_fma32(m[:, 0], x, _fma32(m[:, 1], y, _fma32(m[:, 2], z, m[:, 3].expand(-1, len(x))))))
    buf = torch.stack(rows, -1).double()
    pos = torch.nn.functional.pad(verts, (0, 1), value=1.0) @ VP.double().transpose(-1, -2)
    return pos + (buf - pos).detach()


def _ndc(n):
    """float32 NDC centres of n pixels."""
    return (2 * torch.arange(n, device='cuda') + 1 - n).float() / torch.tensor(float(n), device='cuda')


def _visible(pos, tri, h, w, above=None):
    """Depth keys [h * w] of the nearest fragments of clip positions [V, 4] (float32 values), strictly behind
    ``above`` where given: (sortable float32 z/w) << 32 | triangle, _NONE where there is none."""
    keys = torch.full((h * w,), _NONE, dtype=torch.int64, device='cuda')
    p = pos.detach().float()
    X = torch.round((p[:, 0] / p[:, 3] + 1.0) * (w * 0.5) * 16.0).long()
    Y = torch.round((p[:, 1] / p[:, 3] + 1.0) * (h * 0.5) * 16.0).long()
    t = tri.long()
    area = (X[t[:, 1]] - X[t[:, 0]]) * (Y[t[:, 2]] - Y[t[:, 0]]) - (X[t[:, 2]] - X[t[:, 0]]) * (Y[t[:, 1]] - Y[t[:, 0]])
    ccw = torch.where((area > 0)[:, None], t, t[:, [0, 2, 1]])
    tx, ty = X[t], Y[t]
    c0, c1 = (-((8 - tx.amin(1)).div(16, rounding_mode='floor'))).clamp(min=0), \
        (tx.amax(1) - 8).div(16, rounding_mode='floor').clamp(max=w - 1)
    r0, r1 = (-((8 - ty.amin(1)).div(16, rounding_mode='floor'))).clamp(min=0), \
        (ty.amax(1) - 8).div(16, rounding_mode='floor').clamp(max=h - 1)
    count = torch.where(area != 0, (c1 - c0 + 1).clamp(min=0) * (r1 - r0 + 1).clamp(min=0), 0)
    live = count.nonzero()[:, 0]
    ends = count[live].cumsum(0)
    px, py = _ndc(w), _ndc(h)
    total, start = int(ends[-1]) if len(live) else 0, 0
    while start < total:  # at most about 2^24 (triangle, pixel) candidates at a time
        stop = min(total, start + (1 << 24))
        k = torch.arange(start, stop, device='cuda')
        i = torch.searchsorted(ends, k, right=True)
        f = live[i]
        k = k - (ends[i] - count[f])
        bw = c1[f] - c0[f] + 1
        c, r = c0[f] + k % bw, r0[f] + k // bw
        sx, sy = 16 * c + 8, 16 * r + 8
        ok = torch.ones_like(f, dtype=torch.bool)
        for e in range(3):
            a, b = ccw[f, e], ccw[f, (e + 1) % 3]
            dx, dy = X[b] - X[a], Y[b] - Y[a]
            edge = dx * (sy - Y[a]) - dy * (sx - X[a])
            ok &= (edge > 0) | ((edge == 0) & ((dy < 0) | ((dy == 0) & (dx < 0))))
        f, c, r = f[ok], c[ok], r[ok]
        v = p[t[f]]  # [m, 3, 4]
        ax = _fma32(-v[..., 3], px[c][:, None], v[..., 0])
        ay = _fma32(-v[..., 3], py[r][:, None], v[..., 1])
        e = [_fma32(ax[:, (j + 1) % 3], ay[:, (j + 2) % 3], -(ax[:, (j + 2) % 3] * ay[:, (j + 1) % 3]))
             for j in range(3)]
        zn = _fma32(e[0], v[:, 0, 2], _fma32(e[1], v[:, 1, 2], e[2] * v[:, 2, 2]))
        wn = _fma32(e[0], v[:, 0, 3], _fma32(e[1], v[:, 1, 3], e[2] * v[:, 2, 3]))
        zw = zn / wn
        keep = ((e[0] + e[1]) + e[2] != 0) & (zw >= -1) & (zw <= 1)
        bits = zw.view(torch.int32)
        key = ((bits ^ ((bits >> 31) & 0x7fffffff)).long() << 32) | f
        pix = r * w + c
        if above is not None:
            keep &= key > above[pix]
        keys.scatter_reduce_(0, pix[keep], key[keep], 'amin')
        start = stop
    return keys


class _Frag64:
    """Barycentrics (u, v) and their pixel derivatives at the visible fragments of one image, in 64 bits."""

    def __init__(self, pos, tri, h, w, above=None):
        self.h, self.w, self.tri = h, w, tri.long()
        self.keys = _visible(pos, tri, h, w, above)
        self.pix = (self.keys != _NONE).nonzero()[:, 0]
        self.face = self.keys[self.pix] & 0xffffffff
        hi = (self.keys[self.pix] >> 32).int()
        self.z32 = (hi ^ ((hi >> 31) & 0x7fffffff)).view(torch.float32)
        self.v = pos[self.tri[self.face]]  # [m, 3, 4]
        c, r = self.pix % w, self.pix // w
        px, py = (2 * c + 1 - w).double() / w, (2 * r + 1 - h).double() / h
        W = self.v[..., 3]
        self.X, self.Y = self.v[..., 0] - W * px[:, None], self.v[..., 1] - W * py[:, None]
        X, Y = self.X, self.Y
        self.e = [X[:, (k + 1) % 3] * Y[:, (k + 2) % 3] - X[:, (k + 2) % 3] * Y[:, (k + 1) % 3] for k in range(3)]
        self.s = self.e[0] + self.e[1] + self.e[2]
        self.u, self.t = self.e[0] / self.s, self.e[1] / self.s

    def full(self, values):
        """Fragment values [m, C] as an image [h * w, C], zero elsewhere."""
        out = torch.zeros(self.h * self.w, values.shape[1], dtype=torch.float64, device='cuda')
        return out.index_put((self.pix,), values)

    def rast(self):
        zn = sum(self.e[k] * self.v[:, k, 2] for k in range(3))
        wn = sum(self.e[k] * self.v[:, k, 3] for k in range(3))
        return self.full(torch.stack([self.u, self.t, zn / wn, (self.face + 1).double()], -1))

    def interpolate(self, attr):
        a = attr[self.tri[self.face]]
        return self.full(a[:, 2] + self.u[:, None] * (a[:, 0] - a[:, 2]) + self.t[:, None] * (a[:, 1] - a[:, 2]))

    def db(self):
        """(du/dX, du/dY, dv/dX, dv/dY), pixel units."""
        W, X, Y = self.v[..., 3], self.X, self.Y
        ex = [W[:, (k + 2) % 3] * Y[:, (k + 1) % 3] - W[:, (k + 1) % 3] * Y[:, (k + 2) % 3] for k in range(3)]
        ey = [W[:, (k + 1) % 3] * X[:, (k + 2) % 3] - W[:, (k + 2) % 3] * X[:, (k + 1) % 3] for k in range(3)]
        sx, sy = ex[0] + ex[1] + ex[2], ey[0] + ey[1] + ey[2]
        kx, ky = 2.0 / self.w, 2.0 / self.h
        return ((ex[0] - self.u * sx) / self.s * kx, (ey[0] - self.u * sy) / self.s * ky,
                (ex[1] - self.t * sx) / self.s * kx, (ey[1] - self.t * sy) / self.s * ky)

    def footprint(self, attr):
        """(dA/dX, dA/dY) per channel."""
        a = attr[self.tri[self.face]]
        d0, d1 = a[:, 0] - a[:, 2], a[:, 1] - a[:, 2]
        ux, uy, vx, vy = (x[:, None] for x in self.db())
        return self.full(torch.stack([d0 * ux + d1 * vx, d0 * uy + d1 * vy], -1).flatten(1))

    def antialias(self, color, pos, opposite):
        """[h * w, C] colours blended over the silhouette pairs."""
        h, w = self.h, self.w
        p = pos.detach()
        tri = self.tri
        q = p[tri][:, :, [0, 1, 3]]  # [F, 3, (x, y, w)]
        orient = torch.sign((q[:, 0] * torch.linalg.cross(q[:, 1], q[:, 2])).sum(-1))
        nb = opposite
        silhouette = ((nb < 0) | (orient[nb.clamp(min=0)] != orient[:, None])) & (orient != 0)[:, None]
        screen = torch.stack([(pos[:, 0] / pos[:, 3] + 1) * (w * 0.5), (pos[:, 1] / pos[:, 3] + 1) * (h * 0.5)], -1)
        ids = torch.full((h * w,), -1, dtype=torch.int64, device='cuda')
        ids[self.pix] = self.face
        z = torch.full((h * w,), math.inf, device='cuda')
        z[self.pix] = self.z32
        grid = torch.arange(h * w, device='cuda').view(h, w)
        out = color
        for a, b in ((grid[:, :-1].reshape(-1), grid[:, 1:].reshape(-1)), (grid[:-1].reshape(-1), grid[1:].reshape(-1))):
            pair = ids[a] != ids[b]
            a, b = a[pair], b[pair]
            # candidates: the nearer fragment's triangle first, then the other's
            a_first = (ids[a] >= 0) & ~((ids[b] >= 0) & (z[b] < z[a]))
            done = torch.zeros_like(a_first)
            for turn in range(2):
                from_a = a_first if turn == 0 else ~a_first
                src, dst = torch.where(from_a, a, b), torch.where(from_a, b, a)
                use = ((ids[src] >= 0) & ~done).nonzero()[:, 0]
                s, d = src[use], dst[use]
                f = ids[s]
                f_xy, d_xy = (torch.stack([(k % w).double() + 0.5, (k // w).double() + 0.5], -1) for k in (s, d))
                best = torch.full((len(use),), math.inf, dtype=torch.float64, device='cuda')
                edge = torch.full((len(use),), -1, dtype=torch.int64, device='cuda')

                def crossing(f, e, f_xy, d_xy, screen):
                    p0, p1 = screen[tri[f, e]], screen[tri[f, (e + 1) % 3]]
                    ev = p1 - p0
                    ff = (ev[:, 0] * (f_xy[:, 1] - p0[:, 1]) - ev[:, 1] * (f_xy[:, 0] - p0[:, 0])) * orient[f]
                    ft = (ev[:, 0] * (d_xy[:, 1] - p0[:, 1]) - ev[:, 1] * (d_xy[:, 0] - p0[:, 0])) * orient[f]
                    return ff, ft
                flat = screen.detach()
                for e in range(3):
                    ff, ft = crossing(f, torch.full_like(f, e), f_xy, d_xy, flat)
                    te = ff / (ff - ft)
                    take = (ft < 0) & (te < best)
                    best, edge = torch.where(take, te, best), torch.where(take, e, edge)
                hit = (edge >= 0) & silhouette[f, edge.clamp(min=0)]
                done[use[hit]] = True
                s, d, f, edge, f_xy, d_xy = s[hit], d[hit], f[hit], edge[hit], f_xy[hit], d_xy[hit]
                ff, ft = crossing(f, edge, f_xy, d_xy, screen)
                te = ff / (ff - ft)
                inside = (te >= 0) & (te <= 1)
                te = torch.where(inside, te, te.detach().clamp(0, 1))
                near = te.detach() < 0.5
                recv, give = torch.where(near, s, d), torch.where(near, d, s)
                wgt = torch.where(near, 0.5 - te, te - 0.5)[:, None]
                out = out.index_add(0, recv, wgt * (color[give] - color[recv]))
        return out


def _opposite(tri):
    """[F, 3] the other triangle of each edge, -1 where the edge has not exactly two."""
    t = tri.long()
    n = len(t)
    a, b = t.flatten(), t[:, [1, 2, 0]].flatten()
    key = torch.minimum(a, b) * (int(t.max()) + 1) + torch.maximum(a, b)
    order = key.argsort(stable=True)
    _, counts = torch.unique_consecutive(key[order], return_counts=True)
    start = (counts.cumsum(0) - counts)[counts == 2]
    i, j = order[start], order[start + 1]
    opp = torch.full((3 * n,), -1, dtype=torch.int64, device='cuda')
    opp[i], opp[j] = j // 3, i // 3
    return opp.view(n, 3)


def _sample64(tex, uv):
    """Bilinear sample of [H, W, C] at uv [m, 2], (0, 0) the bottom-left corner, reflected borders."""
    grid = torch.stack([uv[:, 0] * 2 - 1, 1 - uv[:, 1] * 2], -1)
    out = torch.nn.functional.grid_sample(tex.permute(2, 0, 1)[None], grid[None, None], mode='bilinear',
                                          padding_mode='reflection', align_corners=False)
    return out[0, :, 0].t()


def _image_items(case, d):
    """(clip positions, triangles, height, width, attribute rows, target) of each image, on 64-bit leaves."""
    if case['path'] == 'uneven':
        pos, attr = d['pos'].double().requires_grad_(True), d['attr'].double().requires_grad_(True)
        vb = pb = 0
        items = []
        for tri, nv, (h, w) in zip(d['tri'], d['n_verts'], d['res']):
            items.append((pos[vb:vb + nv], tri, h, w, attr[vb:vb + nv], d['target'][pb:pb + h * w].double()))
            vb, pb = vb + nv, pb + h * w
        return {'pos': pos, 'attr': attr}, items
    verts, attr = d['verts'].double().requires_grad_(True), d['attr'].double().requires_grad_(True)
    pos = _clip64(verts, d['VP'])
    h, w = case['height'], case['width']
    tgt = d.get('target')
    return {'verts': verts, 'attr': attr}, \
        [(pos[i], d['tri'], h, w, attr, None if tgt is None else tgt[i].double().view(h * w, -1))
         for i in range(len(pos))]


def exact(case, seed):
    path = case['path']
    if path == 'session':
        return None  # its clip transform is a library product: coverage depends on that product's own rounding
    d = _inputs(case, seed)
    leaves, items = _image_items(case, d)
    tex = d['texture'].double().requires_grad_(True) if path == 'textured' else None
    if tex is not None:
        leaves['texture'] = tex
    grad = path != 'views' or case['grad']
    total = 0.0
    sums = {k: torch.zeros_like(v) for k, v in leaves.items()}
    images, extra = [], []
    opposite = {}
    for i, (pos, tri, h, w, attr, target) in enumerate(items):
        if id(tri) not in opposite:
            opposite[id(tri)] = _opposite(tri)
        frag = _Frag64(pos, tri, h, w)
        loss = 0.0
        if path == 'layers':
            first, rgb, trans = frag, 0.0, 1.0
            for k in range(case['layers']):
                g = frag.interpolate(attr)
                a = g[:, 3:4]
                rgb = rgb + trans * a * g[:, :3]
                trans = trans * (1.0 - a)
                if k + 1 < case['layers']:
                    frag = _Frag64(pos, tri, h, w, above=frag.keys)
            frag = first
        else:
            rgb = frag.interpolate(attr)
        if path == 'textured':
            da = frag.footprint(attr)
            extra.append(da.detach())
            loss = ((da - d['density'][i].double().view(h * w, 4)) ** 2).sum()
            rgb = _sample64(tex, rgb) * (frag.keys != _NONE)[:, None]
        img = frag.antialias(rgb, pos, opposite[id(tri)])
        images.append(img.detach())
        if not grad:
            extra.append(frag.rast().detach())
            continue
        loss = loss + ((img - target) ** 2).sum()
        for k, g in zip(leaves, torch.autograd.grad(loss, list(leaves.values()), retain_graph=i + 1 < len(items))):
            sums[k] += g
        total = total + loss.detach()
        del frag, rgb, img, loss
    if path == 'uneven':
        return {'loss': total, 'image': torch.cat(images), **sums}
    shape = (len(items), case['height'], case['width'], -1)
    image = torch.stack(images).view(shape)
    if not grad:
        return {'image': image, 'rast': torch.stack(extra).view(shape)}
    out = {'loss': total, 'image': image, **sums}
    if path == 'textured':
        out['uv_da'] = torch.stack(extra).view(shape)
    return out
