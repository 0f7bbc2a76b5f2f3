"""Workloads of difftetvr_amd as its users run them, for timing and for comparing results.

Each case is one pass a program makes again and again: a forward render, an optimisation step (forward, MSE loss,
adjoint into the mesh's gradients), a batch of either, the parameter update between two steps, or a burst of
requests to the render server.  Meshes are the library's own synthetic ones: jittered cube grids of 6 tets per
cube with a blob colour field, and Delaunay balls with value-noise density.  Cameras look at the origin.

``exact`` evaluates the same quantities in float64 with plain torch: which pixels a face covers and the depth
order are decided in float32 arithmetic as the renderers define them (they are part of the definition), everything
continuous is float64, and gradients come from autograd.
"""
import math

import numpy as np
import torch

import difftetvr_amd as dtv
from difftetvr_amd import meshgen, optim
from difftetvr_amd.serve import Server

FOVY, ZNEAR, ZFAR = math.pi / 4.0, 0.01, 100.0
ATTENUATION = 1.0
ERT_ALPHA = 1.0 - 1e-4  # the renderers' default early ray termination, used with gradients
LR_POSITIONS, LR_COLORS, ADAM_EPS = 1e-4, 1e-3, 1e-8
REG_LAMBDA, REG_BETA = 0.1, 5.0
RENDERERS = {"ppll": dtv.RendererType.PPLL, "projection": dtv.RendererType.PROJECTION,
             "intersection": dtv.RendererType.INTERSECTION}


def listed():
    return [
        # a preview of a toy mesh, as in an interactive viewer or a unit test: latency and launches
        {"name": "render_small", "kind": "render", "mesh": "grid", "n": 8, "width": 96, "height": 64,
         "renderer": "ppll", "storage": "vertex"},
        # the small optimisation problem (24,576 tets at 256 x 256) through the autograd module and torch's loss
        {"name": "step_small", "kind": "step", "mesh": "grid", "n": 16, "width": 256, "height": 256,
         "renderer": "intersection", "storage": "vertex", "loss": "module", "adjoint": "exact"},
        # per-cell colours with the reference's default renderer, at a viewport that is no multiple of a tile
        {"name": "step_cells", "kind": "step", "mesh": "grid", "n": 32, "width": 507, "height": 389,
         "renderer": "ppll", "storage": "cell", "loss": "fused", "adjoint": "exact"},
        # the headline: 1,572,864 tets at 1024 x 1024
        {"name": "step_large", "kind": "step", "mesh": "grid", "n": 64, "width": 1024, "height": 1024,
         "renderer": "intersection", "storage": "vertex", "loss": "fused", "adjoint": "exact"},
        # an unstructured mesh with slivers and deep rays
        {"name": "step_ball", "kind": "step", "mesh": "ball", "n": 20000, "width": 768, "height": 768,
         "renderer": "intersection", "storage": "vertex", "loss": "fused", "adjoint": "exact"},
        # projected tetrahedra, small and at the headline's size
        {"name": "projection_small", "kind": "step", "mesh": "grid", "n": 24, "width": 333, "height": 250,
         "renderer": "projection", "storage": "vertex", "loss": "module", "adjoint": "exact"},
        {"name": "projection_large", "kind": "step", "mesh": "grid", "n": 64, "width": 1024, "height": 1024,
         "renderer": "projection", "storage": "vertex", "loss": "fused", "adjoint": "exact"},
        # a multi-view step: 16 cameras around the large mesh in one batch
        {"name": "views_16", "kind": "batch", "mesh": "grid", "n": 64, "views": 16, "width": 512, "height": 512,
         "renderer": "intersection", "storage": "vertex"},
        # meshes and viewports of uneven size in one batch
        {"name": "uneven_batch", "kind": "uneven", "mesh": "ball", "n": 8000, "views": 5, "width": 450,
         "height": 450, "renderer": "intersection", "storage": "vertex"},
        # an evaluation render of a mesh larger than the headline's, without early ray termination
        {"name": "render_hd", "kind": "render", "mesh": "grid", "n": 96, "width": 1920, "height": 1080,
         "renderer": "intersection", "storage": "vertex"},
        # what lies between two steps: the tet regulariser's gradient and the fused Adam update
        {"name": "update", "kind": "update", "mesh": "grid", "n": 64, "storage": "vertex"},
        # requests of mixed size that reach the render server together
        {"name": "serve_burst", "kind": "serve", "mesh": "grid", "n": 40, "views": 24, "width": 1024,
         "height": 1024, "renderer": "intersection", "storage": "vertex"},
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["render", "step", "step", "step", "step", "step", "batch", "batch", "uneven", "update"])
    mesh = "ball" if kind == "uneven" else rng.choice(["grid", "grid", "grid", "ball"])
    if kind == "update":
        mesh = "grid"
    # (a Delaunay mesh's number of cells, and so the shape of its cell colours, depends on the seed)
    storages = ["vertex", "vertex", "cell"] if mesh == "grid" else ["vertex"]
    c = {"kind": kind, "mesh": mesh, "storage": rng.choice(storages)}
    if kind == "update":
        c["n"] = _spread(rng, 6, 80)
        return c
    c["renderer"] = rng.choice(["intersection", "intersection", "ppll", "projection"])
    if kind in ("render", "step"):
        c["n"] = _spread(rng, 6, 72) if mesh == "grid" else _spread(rng, 300, 20000)
        c["width"], c["height"] = _spread(rng, 48, 1200), _spread(rng, 48, 1200)
    else:
        c["n"] = _spread(rng, 8, 48) if mesh == "grid" else _spread(rng, 300, 8000)
        c["views"] = rng.randint(2, 12 if kind == "batch" else 5)
        c["width"], c["height"] = _spread(rng, 48, 512), _spread(rng, 48, 512)
    if kind == "step":
        c["loss"] = rng.choice(["module", "fused"])
        plain = c["renderer"] == "intersection" and c["storage"] == "vertex"
        c["adjoint"] = rng.choice(["exact", "exact", "abs"] + (["reference"] if plain else []))
    return c


# ---------------------------------------------------------------------------------------------------------------
# Inputs, from the seed alone.

def _eye(rng, radius):
    while True:
        e = rng.normal(size=3)
        e /= np.linalg.norm(e)
        if abs(e[1]) < 0.95:
            return tuple(radius * e)


def _arrays(kind, n, storage, seed):
    """cells int32 [T,4], positions float32 [V,3], colours float32 [V,4] or [T,4]."""
    rng = np.random.default_rng(seed)
    if kind == "grid":
        pos, cells = meshgen.hex_grid((-0.5, -0.5, -0.5), (0.5, 0.5, 0.5), n + 1, n + 1, n + 1)
        inside = (np.abs(pos) < 0.5 - 0.25 / n).all(axis=1)
        field = pos
        pos = pos + (inside[:, None] * rng.uniform(-0.2 / n, 0.2 / n, size=pos.shape)).astype(np.float32)
    else:
        pos, cells = meshgen.delaunay_ball(n, seed=seed)
        field = pos
    if storage == "cell":
        field = field[cells].mean(axis=1)
    col = meshgen.blob_colors(field if kind == "grid" else 0.5 * field, seed=seed + 1)
    if kind == "ball":
        col[:, 3] = meshgen.value_noise(field, seed=seed + 2, vmax=40.0)
    return cells, pos, col


def _mesh(kind, n, storage, seed, gradients):
    cells, pos, col = _arrays(kind, n, storage, seed)
    m = dtv.TetMesh()
    m.set_use_gradients(gradients)
    if storage == "cell":
        m.set_tet_mesh_data(cells, pos, cell_colors=col)
    else:
        m.set_tet_mesh_data(cells, pos, col)
    return m


def _colors(mesh):
    cell = mesh.get_color_storage() == dtv.ColorStorage.PER_CELL
    return mesh.get_cell_colors() if cell else mesh.get_vertex_colors()


def _radius(case):
    return 2.0 if case["mesh"] == "grid" else 3.0


def _target(height, width, rng):
    low = torch.from_numpy(rng.uniform(0.0, 1.0, size=(1, 4, 9, 9)).astype(np.float32))
    t = torch.nn.functional.interpolate(low, size=(height, width), mode="bilinear", align_corners=True)
    return t[0].permute(1, 2, 0).contiguous().cuda()


def _items(case, seed):
    """(mesh seed, points or cubes, eye, width, height) per view of a batch or request of a burst."""
    rng = np.random.default_rng(seed + 77)
    n, w, h = case["n"], case["width"], case["height"]
    if case["kind"] == "batch":
        eyes = meshgen.fibonacci_sphere(case["views"], _radius(case)) + rng.uniform(-0.05, 0.05, size=3)
        return [(seed, n, tuple(e), w, h) for e in eyes]
    if case["kind"] == "uneven":
        return [(seed + 10 * i, max(300, n >> i), _eye(rng, _radius(case)), max(33, w - 61 * i), max(33, h - 29 * i))
                for i in range(case["views"])]
    if case["kind"] == "serve":
        sizes = [(w, h), (w // 2, h // 2), (w // 4, h // 4)]
        return [(seed + 10 * (i % 4), max(4, n - 8 * (i % 4)), _eye(rng, rng.uniform(1.5, 3.0)), *sizes[i % 3])
                for i in range(case["views"])]
    return [(seed, n, _eye(rng, _radius(case)), w, h)]


def _setup(r):
    r.set_attenuation(ATTENUATION)
    r.set_camera_fovy(FOVY)


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed + 5)
    if kind == "update":
        mesh = _mesh(case["mesh"], case["n"], case["storage"], seed, True)
        pos, col = mesh.get_vertex_positions(), _colors(mesh)
        grads = [torch.from_numpy(rng.normal(0.0, s, size=tuple(p.shape)).astype(np.float32)).cuda()
                 for p, s in ((pos, 1e-3), (col, 1e-4))]
        adam = optim.FusedAdam([{"params": [pos], "lr": LR_POSITIONS},
                                {"params": [col], "lr": LR_COLORS, "clamp_nonneg": True}], eps=ADAM_EPS)
        return {"kind": kind, "mesh": mesh, "grads": grads, "adam": adam,
                "regularizer": dtv.TetRegularizer(mesh, REG_LAMBDA, REG_BETA)}
    items = _items(case, seed)
    meshes = {}
    for mseed, n, _, _, _ in items:
        if mseed not in meshes:
            meshes[mseed] = _mesh(case["mesh"], n, case["storage"], mseed, kind not in ("render", "serve"))
    views = [(meshes[i[0]], meshgen.look_at_view_matrix(i[2]), i[3], i[4]) for i in items]
    state = {"kind": kind, "meshes": list(meshes.values())}
    if kind == "serve":
        server = Server(num_workers=4, max_batch=8, attenuation=ATTENUATION, fovy=FOVY)
        ids = {id(m): server.add_mesh(m) for m in state["meshes"]}
        state.update(server=server, requests=[(ids[id(m)], v, w, h) for m, v, w, h in views])
        return state
    if kind in ("batch", "uneven"):
        r = dtv.BatchRenderer(RENDERERS[case["renderer"]])
        _setup(r)
        r.set_items(views)
        state["targets"] = [_target(h, w, rng) for _, _, w, h in views]
        if kind == "batch":
            state["targets"] = torch.stack(state["targets"])
    else:
        r = dtv.Renderer(RENDERERS[case["renderer"]])
        _setup(r)
        mesh, view, w, h = views[0]
        r.set_viewport_size(w, h)
        r.set_view_matrix(view)
        r.set_tet_mesh(mesh)
        if kind == "step":
            state["target"] = _target(h, w, rng)
            state["abs"] = case["adjoint"] == "abs"
            if case["adjoint"] == "reference":
                r.set_adjoint_mode("reference")
            if case["loss"] == "module":
                state["module"] = dtv.DifferentiableRenderer(r)
                state["module"].set_use_abs_grad(state["abs"])
                state["loss"] = torch.nn.MSELoss()
    state["renderer"] = r
    return state


# ---------------------------------------------------------------------------------------------------------------
# One pass.

def _zero_grads(state):
    for m in state["meshes"]:
        m.get_vertex_positions().grad.zero_()
        _colors(m).grad.zero_()


def _grads(state):
    return [t.grad for m in state["meshes"] for t in (m.get_vertex_positions(), _colors(m))]


def run(state):
    kind = state["kind"]
    if kind == "render":
        return state["renderer"].render()
    if kind == "serve":
        server = state["server"]
        tickets = [server.submit(*q) for q in state["requests"]]
        return [server.wait(t)[0] for t in tickets]
    if kind == "update":
        mesh = state["mesh"]
        pos, col = mesh.get_vertex_positions(), _colors(mesh)
        pos.grad.copy_(state["grads"][0])
        col.grad.copy_(state["grads"][1])
        state["regularizer"].compute_grad()
        state["adam"].step()
        st = state["adam"].state
        return {"grad": pos.grad, "params": [pos, col], "m": [st[pos]["exp_avg"], st[col]["exp_avg"]],
                "v": [st[pos]["exp_avg_sq"], st[col]["exp_avg_sq"]]}
    _zero_grads(state)
    if kind == "step":
        if "module" in state:
            image = state["module"]()
            loss = state["loss"](image, state["target"])
            loss.backward()
        else:
            r = state["renderer"]
            image = r.render()
            loss, dimage = optim.mse_loss_grad(image, state["target"])
            r.render_adjoint(dimage, state["abs"])
        return {"image": image, "loss": loss, "grads": _grads(state)}
    r = state["renderer"]
    images = r.render()
    if kind == "batch":
        loss, dimages = optim.mse_loss_grad_views(images, state["targets"])
    else:
        pairs = [optim.mse_loss_grad(i, t) for i, t in zip(images, state["targets"])]
        loss, dimages = [p[0] for p in pairs], [p[1] for p in pairs]
    r.render_adjoint(dimages)
    return {"image": images, "loss": loss, "grads": _grads(state)}


# ---------------------------------------------------------------------------------------------------------------
# What a pass cannot do without.

def _counts(case, n):
    if case["mesh"] == "grid":
        return 6 * n ** 3, (n + 1) ** 3
    return int(6.7 * n), n


def _segments(case, n, width, height):
    """Ray-tet segments: half the face area crossed per unit length (Cauchy), times the volume, over the pixel's
    area at the mesh's distance."""
    pixel = 2.0 * math.tan(0.5 * FOVY) * _radius(case) / height
    if case["mesh"] == "grid":
        crossings, solid, volume = 3.62 * n, 1.0, 1.0
    else:
        solid = volume = 4.0 * math.pi / 3.0
        crossings = 4.04 * (n / solid) ** (1.0 / 3.0)
    # the part of the mesh outside a tall viewport is not crossed
    seen = min(1.0, width / height / (0.6 if case["mesh"] == "grid" else 0.8))
    return crossings * volume * seen / pixel ** 2


def _edge_pixels(case, n, height):
    pixel = 2.0 * math.tan(0.5 * FOVY) * _radius(case) / height
    return (1.0 / n if case["mesh"] == "grid" else (4.0 * math.pi / 3.0 / n) ** (1.0 / 3.0)) / pixel


def work(case):
    # flops a segment: entry and exit of the ray (planes, barycentrics, colours) and its four sub-segments, about
    # 250 forward and 400 more backward; a projected-tetrahedra fragment about 40 and 80
    forward, backward = (40, 80) if case.get("renderer") == "projection" else (250, 400)
    if case["kind"] == "update":
        T, V = _counts(case, case["n"])
        params = 3 * V + 4 * (T if case["storage"] == "cell" else V)
        return {"bytes": 16 * T + 24 * V + 28 * params + 8 * params, "flops": 200 * T + 12 * params}
    total = {"bytes": 0, "flops": 0}
    known = set()
    for mseed, n, _, w, h in _items(case, 0):
        T, V = _counts(case, n)
        colors = 16 * (T if case["storage"] == "cell" else V)
        grad = case["kind"] not in ("render", "serve")
        if mseed not in known:
            total["bytes"] += 16 * T + (12 * V + colors) * (2 if grad else 1)
            known.add(mseed)
        total["bytes"] += 16 * w * h * (3 if grad else 1)
        total["flops"] += _segments(case, n, w, h) * (forward + (backward if grad else 0))
    return total


# ---------------------------------------------------------------------------------------------------------------
# The same in 64 bits.

FACES = [[0, 1, 2], [1, 0, 3], [0, 2, 3], [2, 1, 3]]
MOST_SEGMENTS = 1.2e8  # beyond this the float64 evaluation takes too long


class _Sliver(Exception):
    """A projected triangle thinner than the screen's 1/256 pixel grid: its pixels lie far outside the true triangle,
    where the interpolation has no stable value."""


class _Camera:
    def __init__(self, view, width, height, dev):
        V = torch.tensor(view, dtype=torch.float64, device=dev).reshape(4, 4).t()
        th = math.tan(0.5 * float(np.float32(FOVY)))
        zn, zf = float(np.float32(ZNEAR)), float(np.float32(ZFAR))
        P = torch.zeros(4, 4, dtype=torch.float64, device=dev)
        P[0, 0], P[1, 1], P[3, 2] = height / (width * th), -1.0 / th, -1.0
        P[2, 2], P[2, 3] = zf / (zn - zf), -(zf * zn) / (zf - zn)
        self.VP, self.iP, iV = P @ V, torch.linalg.inv(P), torch.linalg.inv(V)
        self.iV, self.eye, self.axis = iV, iV[:3, 3], -V[2, :3]
        self.width, self.height = width, height

    def ndc(self, p, dtype):
        """Normalised device coordinates [..., 3], each product and sum rounded by itself."""
        M = self.VP.to(dtype)
        p = p.to(dtype)
        c = [((M[r, 0] * p[..., 0] + M[r, 1] * p[..., 1]) + M[r, 2] * p[..., 2]) + M[r, 3] for r in range(4)]
        return torch.stack([c[0] / c[3], c[1] / c[3], c[2] / c[3]], dim=-1)

    def pixel(self, pix):
        x = (pix % self.width).double() + 0.5
        y = torch.div(pix, self.width, rounding_mode="floor").double() + 0.5
        return 2.0 * (x / self.width) - 1.0, 2.0 * (y / self.height) - 1.0

    def rays(self, pix):
        nx, ny = self.pixel(pix)
        one = torch.ones_like(nx)
        d = torch.stack([nx, ny, one, one], dim=-1) @ self.iP[:3].t()
        return (d / d.norm(dim=-1, keepdim=True)) @ self.iV[:3, :3].t()


def _screen(ndc, cam):
    """Corner pixels in 1/256 [N,3] of float32 triangles [N,3,>=2], turned to positive area."""
    hw, hh = 0.5 * cam.width, 0.5 * cam.height
    X = torch.round((ndc[..., 0] * hw + hw) * 256.0).long()
    Y = torch.round((ndc[..., 1] * hh + hh) * 256.0).long()
    area = (X[:, 1] - X[:, 0]) * (Y[:, 2] - Y[:, 0]) - (Y[:, 1] - Y[:, 0]) * (X[:, 2] - X[:, 0])
    turn = torch.tensor([0, 2, 1], device=X.device)
    back = (area < 0)[:, None]
    return torch.where(back, X[:, turn], X), torch.where(back, Y[:, turn], Y), area != 0


def _covered(X, Y, live, width, y0, y1):
    """(triangle, pixel) pairs whose pixel centre lies in the triangle, rows y0 <= y < y1."""
    def low(v):
        return -torch.div(128 - v, 256, rounding_mode="floor")

    def high(v):
        return torch.div(v - 128, 256, rounding_mode="floor")
    ax, bx = low(X.min(1)[0]).clamp(min=0), high(X.max(1)[0]).clamp(max=width - 1)
    ay, by = low(Y.min(1)[0]).clamp(min=y0), high(Y.max(1)[0]).clamp(max=y1 - 1)
    w, h = (bx - ax + 1).clamp(min=0), (by - ay + 1).clamp(min=0)
    count = w * h * live
    tri = torch.repeat_interleave(torch.arange(X.shape[0], device=X.device), count)
    first = torch.cumsum(count, 0) - count
    k = torch.arange(tri.shape[0], device=X.device) - first[tri]
    row = torch.div(k, w[tri], rounding_mode="floor")
    x, y = ax[tri] + k - row * w[tri], ay[tri] + row
    inside = torch.ones_like(x, dtype=torch.bool)
    for a, b in ((0, 1), (1, 2), (2, 0)):
        dx, dy = (X[:, b] - X[:, a])[tri], (Y[:, b] - Y[:, a])[tri]
        e = dx * (256 * y + 128 - Y[tri, a]) - dy * (256 * x + 128 - X[tri, a])
        inside &= (e > 0) | ((e == 0) & ((dy < 0) | ((dy == 0) & (dx > 0))))
    return tri[inside], (y * width + x)[inside]


def _faces(cells, p32, cam):
    """Front faces of all tets: (tet, face), screen corners, depth keys."""
    tv = p32[cells]
    eye = cam.eye.float()
    ndc = cam.ndc(tv, torch.float32)
    tets, faces, corners, keys = [], [], [], []
    for f, (a, b, c) in enumerate(FACES):
        o = 6 - a - b - c
        n = torch.linalg.cross(tv[:, b] - tv[:, a], tv[:, c] - tv[:, a])
        d = -(n * tv[:, a]).sum(-1)
        sc, so = torch.sign(n @ eye + d), torch.sign((n * tv[:, o]).sum(-1) + d)
        t = ((sc != 0) & (sc != so)).nonzero()[:, 0]
        q = ndc[t][:, [a, b, c]]
        tets.append(t)
        faces.append(torch.full_like(t, f))
        corners.append(q)
        keys.append(((q[:, 0, 2] + q[:, 1, 2]) + q[:, 2, 2]) / 3.0)
    t, f, q, k = (torch.cat(v) for v in (tets, faces, corners, keys))
    by = torch.argsort(t * 4 + f)
    return t[by], q[by], k[by]


def _pick(rows, index):
    """rows [F,R,...], index [F,...k]: rows[f, index[f]]."""
    return rows[torch.arange(rows.shape[0], device=rows.device).reshape(-1, *[1] * (index.dim() - 1)), index]


def _tet_values(p, c, rd, cam, linear, per_cell):
    """(colour part, optical depth, hit) of rays rd through tets p [F,4,3] with colours c [F,4,4] or [F,4]."""
    faces = torch.tensor(FACES, device=p.device)
    v = p[:, faces]  # [F, face, corner, 3]
    n = torch.linalg.cross(v[:, :, 1] - v[:, :, 0], v[:, :, 2] - v[:, :, 0])
    den = (n * rd[:, None]).sum(-1)
    t = -(n * (cam.eye - v[:, :, 0])).sum(-1) / den
    outward = ((n[:, 0] * (p[:, 3] - p[:, 0])).sum(-1) < 0)[:, None]
    entering = torch.where(outward, den < 0, den > 0)
    inf = float("inf")
    fi = torch.where(entering, t, -inf).detach().argmax(1)
    fo = torch.where(entering, inf, t).detach().argmin(1)
    tin, tout = _pick(t, fi), _pick(t, fo)
    hit = (tout >= tin) & (tin >= 0)
    length = (tout - tin) * ((rd * cam.axis).sum(-1) if linear else 1.0)
    if per_cell:
        tau = c[:, 3] * ATTENUATION * length
        return c[:, :3] * (1.0 - torch.exp(-tau))[:, None], tau, hit
    ends = []
    for f, at in ((fi, tin), (fo, tout)):
        q, m = _pick(v, f), _pick(n, f)
        x = cam.eye + at[:, None] * rd
        mm = (m * m).sum(-1)
        u = (m * torch.linalg.cross(q[:, 2] - q[:, 1], x - q[:, 1])).sum(-1) / mm
        w = (m * torch.linalg.cross(q[:, 0] - q[:, 2], x - q[:, 2])).sum(-1) / mm
        k = _pick(c, faces[f])
        ends.append(u[:, None] * k[:, 0] + w[:, None] * k[:, 1] + (1.0 - u - w)[:, None] * k[:, 2])
    c0, c1 = ends
    seg = length / 4.0
    tau, rgb = torch.zeros_like(seg), torch.zeros_like(c0[:, :3])
    for s in range(4):
        a = (c0[:, 3] + (s + 0.5) / 4.0 * (c1[:, 3] - c0[:, 3])) * ATTENUATION
        full = a >= 1e-6
        ia = 1.0 / torch.where(full, a, 1.0)
        part = torch.where(full, a * seg, 0.0)
        A = torch.exp(-part)
        d = c1[:, :3] - c0[:, :3]
        k = (seg + ia) * A - ia
        out = (1.0 - A)[:, None] * (c0[:, :3] + s / 4.0 * d) - (0.25 * k)[:, None] * d
        rgb = rgb + (torch.exp(-tau) * full)[:, None] * out
        tau = tau + part
    return rgb, tau, hit


def _decide(nd):
    """Projected-tetrahedra class of tets with corners nd [T,4,3] (float32): edges, class, reversal, live."""
    e = nd - nd[:, :1]
    v1, v2, v3 = e[:, 1], e[:, 2], e[:, 3]

    def turn(a, b):
        return a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0]
    d1, d2, d3 = turn(v3, v2), turn(v1, v3), turn(v2, v1)
    first = (d1 * d2 >= 0) & ((d1 != 0) | (d2 != 0))
    second = ~first & (d1 * d3 >= 0)
    kind = torch.where(first, 0, torch.where(second, 1, 2))
    seg = torch.tensor([[0, 3, 1, 2], [0, 2, 1, 3], [0, 1, 2, 3]], device=nd.device)[kind]
    A, B, C = _edges(nd, seg)[:3]
    den = turn(A, B)
    alpha = (B[:, 1] * C[:, 0] - B[:, 0] * C[:, 1]) / den
    crossed = (alpha >= 0) & (alpha <= 1)
    return seg, crossed, ~crossed & (alpha <= 0), den.abs() >= 1e-8


def _edges(nd, seg):
    q = _pick(nd, seg)
    return q[:, 1] - q[:, 0], q[:, 3] - q[:, 2], q[:, 2] - q[:, 0], q


def _five(nd, c, decided, cam, per_cell):
    """The five projected vertices of each tet: [T,5,3] positions, [T,5,4] colours, [T,5] thicknesses."""
    seg, crossed, flip, _ = decided
    dtype = nd.dtype
    A, B, C, q = _edges(nd, seg)
    den = A[:, 0] * B[:, 1] - A[:, 1] * B[:, 0]
    alpha = ((B[:, 1] * C[:, 0] - B[:, 0] * C[:, 1]) / den)[:, None]
    beta = ((A[:, 1] * C[:, 0] - A[:, 0] * C[:, 1]) / den)[:, None]
    cross = q[:, 0] + alpha * A
    five = torch.cat([nd, torch.where(crossed[:, None], cross, torch.zeros_like(cross))[:, None]], 1)
    if c is None:
        return five
    k = _pick(c, seg)
    two = crossed[:, None]
    # class 1: the thick corner (segment 1's far end, its near end when reversed) and the corner opposite
    thick, other = torch.where(flip, seg[:, 0], seg[:, 1]), torch.where(flip, seg[:, 1], seg[:, 0])
    al = torch.where(two, torch.ones_like(alpha), torch.where(flip[:, None], 1.0 - alpha, alpha))
    pt, po, ct, co = _pick(nd, thick), _pick(nd, other), _pick(c, thick), _pick(c, other)
    face_z = ((q[:, 2, 2:] + beta * B[:, 2:]) + (al - 1.0) * po[:, 2:]) / al
    xy = torch.where(two, cross[:, :2], pt[:, :2])
    z1 = torch.where(two, cross[:, 2:], pt[:, 2:])
    z2 = torch.where(two, q[:, 2, 2:] + beta * B[:, 2:], face_z)
    one = torch.ones_like(z1)
    e1, e2 = (torch.cat([xy, z, one], 1) @ cam.iP.to(dtype).t() for z in (z1, z2))
    depth = ATTENUATION * (e1[:, :3] / e1[:, 3:] - e2[:, :3] / e2[:, 3:]).norm(dim=1)
    edge = k[:, 2] + beta * (k[:, 3] - k[:, 2])
    col = torch.where(two, 0.5 * (k[:, 0] + alpha * (k[:, 1] - k[:, 0]) + edge),
                      0.5 * ((edge + (al - 1.0) * co) / al + ct))
    slot = torch.where(crossed, 4, thick)
    at = torch.nn.functional.one_hot(slot, 5).bool()
    thickness = torch.where(at, depth[:, None], torch.zeros_like(depth)[:, None])
    colours = torch.cat([c, c[:, :1]], 1)
    if not per_cell:
        colours = torch.where(at[..., None], col[:, None], colours)
    return five, colours, thickness


def _triangles(cells, p32, cam):
    """Triangles of all projected tets: tet, corner slots [N,3], screen corners, depth keys."""
    nd = cam.ndc(p32[cells], torch.float32)
    decided = _decide(nd)
    seg, crossed, flip, live = decided
    five = _five(nd, None, decided, cam, False)
    a0, a1 = torch.where(flip, seg[:, 1], seg[:, 0]), torch.where(flip, seg[:, 0], seg[:, 1])
    b0, b1 = seg[:, 2], seg[:, 3]
    fan2 = torch.stack([torch.full_like(a0, 4), a0, b0, a1, b1, a0], 1)
    fan1 = torch.stack([a1, a0, b0, b1, a0, a0], 1)
    fan = torch.where(crossed[:, None], fan2, fan1)
    tets, slots = [], []
    for k in range(4):
        t = (live & (crossed if k == 3 else torch.ones_like(crossed))).nonzero()[:, 0]
        tets.append(t * 4 + k)
        slots.append(fan[t][:, [0, k + 1, k + 2]])
    t, s = torch.cat(tets), torch.cat(slots)
    by = torch.argsort(t)
    t, s = torch.div(t[by], 4, rounding_mode="floor"), s[by]
    q = five[t[:, None], s]
    return t, s, q, ((q[:, 0, 2] + q[:, 1, 2]) + q[:, 2, 2]) / 3.0, decided


def _exact_view(case, cells, pos, col, view, width, height, target, scale, terminate, gradients):
    """Image [H,W,4] and loss (terminate: with early ray termination); with gradients the loss's gradients are
    accumulated in pos.grad and col.grad."""
    cam = _Camera(view, width, height, pos.device)
    per_cell = case["storage"] == "cell"
    proj = case["renderer"] == "projection"
    p32 = pos.detach().float()
    if proj:
        owner, slots, q, keys, decided = _triangles(cells, p32, cam)
    else:
        owner, q, keys = _faces(cells, p32, cam)
    X, Y, live = _screen(q, cam)
    segments = max(1.0, _segments(case, case["n"], width, height))
    rows = max(1, min(height, int(height * 1.5e6 / segments)))
    image = torch.zeros(height * width, 4, dtype=torch.float64, device=pos.device)
    loss = 0.0
    for y0 in range(0, height, rows):
        y1 = min(height, y0 + rows)
        near = live & (Y.min(1)[0] <= 256 * y1) & (Y.max(1)[0] >= 256 * y0)
        some = near.nonzero()[:, 0]
        tri, pix = _covered(X[some], Y[some], torch.ones_like(some), width, y0, y1)
        tri = some[tri]
        by = torch.argsort(keys[tri], stable=True)
        by = by[torch.argsort(pix[by], stable=True)]
        tri, pix = tri[by], pix[by]
        tet = owner[tri]
        with torch.set_grad_enabled(gradients):
            if proj:
                tets, inv = torch.unique(tet, return_inverse=True)
                nd = cam.ndc(pos[cells[tets]], torch.float64)
                c = col[tets][:, None].expand(-1, 4, -1) if per_cell else col[cells[tets]]
                five, colours, thick = _five(nd, c, [d[tets] for d in decided], cam, per_cell)
                s = slots[tri]
                v, k, d = five[inv[:, None], s], colours[inv[:, None], s], thick[inv[:, None], s]
                px, py = cam.pixel(pix)
                at = torch.stack([px, py], 1)[:, None]
                e = v[..., :2] - at

                def turn(a, b):
                    return a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0]
                area = turn(v[:, 1, :2] - v[:, 0, :2], v[:, 2, :2] - v[:, 0, :2])
                lam = torch.stack([turn(e[:, 1], e[:, 2]), turn(e[:, 2], e[:, 0]), turn(e[:, 0], e[:, 1])], 1)
                lam = lam / area[:, None]
                if lam.numel() and float(lam.detach().abs().max()) > 64.0:
                    raise _Sliver()
                rgba, dep = (lam[..., None] * k).sum(1), (lam * d).sum(1)
                tau = rgba[:, 3] * dep
                rgb = rgba[:, :3] * (1.0 - torch.exp(-tau))[:, None]
                hit = torch.ones_like(tau, dtype=torch.bool)
            else:
                c = col[tet] if per_cell else col[cells[tet]]
                rgb, tau, hit = _tet_values(pos[cells[tet]], c, cam.rays(pix), cam, case["renderer"] == "ppll",
                                            per_cell)
            rgb, tau = rgb * hit[:, None], torch.where(hit, tau, torch.zeros_like(tau))
            here = pix - y0 * width
            n = (y1 - y0) * width
            total = torch.cumsum(tau, 0) - tau
            first = torch.searchsorted(here, torch.arange(n, device=pos.device))
            pad = torch.cat([total, total.new_zeros(1)])
            before = total - pad[first][here]
            alive = torch.ones_like(hit)
            if terminate and not proj:
                alive = 1.0 - torch.exp(-before.detach()) <= ERT_ALPHA
            out = torch.zeros(n, 3, dtype=torch.float64, device=pos.device)
            out = out.index_add(0, here, rgb * (torch.exp(-before) * alive)[:, None])
            depth = torch.zeros(n, dtype=torch.float64, device=pos.device).index_add(0, here, tau * alive)
            band = torch.cat([out, (1.0 - torch.exp(-depth))[:, None]], 1)
            image[y0 * width:y1 * width] = band.detach()
            if target is not None:
                part = ((band - target.reshape(-1, 4)[y0 * width:y1 * width].double()) ** 2).sum() * scale
                loss += float(part.detach())
                if gradients:
                    part.backward()
    return image.reshape(height, width, 4), loss


def _double(kind, n, storage, seed):
    cells, pos, col = _arrays(kind, n, storage, seed)
    pos, col = (torch.from_numpy(a).cuda().double().requires_grad_(True) for a in (pos, col))
    return torch.from_numpy(cells).cuda().long(), pos, col


def _exact_update(case, seed):
    cells, pos, col = _double(case["mesh"], case["n"], case["storage"], seed)
    pos, col = pos.detach(), col.detach()
    rng = np.random.default_rng(seed + 5)
    gp, gc = (torch.from_numpy(rng.normal(0.0, s, size=tuple(p.shape)).astype(np.float32)).cuda().double()
              for p, s in ((pos, 1e-3), (col, 1e-4)))
    p = pos[cells]
    a, b, c = p[:, 1] - p[:, 0], p[:, 2] - p[:, 0], p[:, 3] - p[:, 0]
    D = (torch.linalg.cross(a, b) * c).sum(-1)
    S = sum(((p[:, i] - p[:, j]) ** 2).sum(-1) for i in range(4) for j in range(i + 1, 4))
    k12 = 12.0 * math.sqrt(3.0)
    dq = -REG_LAMBDA / (1.0 + torch.exp(-REG_BETA * k12 * D / S ** 1.5))
    dD = [torch.linalg.cross(b, c), torch.linalg.cross(c, a), torch.linalg.cross(a, b)]
    dD = torch.stack([-(dD[0] + dD[1] + dD[2])] + dD, 1)
    dS = 2.0 * (4.0 * p - p.sum(1, keepdim=True))
    g = (dD * (k12 * S)[:, None, None] - dS * (1.5 * k12 * D)[:, None, None])
    g = g * (-dq / (S ** 2.5).clamp(min=1e-5))[:, None, None]
    gp = gp.index_add(0, cells.reshape(-1), g.reshape(-1, 3))
    new, ms, vs = [], [], []
    for x, y, lr in ((pos, gp, LR_POSITIONS), (col, gc, LR_COLORS)):
        m, v = 0.1 * y, 0.001 * y * y
        new.append(x - lr * (m / 0.1) / (torch.sqrt(v / 0.001) + ADAM_EPS))
        ms.append(m)
        vs.append(v)
    new[1] = new[1].clamp(min=0.0)
    return {"grad": gp, "params": new, "m": ms, "v": vs}


def exact(case, seed):
    kind = case["kind"]
    if kind == "update":
        return _exact_update(case, seed)
    items = _items(case, seed)
    if sum(_segments(case, n, w, h) for _, n, _, w, h in items) > MOST_SEGMENTS:
        return None
    rng = np.random.default_rng(seed + 5)
    grad = kind not in ("render", "serve")
    meshes, images, losses = {}, [], []
    for mseed, n, eye, w, h in items:
        if mseed not in meshes:
            meshes[mseed] = _double(case["mesh"], n, case["storage"], mseed)
        view = meshgen.look_at_view_matrix(eye)
        target = _target(h, w, rng) if grad else None
        try:
            image, loss = _exact_view(dict(case, n=n), *meshes[mseed], view, w, h, target, 1.0 / (4 * w * h), grad,
                                      grad and case.get("adjoint", "exact") == "exact")
        except _Sliver:
            return None
        images.append(image)
        losses.append(loss)
    if not grad:
        return images if kind == "serve" else images[0]
    # a ray that grazes a face gives its vertices an unbounded position gradient; with small tets or many rays
    # such rays dominate the sum, and it has no value that 32-bit decisions and 64-bit ones share
    steady = all(_segments(case, n, w, h) < 2e7 and _edge_pixels(case, n, h) > 6.0 for _, n, _, w, h in items)
    grads = [t.grad if steady or t.shape[1] == 4 else None for m in meshes.values() for t in m[1:]]
    if kind == "step":
        return {"image": images[0], "loss": losses[0], "grads": grads}
    if kind == "batch":
        return {"image": torch.stack(images), "loss": sum(losses), "grads": grads}
    return {"image": images, "loss": losses, "grads": grads}
