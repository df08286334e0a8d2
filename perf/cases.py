"""Performance cases: what a program that uses this path-tracing core has it
do, through the package's public entry points.

A program keeps one device context per scene it works on (tree built and
uploaded once), and calls it with new inputs: ray batches, cameras and sampler
seeds, guide queries and records. `prepare` makes those inputs from the seed;
the scene and its context are shared by the states of a case, as a program
shares them between calls.
"""
import collections
import ctypes as C
import math
import random

import numpy as np
import torch

from swpathtracer_amd import _lib as L
from swpathtracer_amd import api, scenes

HIDDEN, ENC, OUT, OUT_PAD, LOBES = 64, 32, 40, 48, 8


def listed():
    return [
        # a few thousand visibility or picking queries against a small scene:
        # the smallest call, where launch latency is all there is
        {"name": "trace_box_3000", "kind": "trace", "scene": "box", "detail": 5, "rays": "incoherent", "n": 3000},
        # the closest hit of a full-HD frame's primary rays on a 1M-triangle mesh
        {"name": "trace_primary_1080p", "kind": "trace", "scene": "mesh", "detail": 512, "rays": "primary",
         "width": 1920, "height": 1080},
        # a bulk batch of incoherent rays (another integrator's bounces, ambient
        # occlusion, a bake), an odd number of them
        {"name": "trace_incoherent_4m", "kind": "trace", "scene": "mesh", "detail": 512, "rays": "incoherent",
         "n": 4_194_301},
        # the normal ray caster: a modelling preview of the same mesh
        {"name": "raycast_normal_1080p", "kind": "raycast", "scene": "mesh", "detail": 512, "value": "normal",
         "width": 1920, "height": 1080},
        # the plain tracer on the 1M-triangle layered mesh in the box, the
        # benchmark's image: Russian roulette from depth 3, at most 16 bounces
        {"name": "render_mesh_1024spp", "kind": "render", "scene": "mesh", "detail": 512, "width": 800, "height": 600,
         "spp": 1024, "sampler": "jittered", "rr": 3, "depth": 16, "film64": False, "per_path": False},
        # one progressive step of the same image, as an interactive viewer asks for it
        {"name": "render_mesh_4spp", "kind": "render", "scene": "mesh", "detail": 512, "width": 800, "height": 600,
         "spp": 4, "sampler": "jittered", "rr": 3, "depth": 16, "film64": False, "per_path": False},
        # a thumbnail with ragged sides: a render of a few thousand paths
        {"name": "render_box_97x61", "kind": "render", "scene": "box", "detail": 5, "width": 97, "height": 61, "spp": 1,
         "sampler": "uniform", "rr": -1, "depth": 5, "film64": False, "per_path": False},
        # the box + 20,480-triangle icosphere image, 256 x 256, 16 samples, depth 5
        {"name": "render_box_256", "kind": "render", "scene": "box", "detail": 5, "width": 256, "height": 256,
         "spp": 16, "sampler": "jittered", "rr": -1, "depth": 5, "film64": False, "per_path": False},
        # the path guide's network on a batch of hit points
        {"name": "guide_eval_1m", "kind": "eval", "scene": "box", "detail": 3, "n": 1_000_003},
        # the gradient of one training step of the guide at its default batch
        {"name": "guide_gradient_256k", "kind": "gradient", "scene": "box", "detail": 3, "n": 262_144},
        # a guided pass of the slit-lit scene with a kept guide
        {"name": "guided_slit_36spp", "kind": "guided", "scene": "slit", "detail": 256, "width": 400, "height": 300,
         "spp": 36, "flags": 0},
        # a batch of small scenes rendered in one call
        {"name": "batch_8_scenes", "kind": "batch", "n": 8, "side": 192, "spp": 16, "min_tris": 1000,
         "max_tris": 50_000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trace", "trace", "trace", "raycast", "raycast", "render", "render", "render", "render", "eval",
                       "gradient", "guided", "batch"])
    scene = rng.choice(["box", "mesh", "mesh", "spheres", "slit"])
    detail = {"box": rng.randint(2, 6), "mesh": _log_int(rng, 24, 512), "slit": _log_int(rng, 24, 384),
              "spheres": rng.randint(0, 5)}[scene]
    case = {"kind": kind, "scene": scene, "detail": detail}
    if kind in ("trace", "raycast", "render"):
        case["width"], case["height"] = _log_int(rng, 40, 1920), _log_int(rng, 30, 1080)
    if kind == "trace":
        case["rays"] = rng.choice(["incoherent", "primary"]) if scene != "spheres" else "primary"
        if case["rays"] == "incoherent":
            del case["width"], case["height"]
            case["n"] = _log_int(rng, 1000, 8_000_000)
    elif kind == "raycast":
        case["value"] = rng.choice(["normal", "depth", "count"])
    elif kind == "render":
        pixels = case["width"] * case["height"]
        case["spp"] = _log_int(rng, 1, max(1, min(256, 60_000_000 // pixels)))
        case["sampler"] = rng.choice(["jittered", "jittered", "uniform", "regular"])
        case["rr"] = rng.choice([3, 3, 5, -1])
        case["depth"] = rng.choice([16, 8]) if case["rr"] >= 0 else rng.randint(2, 8)
        case["film64"] = rng.random() < 0.2
        case["per_path"] = pixels * math.ceil(math.sqrt(case["spp"])) ** 2 < 4_000_000 and rng.random() < 0.3
    elif kind in ("eval", "gradient"):
        case["scene"], case["detail"] = "box", rng.randint(1, 4)
        case["n"] = _log_int(rng, 1000, 4_000_000 if kind == "eval" else 600_000)
    elif kind == "guided":
        case["scene"], case["detail"] = "slit", _log_int(rng, 24, 256)
        case["width"], case["height"] = _log_int(rng, 40, 800), _log_int(rng, 30, 600)
        case["spp"] = _log_int(rng, 1, max(1, min(64, 20_000_000 // (case["width"] * case["height"]))))
        case["flags"] = rng.choice([0, 0, L.SPT_GUIDE_COATED])
    else:
        del case["scene"], case["detail"]
        case.update(n=rng.randint(2, 12), side=_log_int(rng, 32, 256), spp=rng.choice([1, 4, 16]), min_tris=1000,
                    max_tris=_log_int(rng, 2000, 50_000))
    return case


# ----------------------------------------------------------------------------
# scenes: a program builds and uploads each once
# ----------------------------------------------------------------------------

_FURNACE = ["lambertian", "smooth_conductor", "smooth_dielectric", "cook_torrance", "plastic", "coating"]
_open = collections.OrderedDict()  # the scenes in use: the last two


class _Scene:
    def __init__(self, scene, detail):
        make = {"box": lambda: scenes.cornell_icosphere(subdiv=detail),
                "mesh": lambda: scenes.mesh_in_box(rings=detail, segments=2 * detail),
                "slit": lambda: scenes.slit_box(rings=detail, segments=2 * detail),
                "spheres": lambda: scenes.reference_furnace(_FURNACE[detail]),
                "none": lambda: None}[scene]
        self.data = make()
        self.dev = api.Device(0)
        if self.data is not None:
            bvh = api.Bvh(self.data.verts, kinds=self.data.kinds)
            self.dev.set_scene(bvh, self.data.normals, self.data.mat_ids)
            self.dev.set_materials(self.data.materials)
        # the context's own stream, for work that has to be ordered with its calls
        self.stream = torch.cuda.ExternalStream(self.dev.stream)


def _scene(case):
    key = (case.get("scene", "none"), case.get("detail", 0), case["kind"] in ("guided", "eval", "gradient"))
    if key not in _open:
        while len(_open) > 1:
            _open.popitem(last=False)
        _open[key] = _Scene(*key[:2])
    _open.move_to_end(key)
    return _open[key]


def _camera(case, sc, seed):
    """The scene's camera at the case's size, moved a little by the seed (a frame of a fly-through)."""
    rng = random.Random(seed)
    src = sc.data.camera
    pos = [p + rng.uniform(-0.03, 0.03) for p in src.position]
    w, h = case["width"], case["height"]
    if src.type == L.SPT_CAMERA_ORTHOGRAPHIC:
        return api.orthographic(w, h, src.min_x, src.max_x, src.min_y, src.max_y, position=pos,
                                look_at=list(src.look_at), up=list(src.up))
    return api.pinhole(w, h, position=pos, look_at=list(src.look_at), up=list(src.up), fov=src.fov_deg)


def _box_of(sc):
    v = torch.from_numpy(sc.data.verts).cuda().view(-1, 3)
    return v.amin(0), v.amax(0)


def _unit(g, n):
    v = torch.randn(n, 3, generator=g, device="cuda")
    return v / v.norm(dim=1, keepdim=True)


def _surface_rays(sc, n, g):
    """Origins spread over the scene's surfaces by area and moved off them by
    1e-3 along a direction uniform on the sphere: what bounces look like."""
    v = torch.from_numpy(sc.data.verts).cuda().view(-1, 3, 3)
    area = torch.linalg.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]).norm(dim=1).double().cumsum(0)
    tri = torch.searchsorted(area, torch.rand(n, generator=g, device="cuda").double() * area[-1])
    tri = tri.clamp(max=v.shape[0] - 1)
    r1, r2 = torch.rand(n, 1, generator=g, device="cuda").sqrt(), torch.rand(n, 1, generator=g, device="cuda")
    p = (1 - r1) * v[tri, 0] + r2 * r1 * v[tri, 1] + (1 - r2) * r1 * v[tri, 2]
    d = _unit(g, n)
    rays = torch.zeros(n, 8, device="cuda")
    rays[:, 0:3], rays[:, 4:7] = p + 1e-3 * d, d
    return rays


def _guide_params():
    """Guide parameters as a program loads them: a fixed network whose eight
    lobes are broad, one towards the light above and the others spread."""
    rng = np.random.RandomState(11)
    parts = []
    for fan_in, rows, used, scale in ((ENC, HIDDEN, HIDDEN, 1.0), (HIDDEN, HIDDEN, HIDDEN, 1.0),
                                      (HIDDEN, HIDDEN, HIDDEN, 1.0), (HIDDEN, OUT_PAD, OUT, 0.5)):
        w = rng.uniform(-1, 1, (rows, fan_in)) * scale * math.sqrt(3.0 / fan_in)
        w[used:] = 0
        b = np.zeros(rows)
        if rows == OUT_PAD:
            for lobe in range(LOBES):
                mu = np.array([0.0, 1.0, 0.0]) if lobe == 0 else rng.normal(size=3)
                b[5 * lobe:5 * lobe + 3] = mu / np.linalg.norm(mu)
                b[5 * lobe + 3] = 0.3 * lobe
        parts += [w.reshape(-1), b]
    return np.concatenate(parts).astype(np.float32)


def _guide(sc, flags=0):
    sc.dev.guide_init(seed=1, flags=flags)
    sc.dev.guide_set_params(_guide_params())


def _queries(sc, n, g):
    lo, hi = _box_of(sc)
    q = torch.empty(n, 9, device="cuda")
    q[:, 0:3] = lo + torch.rand(n, 3, generator=g, device="cuda") * (hi - lo)
    q[:, 3:6] = _unit(g, n)
    wo = _unit(g, n)
    q[:, 6:9] = wo * torch.where((wo * q[:, 3:6]).sum(1, keepdim=True) < 0, -1.0, 1.0)
    return q


def _records(sc, n, g):
    """Training records: where the paths were, where they went and the radiance that came back."""
    r = torch.zeros(n, L.SPT_GUIDE_RECORD_FLOATS, device="cuda")
    r[:, 0:9] = _queries(sc, n, g)
    wi = _unit(g, n)
    r[:, 9:12] = wi * torch.where((wi * r[:, 3:6]).sum(1, keepdim=True) < 0, -1.0, 1.0)
    w = torch.rand(n, generator=g, device="cuda")
    r[:, 12] = torch.where(w < 0.4, torch.zeros_like(w), 4.0 * w * w)  # many paths return nothing
    return r


# ----------------------------------------------------------------------------
# the cases
# ----------------------------------------------------------------------------

def _primary_rays(sc, case, seed):
    cam = _camera(case, sc, seed)
    rays = torch.empty(case["width"] * case["height"], 8, device="cuda")
    sc.dev._check(sc.dev.lib.spt_camera_rays(sc.dev.h, C.byref(cam), rays.data_ptr()))
    sc.dev.sync()
    return rays


def prepare(case, seed):
    kind = case["kind"]
    sc = _scene(case)
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    st = {"kind": kind, "scene": sc, "dev": sc.dev}
    if kind == "trace":
        rays = _surface_rays(sc, case["n"], g) if case["rays"] == "incoherent" else _primary_rays(sc, case, seed)
        hits = torch.zeros(rays.shape[0], 2, dtype=torch.int32, device="cuda")
        st.update(rays=rays, hits=hits, out={"t": hits.view(torch.float32)[:, 0], "prim": hits[:, 1]})
    elif kind == "raycast":
        value = {"normal": L.SPT_RAYCAST_NORMAL, "depth": L.SPT_RAYCAST_DEPTH, "count": L.SPT_RAYCAST_COUNT}
        shape = (case["height"], case["width"]) + ((3,) if case["value"] == "normal" else ())
        st.update(camera=_camera(case, sc, seed), value=value[case["value"]],
                  out=torch.zeros(shape, device="cuda", dtype=torch.int32 if case["value"] == "count" else torch.float32))
    elif kind in ("render", "guided"):
        if kind == "guided":
            _guide(sc, case["flags"])
            case = dict(case, sampler="jittered", rr=3, depth=16, film64=False, per_path=False)
        integ = api.Integrator(spp=case["spp"], pixel_sampler=case["sampler"],
                               termination="russian-roulette" if case["rr"] >= 0 else "max-length",
                               path_length=case["rr"] if case["rr"] >= 0 else case["depth"], max_depth=case["depth"],
                               seed=seed)
        p = integ.params()
        film = torch.zeros(case["height"], case["width"], 3, device="cuda",
                           dtype=torch.float64 if case["film64"] else torch.float32)
        p.flags = L.SPT_RENDER_FILM64 if case["film64"] else L.SPT_RENDER_FILM32
        p.flags |= L.SPT_RENDER_GUIDED if kind == "guided" else 0
        paths = None
        if case["per_path"]:
            p.flags |= L.SPT_RENDER_PER_PATH
            paths = torch.zeros(case["height"] * case["width"] * integ.effective_spp(), 3, device="cuda")
        st.update(kind="render", camera=_camera(case, sc, seed), params=p, film=film, stream=sc.stream,
                  film32=None if case["film64"] else film.data_ptr(),
                  film64=film.data_ptr() if case["film64"] else None,
                  path=paths.data_ptr() if paths is not None else None,
                  out=[film] + ([paths] if paths is not None else []))
    elif kind == "eval":
        _guide(sc)
        st.update(queries=_queries(sc, case["n"], g), out=torch.zeros(case["n"], OUT, device="cuda"))
    elif kind == "gradient":
        _guide(sc)
        st.update(records=_records(sc, case["n"], g), grad=np.zeros(L.SPT_GUIDE_PARAMS, np.float32),
                  loss=C.c_float())
    else:
        scs = scenes.batch_scenes(n=case["n"], seed=seed, min_tris=case["min_tris"], max_tris=case["max_tris"],
                                  min_side=case["side"], max_side=case["side"], spp_choices=(case["spp"],))
        st["batch"] = api.Batch(sc.dev, scs)
    torch.cuda.synchronize()
    return st


def run(st):
    kind, dev = st["kind"], st["dev"]
    if kind == "trace":
        dev.trace(st["rays"].data_ptr(), st["rays"].shape[0], st["hits"].data_ptr())
        return st["out"]
    if kind == "raycast":
        dev._check(dev.lib.spt_raycast(dev.h, C.byref(st["camera"]), st["value"], st["out"].data_ptr()))
        return st["out"]
    if kind == "render":  # the film accumulates sums: a new image starts from zero
        with torch.cuda.stream(st["stream"]):
            st["film"].zero_()
        dev.render(st["camera"], st["params"], st["film32"], st["film64"], st["path"])
        return st["out"]
    if kind == "eval":
        dev._check(dev.lib.spt_guide_eval(dev.h, st["queries"].data_ptr(), st["queries"].shape[0],
                                          st["out"].data_ptr()))
        return st["out"]
    if kind == "gradient":
        dev._check(dev.lib.spt_guide_gradient(dev.h, st["records"].data_ptr(), st["records"].shape[0],
                                              st["grad"].ctypes.data, C.byref(st["loss"])))
        return {"grad": st["grad"], "loss": st["loss"].value}
    b = st["batch"]
    b.clear()
    b.render()
    return [b.image(i) for i in range(len(b.films))]


def _triangles(case):
    return {"box": lambda d: 12 + 20 * 4 ** d, "mesh": lambda d: 12 + 4 * d * d, "slit": lambda d: 16 + 4 * d * d,
            "spheres": lambda d: 2}[case["scene"]](case["detail"])


def work(case):
    """Per ray: 32 B in and 8 B out (the 16-B origin and direction of a camera
    ray stay on the chip), one descent of a four-wide tree (4 boxes of 12
    operations a level) and one triangle test (50); per path vertex about 250
    operations of shading; the scene read once (48 B of geometry and 48 B of
    normals a triangle). Guide: 25,600 operations a query, three times that a
    record."""
    kind = case["kind"]
    if kind == "eval":
        return {"bytes": case["n"] * (36 + 160), "flops": case["n"] * 25600}
    if kind == "gradient":
        return {"bytes": case["n"] * 52 + 4 * L.SPT_GUIDE_PARAMS, "flops": case["n"] * 76800}
    if kind == "batch":
        tris = case["n"] * math.sqrt(case["min_tris"] * case["max_tris"])
        paths = case["n"] * case["side"] ** 2 * math.ceil(math.sqrt(case["spp"])) ** 2
        per_ray = 48 * math.log(max(tris / case["n"], 4), 4) + 50
        return {"bytes": 96 * tris + 24 * case["n"] * case["side"] ** 2, "flops": paths * 3 * (per_ray + 250)}
    tris = _triangles(case)
    per_ray = 48 * math.ceil(math.log(max(tris, 4), 4)) + 50
    if kind == "trace":
        n = case["n"] if case["rays"] == "incoherent" else case["width"] * case["height"]
        return {"bytes": 40 * n + 48 * min(tris, n), "flops": n * per_ray}
    pixels = case["width"] * case["height"]
    if kind == "raycast":
        return {"bytes": pixels * (12 if case["value"] == "normal" else 4) + 96 * min(tris, pixels),
                "flops": pixels * per_ray}
    spp = case["spp"] if case.get("sampler") == "uniform" else math.ceil(math.sqrt(case["spp"])) ** 2
    rays = pixels * spp * min(4.0, 0.8 * case.get("depth", 16))
    guide = 25600 * 0.6 * rays if kind == "guided" else 0
    return {"bytes": pixels * (24 if case.get("film64") else 12) + 96 * min(tris, rays) +
            (12 * pixels * spp if case.get("per_path") else 0), "flops": rays * (per_ray + 250) + guide}


# ----------------------------------------------------------------------------
# the same values in 64 bits
# ----------------------------------------------------------------------------

def _closest(rays, tris):
    """Closest hit of every ray by testing all triangles: t and triangle, chunked."""
    o, d = rays[:, 0:3].double(), rays[:, 4:7].double()
    v0, e1, e2 = tris[:, 0], tris[:, 1] - tris[:, 0], tris[:, 2] - tris[:, 0]
    best = torch.full((o.shape[0],), math.inf, dtype=torch.float64, device="cuda")
    step = max(1, 20_000_000 // tris.shape[0])
    n1 = torch.linalg.cross(e1, e2)
    for i in range(0, o.shape[0], step):
        oo, dd = o[i:i + step], d[i:i + step]
        # t = n.(v0 - o) / n.d and the edge functions of the hit point, as products of matrices
        det = -(dd @ n1.T)
        m = torch.linalg.cross(oo, dd)
        u = dd @ torch.linalg.cross(v0, e2).T + m @ e2.T
        v = -(dd @ torch.linalg.cross(v0, e1).T + m @ e1.T)
        t = (oo @ n1.T) - (v0 * n1).sum(1)
        u, v, t = u / det, v / det, t / det
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t > 0) & (det.abs() >= 1e-6)
        best[i:i + step] = torch.where(ok, t, math.inf).amin(1)
        del det, m, u, v, t, ok
    return best


def _exact_mlp(theta, box, q):
    lo, hi = box
    x = ((q[:, 0:3] - lo) / (hi - lo).clamp(min=1e-6)).clamp(0, 1)
    f = [x]
    for k in range(3):
        a = 2 * math.pi * (1 << k) * x
        f.append(torch.stack([a.sin(), a.cos()], -1).reshape(-1, 6))
    c = 0.5 * ((q[:, 3:6] * q[:, 6:9]).sum(1, keepdim=True) + 1)
    bins = (torch.arange(4, device=q.device, dtype=q.dtype) + 0.5) * 0.25
    h = torch.cat(f + [q[:, 3:9], torch.exp(-8 * (c - bins) ** 2), torch.ones_like(c)], 1)
    at = 0
    for rows, cols in ((HIDDEN, ENC), (HIDDEN, HIDDEN), (HIDDEN, HIDDEN), (OUT_PAD, HIDDEN)):
        w, b = theta[at:at + rows * cols].view(rows, cols), theta[at + rows * cols:at + rows * cols + rows]
        at += rows * cols + rows
        h = h @ w.T + b
        if rows == HIDDEN:
            h = h.relu()
    return h[:, :OUT]


def _exact_loss(theta, box, r, total):
    """-sum W log q(wi) / total over the mixture's log density."""
    y = _exact_mlp(theta, box, r[:, 0:9]).view(-1, LOBES, 5)
    mu = y[..., 0:3] / (y[..., 0:3].square().sum(-1, keepdim=True) + 1e-12).sqrt()
    s = y[..., 3].clamp(math.log(1e-2), math.log(1e4))
    k = s.exp()
    lv = s - math.log(2 * math.pi) - torch.log(-torch.expm1(-2 * k)) + k * ((mu * r[:, None, 9:12]).sum(-1) - 1)
    logq = torch.logsumexp(torch.log_softmax(y[..., 4], -1) + lv, -1)
    return -(r[:, 12] * logq).sum() / total


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("trace", "raycast", "eval", "gradient") or case.get("value") == "count":
        return None
    if kind in ("trace", "raycast"):
        n = case["n"] if case.get("rays") == "incoherent" else case["width"] * case["height"]
        if case["scene"] == "spheres" or n * _triangles(case) > 2e10 or case.get("value") == "normal":
            return None
    st = prepare(case, seed)
    sc = st["scene"]
    if kind in ("trace", "raycast"):
        rays = st["rays"] if kind == "trace" else _primary_rays(sc, case, seed)
        t = _closest(rays, torch.from_numpy(sc.data.verts).cuda().double().view(-1, 3, 3))
        if kind == "trace":
            return {"t": t, "prim": None}
        return torch.where(t.isinf(), -1.0, t).view(case["height"], case["width"])
    theta = torch.from_numpy(_guide_params()).cuda().double()
    box = tuple(b.double() for b in _box_of(sc))
    if kind == "eval":
        return torch.cat([_exact_mlp(theta, box, q.double()) for q in st["queries"].split(1 << 18)])
    theta.requires_grad_(True)
    r = st["records"].double()
    total, loss = r[:, 12].sum(), 0.0
    for part in r.split(1 << 17):
        e = _exact_loss(theta, box, part, total)
        e.backward()
        loss += float(e)
    grad = theta.grad.clone()
    grad[-OUT_PAD + OUT:] = 0
    return {"grad": grad.cpu().numpy(), "loss": loss}
