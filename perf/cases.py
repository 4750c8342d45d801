"""Timed cases of the path tracer, through its public entry points (srt_amd.abi).

A case is a dict of plain values; `prepare` sets up what a program holds
before the call (a context with the scene resident, its tree, device
buffers), `run` makes one pass and returns what the program gets back.

  kind      one pass
  frame     Context.render into device memory (path tracer; with `mlp` the
            radiance MLP answers after vertex 2)
  skinned   Context.skin_refit to a pose, then the frame
  train     Context.mlp_train_frame, then the updated weights
  rays      Context.trace_noalloc on device arrays: closest hits, then any hits
  rebuild   Context.build_bvh, then closest hits of a few rays
  post      srt_accumulate, denoise and srt_tonemap of a film in device memory
  serve     a batch of requests submitted to a running server, until all are done
"""
import ctypes as C
import functools
import math

import numpy as np
import torch

from srt_amd import abi, scenes

SPHERES = 3125            # the 1,000,008-triangle field
TONEMAP_ACES = abi.TONEMAP["ACES"]


def _frame(name, scene, width, height, spp, depth, spheres=0, mlp=False):
    c = dict(kind="frame", scene=scene, width=width, height=height, spp=spp, depth=depth, spheres=spheres, mlp=mlp)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a thumbnail or material preview: a few launches, latency is everything
        _frame("thumbnail", "cornell", 64, 64, 4, 5),
        # the small closed scene at its configured size: every path bounces to the depth limit
        _frame("cornell", "cornell", 256, 256, 16, 5),
        # interactive display: one sample per pixel at the pass's default depth
        _frame("interactive", "spheres", 1280, 720, 1, 16, spheres=SPHERES),
        # the headline frame: 1M triangles, 132.7 M paths
        _frame("headline", "spheres", 1920, 1080, 64, 8, spheres=SPHERES),
        # repeated meshes: the two-level tree
        _frame("instanced", "spheres_instanced", 1280, 720, 8, 8, spheres=SPHERES),
        # character animation: a new pose of the 200k-triangle tube per frame
        dict(name="skinned", kind="skinned", scene="tube", width=1280, height=720, spp=16, depth=6),
        # paths cut at vertex 2 by the trained radiance MLP
        _frame("mlp_frame", "cornell", 256, 256, 64, 5, mlp=True),
        # one online training frame: samples traced, then 8 Adam steps
        dict(name="mlp_train", kind="train", scene="cornell", width=256, height=256, spp=8, depth=5, steps=8),
        # ray queries of a simulation on device arrays, an odd count
        dict(name="rays", kind="rays", scene="spheres", spheres=SPHERES, rays=1000003),
        # geometry that changed too much for a refit: a new tree, then picking rays
        dict(name="rebuild", kind="rebuild", scene="spheres", spheres=SPHERES, rays=16384),
        # the film's way to the screen: accumulate, denoise, tone-map
        dict(name="post", kind="post", width=1920, height=1080),
        # requests of mixed sizes on two resident scenes
        dict(name="serve", kind="serve", requests=8, largest=1280, spp=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cornell", "spheres", "spheres", "instanced", "skinned", "mlp", "train", "rays", "rebuild", "post",
                       "serve"])
    # widths down to a thumbnail's, any remainder against the 8x8 pixel tiles; heights of common aspect ratios
    w = _log_int(rng, 48, 1920)
    h = max(27, int(w * rng.uniform(0.5, 1.0)))
    if kind == "cornell":
        return _frame(None, "cornell", w, h, _log_int(rng, 1, 32), rng.choice([5, 8, 16]))
    if kind == "spheres":
        return _frame(None, "spheres", w, h, _log_int(rng, 1, 32), rng.choice([5, 8, 16]),
                      spheres=_log_int(rng, 30, SPHERES))
    if kind == "instanced":
        return _frame(None, "spheres_instanced", w, h, _log_int(rng, 1, 16), rng.choice([5, 8]),
                      spheres=_log_int(rng, 30, SPHERES))
    if kind == "skinned":
        return dict(kind="skinned", scene="tube", width=w, height=h, spp=_log_int(rng, 1, 16), depth=rng.choice([4, 6]))
    if kind == "mlp":
        return _frame(None, "cornell", min(w, 700), min(h, 500), _log_int(rng, 4, 64), 5, mlp=True)
    if kind == "train":
        return dict(kind="train", scene="cornell", width=rng.randint(128, 320), height=rng.randint(128, 320),
                    spp=rng.randint(4, 12), depth=rng.choice([5, 8]), steps=rng.choice([4, 8, 16]))
    if kind == "rays":
        return dict(kind="rays", scene="spheres", spheres=_log_int(rng, 30, SPHERES), rays=_log_int(rng, 1000, 2000000))
    if kind == "rebuild":
        return dict(kind="rebuild", scene="spheres", spheres=_log_int(rng, 30, SPHERES), rays=_log_int(rng, 256, 16384))
    if kind == "post":
        return dict(kind="post", width=w, height=h)
    return dict(kind="serve", requests=rng.randint(2, 12), largest=rng.choice([256, 512, 1280]), spp=rng.choice([4, 16]))


# ---------------------------------------------------------------------------
# what a program holds before the call
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=3)
def _scene(name, spheres, seed):
    if name == "spheres":
        return scenes.spheres(num_spheres=spheres, seed=seed)
    if name == "spheres_instanced":
        return scenes.spheres_instanced(num_spheres=spheres, seed=seed)
    if name == "tube":
        return scenes.tube(seed=seed)
    return scenes.cornell()


def _view(scene, seed):
    """The scene's camera, moved a little by the seed (1 % of its distance)."""
    rng = np.random.default_rng(seed + 1)
    cam = dict(scene.camera)
    pos, target = np.asarray(cam["position"], float), np.asarray(cam["target"], float)
    step = 0.01 * np.linalg.norm(target - pos)
    cam["position"] = tuple(float(x) for x in pos + rng.uniform(-step, step, 3))
    return cam


def _resident(case, seed):
    """A context with the case's scene uploaded and its tree built."""
    s = _scene(case["scene"], case.get("spheres", 0), seed)
    ctx = abi.Context(0)
    h = ctx.upload(s)
    ctx.build_bvh(h)
    return s, ctx, h


def _film(w, h):
    return torch.empty((h * w, 4), dtype=torch.float32, device="cuda")


def _rays_in(s, n, seed):
    """Origins inside the scene box, uniform directions, finite lengths (host arrays)."""
    rng = np.random.default_rng(seed + 2)
    lo, hi = s.positions.min(0), s.positions.max(0)
    o = rng.uniform(lo, hi, size=(n, 3)).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    tmax = rng.uniform(0.25, 1.0, size=n).astype(np.float32) * np.float32(np.linalg.norm(hi - lo))
    return o, d, tmax


def _ray_buffers(s, n, seed):
    o, d, tmax = (torch.from_numpy(a).cuda() for a in _rays_in(s, n, seed))
    return dict(o=o, d=d, tmax=tmax, t=torch.empty_like(tmax), u=torch.empty_like(tmax), v=torch.empty_like(tmax),
                prim=torch.empty(n, dtype=torch.int32, device="cuda"),
                any=torch.empty(n, dtype=torch.int32, device="cuda"))


def _noisy_film(case, seed):
    """A film as low-sample path tracing leaves it: a smooth image times heavy-tailed noise, some pixels black."""
    w, h = case["width"], case["height"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    y = torch.linspace(0, 1, h, device="cuda")[:, None, None]
    x = torch.linspace(0, 1, w, device="cuda")[None, :, None]
    phase = torch.rand(3, device="cuda", generator=g) * 6.0
    smooth = 0.6 + 0.5 * torch.sin(9.0 * x + phase) * torch.cos(7.0 * y + 2.0 * phase)
    noise = -torch.log(torch.rand((h, w, 1), device="cuda", generator=g) + 1e-6)
    film = torch.ones((h, w, 4), dtype=torch.float32, device="cuda")
    film[..., :3] = smooth * noise
    film[..., :3] *= (torch.rand((h, w, 1), device="cuda", generator=g) > 0.05).float()
    return film.reshape(h * w, 4).contiguous()


def _requests(case, seed):
    rng = np.random.default_rng(seed + 3)
    sizes = [r for r in ((256, 256), (512, 512), (1280, 720)) if r[0] <= case["largest"]]
    out = []
    for i in range(case["requests"]):
        w, h = sizes[-1 - i % len(sizes)]
        out.append(dict(scene=i % 2, width=w, height=h, spp=case["spp"], seed=int(rng.integers(1 << 30))))
    return out


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case, seed=seed)
    if kind == "post":
        st["ctx"] = abi.Context(0)
        st["film"] = _noisy_film(case, seed)
        st["acc"] = torch.zeros_like(st["film"])
    elif kind == "serve":
        ctx = abi.Context(0)
        loaded = []
        for s in (_scene("cornell", 0, 0), _scene("tube", 0, 11)):
            h = ctx.upload(s)
            ctx.build_bvh(h)
            loaded.append((h, _view(s, seed), s.render["max_depth"]))
        st.update(ctx=ctx, scenes=loaded, requests=_requests(case, seed))
        ctx.serve_start()
    else:
        s, ctx, h = _resident(case, seed)
        st.update(ctx=ctx, h=h, cam=_view(s, seed))
        if kind in ("rays", "rebuild"):
            st["rays"] = _ray_buffers(s, case["rays"], seed)
        else:
            st["film"] = _film(case["width"], case["height"])
        if kind == "skinned":
            ctx.set_skin(h, s.skin["bone_ids"], s.skin["bone_weights"])
            st["pose"] = s.skin["matrices"](seed % 60)
        if kind == "train" or case.get("mlp"):
            ctx.mlp_create(seed=seed % 1000 + 1, lr=1e-3)
        if case.get("mlp"):
            for f in range(4):
                ctx.mlp_train_frame(h, st["cam"], 256, 256, 8, 5, 4, seed=5000 + f, max_samples=1 << 18, steps=8)
    torch.cuda.synchronize()
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _closest(st):
    ctx, r = st["ctx"], st["rays"]
    ctx.trace_noalloc(st["h"], r["tmax"].numel(), r["o"].data_ptr(), r["d"].data_ptr(), r["tmax"].data_ptr(),
                      r["t"].data_ptr(), r["u"].data_ptr(), r["v"].data_ptr(), r["prim"].data_ptr())
    return dict(t=r["t"], u=r["u"], v=r["v"], prim=r["prim"])


def run(st):
    case, ctx = st["case"], st["ctx"]
    kind = case["kind"]
    if kind in ("frame", "skinned"):
        if kind == "skinned":
            ctx.skin_refit(st["h"], st["pose"])
        ctx.render(st["h"], st["cam"], case["width"], case["height"], case["spp"], case["depth"], 4, 1, 1,
                   st["seed"] % 65536, device_ptr=st["film"].data_ptr(), mlp_mode=1 if case.get("mlp") else 0)
        return st["film"]
    if kind == "train":
        loss, n = ctx.mlp_train_frame(st["h"], st["cam"], case["width"], case["height"], case["spp"], case["depth"], 4,
                                      seed=st["seed"] % 65536, max_samples=1 << 18, steps=case["steps"])
        return dict(loss=loss, samples=n, weights=ctx.mlp_params())
    if kind == "rays":
        out = _closest(st)
        r = st["rays"]
        ctx.trace_noalloc(st["h"], r["tmax"].numel(), r["o"].data_ptr(), r["d"].data_ptr(), r["tmax"].data_ptr(),
                          0, 0, 0, r["any"].data_ptr(), any_hit=True)
        return dict(out, any=r["any"])
    if kind == "rebuild":
        ctx.build_bvh(st["h"])
        return _closest(st)
    if kind == "post":
        film, acc = st["film"], st["acc"]
        n = film.shape[0]
        ctx.check(ctx.lib.srt_accumulate(ctx.h, C.c_void_p(acc.data_ptr()), C.c_void_p(film.data_ptr()), n, 0, 1))
        ctx.denoise_device(acc.data_ptr(), case["width"], case["height"])
        ctx.check(ctx.lib.srt_tonemap(ctx.h, C.c_void_p(acc.data_ptr()), n, TONEMAP_ACES, C.c_float(0.0), 1, 1))
        return acc
    tickets = []
    for q in st["requests"]:
        h, cam, depth = st["scenes"][q["scene"]]
        tickets.append(ctx.submit(h, cam, q["width"], q["height"], q["spp"], depth, 4, 1, 1, q["seed"]))
    for t, _ in tickets:
        ctx.wait(t)
    ctx.forget_tickets()
    return [img for _, img in tickets]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _triangles(case):
    return {"cornell": 36, "tube": 200004}.get(case.get("scene"), 320 * case.get("spheres", 0) + 8)


def _path_flops(triangles, depth, closed, paths, cut=None):
    """Segments of `paths` camera paths: in the closed box nearly every path
    reaches the depth limit or roulette (about 4 segments), in the open scenes
    most leave after the first (1.6).  A segment and its light sample cost two
    descents of a balanced tree (2 box tests of 12 operations per level), two
    triangle tests of 45 each and about 300 operations of shading."""
    segments = (min(depth, cut or 4) if closed else min(depth, 1.6)) * paths
    return segments * (2 * (24.0 * max(1.0, math.log2(triangles)) + 90.0) + 300.0)


def work(case):
    kind = case["kind"]
    tri = _triangles(case)
    scene_bytes = 36.0 * tri                    # each triangle's corners once
    if kind == "post":
        n = case["width"] * case["height"]
        # film in, screen out; per pixel 5 passes of 25 taps (difference, weight, three sums)
        return {"bytes": 32.0 * n, "flops": n * 5 * 25 * 25.0}
    if kind in ("rays", "rebuild"):
        n = case["rays"]
        rays = n * (24.0 * math.log2(tri) + 90.0)
        if kind == "rays":
            return {"bytes": scene_bytes + n * (28.0 + 16.0 + 4.0), "flops": 2 * rays}
        # every triangle read and written in tree order with its box, and the tree's nodes written
        return {"bytes": 2 * scene_bytes + 64.0 * tri + 44.0 * n, "flops": 20.0 * tri * math.log2(tri) + rays}
    if kind == "serve":
        qs = _requests(case, 0)
        px = sum(q["width"] * q["height"] for q in qs)
        f = sum(_path_flops((36, 200004)[q["scene"]], 5, q["scene"] == 0, q["width"] * q["height"] * q["spp"]) for q in qs)
        return {"bytes": 36.0 * 200040 + 16.0 * px, "flops": f}
    px = case["width"] * case["height"]
    closed = case["scene"] == "cornell"
    cut = 2 if case.get("mlp") else None
    f = _path_flops(tri, case["depth"], closed, px * case["spp"], cut)
    b = scene_bytes + 16.0 * px
    if case["scene"] == "spheres_instanced":
        b = 36.0 * 16 * 320 + 96.0 * case["spheres"] + 16.0 * px
    if case.get("mlp"):
        f += 33024.0 * px * case["spp"]
    if kind == "train":
        n = min(1 << 18, px * case["spp"])
        f += 99072.0 * n
        b = scene_bytes + 48.0 * n + 4.0 * 16771 * 2
    if kind == "skinned":
        b += 100108 * (3 * 24.0 + 32.0) + 48.0 * 64
        f += 100108 * 4 * 60.0
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------
def _exact_post(case, seed):
    w, h = case["width"], case["height"]
    img = _noisy_film(case, seed).double().reshape(h, w, 4)[..., :3]
    taps = [1 / 16, 1 / 4, 3 / 8, 1 / 4, 1 / 16]
    for it in range(5):
        step, inv = 1 << it, 1.0 / (0.2 * 2.0 ** -it) ** 2
        g = torch.log(1.0 + img)
        total = torch.zeros_like(img)
        weight = torch.zeros((h, w, 1), dtype=torch.float64, device=img.device)
        for j in range(-2, 3):
            for i in range(-2, 3):
                dy, dx = j * step, i * step
                y0, y1, x0, x1 = max(0, -dy), min(h, h - dy), max(0, -dx), min(w, w - dx)
                if y0 >= y1 or x0 >= x1:
                    continue
                here = (slice(y0, y1), slice(x0, x1))
                there = (slice(y0 + dy, y1 + dy), slice(x0 + dx, x1 + dx))
                k = taps[j + 2] * taps[i + 2] * torch.exp(-((g[here] - g[there]) ** 2).sum(-1, keepdim=True) * inv)
                total[here] += img[there] * k
                weight[here] += k
        img = total / weight
    c = img * 0.6
    c = ((c * (2.51 * c + 0.03)) / (c * (2.43 * c + 0.59) + 0.14)).clamp(0.0, 1.0) ** (1.0 / 2.2)
    return torch.cat([c, torch.ones_like(c[..., :1])], -1).reshape(h * w, 4)


def _exact_closest(case, seed):
    """Hit distances by testing every triangle (Moeller and Trumbore); 0 for a miss."""
    s = _scene(case["scene"], case["spheres"], seed)
    o, d, tmax = (torch.from_numpy(a).cuda().double() for a in _rays_in(s, case["rays"], seed))
    tri = torch.from_numpy(s.positions[s.indices.astype(np.int64)]).cuda().double()
    v0, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    n = torch.linalg.cross(e1, e2)
    best = torch.full((o.shape[0],), math.inf, dtype=torch.float64, device="cuda")
    chunk = max(1, (1 << 26) // max(1, o.shape[0]))
    # the triple products as matrix products of per-ray and per-triangle vectors:
    # (o - v0) . (d x e) = e . (o x d) + d . (v0 x e)
    ray = torch.cat([d, torch.linalg.cross(o, d)], 1)
    for k in range(0, v0.shape[0], chunk):
        a, x, y, nn = v0[k:k + chunk], e1[k:k + chunk], e2[k:k + chunk], n[k:k + chunk]
        det = -(d @ nn.T)
        inv = 1.0 / det
        t = (o @ nn.T - (a * nn).sum(1)) * inv
        u = (ray @ torch.cat([torch.linalg.cross(a, y), y], 1).T) * inv
        v = -(ray @ torch.cat([torch.linalg.cross(a, x), x], 1).T) * inv
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= 1e-3) & (t <= tmax[:, None])
        best = torch.minimum(best, torch.where(ok, t, math.inf).amin(1))
    return torch.where(torch.isinf(best), 0.0, best)


def exact(case, seed):
    if case["kind"] == "post":
        return _exact_post(case, seed)
    if case["kind"] in ("rays", "rebuild") and case["rays"] * _triangles(case) <= 2e10:
        # the distance alone: on a shared edge the triangle, and with it u and v, is either one's
        out = dict(t=_exact_closest(case, seed), u=None, v=None, prim=None)
        return dict(out, any=None) if case["kind"] == "rays" else out
    return None
