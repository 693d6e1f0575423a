"""Cases that measure the framework as its users call it.

Every case goes through the public Python entry points: the raw traces
(``Accel.trace_closest`` / ``trace_any``), the progressive frame loop
(``PathTracer.launch_frame``), whole renders (``PathTracer.render`` +
``resolve``), batched serving (``Server.render``) and the learned guide
(guided renders, ``Guide.train``).  Sizes come from the benchmark and the
tests, or are odd ones from the same ranges.

A program loads a scene's geometry once and keeps its acceleration structure
and context, so those are kept per process; rays, material colours, frame
offsets, network weights and training samples come from the seed.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import wayland_amd as wl
from wayland_amd import scenes

INF = float("inf")

# Arithmetic a ray cannot do without, for work(): about six 8-wide node
# visits of 8 x 6 plane distances and their comparisons, and one triangle test.
RAY_FLOPS = 6 * 8 * 16 + 60
# One surface vertex: the BSDF's sample, pdf and value, and the same for the
# light sample.
VERTEX_FLOPS = 800


# ---- the cases ---------------------------------------------------------------
def listed():
    return [
        # picking and probe queries of an editor: a few hundred rays, launch latency
        dict(name="pick_cornell", kind="closest", scene="cornell", rays=333),
        # a light-baking or visibility batch on a mid-size model, ragged length
        dict(name="closest_mid", kind="closest", scene="ico", count=25, subdiv=4, rays=100_003),
        # the traversal workload: 2,048,000 triangles, 2^23 incoherent rays
        dict(name="closest_large", kind="closest", scene="ico", count=25, subdiv=6, rays=1 << 23),
        # occlusion over the same model, ragged length
        dict(name="any_large", kind="any", scene="ico", count=25, subdiv=6, rays=(1 << 23) - 77),
        # the interactive frame loop: two progressive frames at the default depth
        dict(name="frames_cornell_1024", kind="frames", scene="cornell", width=1024, height=1024,
             spp=2, depth=25, strategy=2, sort=False),
        # the plain path-tracing workload: Cornell box, 16 spp, depth 8
        dict(name="render_cornell_256", kind="render", scene="cornell", width=256, height=256,
             spp=16, depth=8, strategy=2, sort=False),
        # the wavefront workload: 1080p, 64 spp, depth 16 on 2,048,000 triangles
        dict(name="render_wavefront_1080", kind="render", scene="wave", count=25, subdiv=6,
             width=1920, height=1080, spp=64, depth=16, strategy=2, sort=False),
        # a preview of a textured scene at an odd size, light sampling only
        dict(name="render_textured_odd", kind="render", scene="textured", width=517, height=389,
             spp=3, depth=25, strategy=1, sort=False),
        # the serving mix: 64 requests, 128^2 .. 1024^2, 1 .. 64 spp
        dict(name="serve_mix_64", kind="serve", requests=64, res_lo=128, res_hi=1024, spp=64,
             lanes=2),
        # thumbnails: 256 small requests
        dict(name="serve_small_256", kind="serve", requests=256, res_lo=64, res_hi=256, spp=4,
             lanes=1),
        # one guided pass of the glossy caustic with a given network
        dict(name="guided_caustic_1024", kind="guided", width=1024, height=1024, spp=1, depth=16),
        # the training of one render pass: 8 Adam steps of 16,384 samples
        dict(name="guide_train_8", kind="train", samples=131_072, batch=16_384, steps=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["closest", "any", "frames", "render", "render", "render", "serve",
                       "guided", "train"])
    if kind in ("closest", "any"):
        c = dict(kind=kind, scene="ico", count=rng.choice([8, 25]), subdiv=rng.choice([4, 5, 6]),
                 rays=_log_int(rng, 200, 1 << 23))
        if rng.random() < 0.25:
            c = dict(kind=kind, scene="cornell", rays=_log_int(rng, 200, 1 << 22))
        return c
    if kind == "frames":
        return dict(kind=kind, scene=rng.choice(["cornell", "textured"]),
                    width=_log_int(rng, 100, 1400), height=_log_int(rng, 100, 1100),
                    spp=rng.randint(1, 3), depth=rng.randint(8, 25), strategy=2, sort=False)
    if kind == "render":
        scene = rng.choice(["cornell", "textured", "wave"])
        w, h = _log_int(rng, 97, 1920), _log_int(rng, 97, 1080)
        spp = max(1, min(64, _log_int(rng, 1, 64)))
        c = dict(kind=kind, scene=scene, width=w, height=h, spp=spp, depth=rng.randint(8, 25),
                 strategy=rng.choice([0, 1, 2, 2]), sort=rng.random() < 0.2)
        if scene == "wave":
            c.update(count=25, subdiv=rng.choice([4, 5, 6]), depth=rng.randint(8, 16))
        elif w * h * spp > 1 << 25:  # a closed box: every path runs long
            c["spp"] = max(1, (1 << 25) // (w * h))
        return c
    if kind == "serve":
        lo = rng.randint(64, 300)
        return dict(kind=kind, requests=_log_int(rng, 2, 96), res_lo=lo,
                    res_hi=rng.randint(lo, 700), spp=_log_int(rng, 1, 24), lanes=rng.choice([1, 2]))
    if kind == "guided":
        return dict(kind=kind, width=_log_int(rng, 128, 1024), height=_log_int(rng, 128, 1024),
                    spp=rng.randint(1, 4), depth=rng.randint(8, 16))
    batch = 32 * _log_int(rng, 8, 1024)
    return dict(kind="train", samples=_log_int(rng, batch, 8 * batch) + rng.randint(0, 31),
                batch=batch, steps=rng.randint(1, 8))


# ---- what a program keeps: context, geometry, acceleration structures --------
@functools.lru_cache(maxsize=1)
def _ctx():
    return wl.Context(0)


@functools.lru_cache(maxsize=6)
def _geometry(name, count, subdiv):
    """(scene, accel) of a model; its triangles do not depend on the seed."""
    if name == "cornell":
        sc = scenes.cornell_box()
    elif name == "textured":
        sc = scenes.textured_cornell_box()
    elif name == "caustic":
        sc = scenes.glossy_caustic()
    elif name == "wave":
        sc = scenes.wavefront_scene(count, subdiv)
    else:
        sc = scenes.icosphere_scene(count, subdiv)
    return sc, wl.Accel(_ctx(), sc)


def _model(case):
    return _geometry(case["scene"], case.get("count", 0), case.get("subdiv", 0))


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _rays(case, seed):
    """Incoherent rays, origins uniform in the model's box, directions uniform."""
    n, g = case["rays"], _generator(seed)
    u = torch.rand((n, 5), generator=g, device="cuda", dtype=torch.float32)
    lo, hi = ((-1.0, 0.0, -1.0), (1.0, 2.0, 1.0)) if case["scene"] == "cornell" else \
        ((0.0,) * 3, (1.0,) * 3)
    lo, hi = torch.tensor(lo, device="cuda"), torch.tensor(hi, device="cuda")
    rays = torch.empty((n, 8), device="cuda", dtype=torch.float32)
    rays[:, 0:3] = lo + (hi - lo) * u[:, 0:3]
    rays[:, 3] = 0.0
    z = 1.0 - 2.0 * u[:, 3]
    r = (1.0 - z * z).clamp(min=0.0).sqrt()
    phi = 2.0 * math.pi * u[:, 4]
    rays[:, 4] = r * phi.cos()
    rays[:, 5] = r * phi.sin()
    rays[:, 6] = z
    rays[:, 7] = INF
    return rays


def _scene(case, seed):
    """The model with the case's camera and the seed's base colours."""
    base, accel = _model(case)
    w, h = case["width"], case["height"]
    rng = np.random.default_rng(seed)
    meshes = []
    for m in base.meshes:
        mat = np.array(m.material, np.float32)
        if m.light_L is None:
            mat[0:3] = rng.uniform(0.1, 0.9, 3).astype(np.float32)
        meshes.append(scenes.Mesh(m.vertices, m.indices, m.normals, mat, m.light_L, m.two_sided,
                                  m.uv, m.texture))
    c = base.camera
    aspect = np.float32(w / h) * np.sqrt((c.up ** 2).sum() / (c.right ** 2).sum())
    cam = scenes.Camera(c.pos, c.lookat, c.up, (c.right * aspect).astype(np.float32))
    return scenes.Scene(meshes, cam, base.bg, base.name, base.textures), accel


def _guide_params(seed):
    """Network weights at the scale of a trained guide: He-uniform hidden
    layers, a smaller output layer, moderate concentrations."""
    rng = np.random.default_rng(seed)
    out = []
    for layer in range(5):
        n = 64 if layer < 4 else 32
        bound = math.sqrt(6.0 / 64.0) * (1.0 if layer < 4 else 0.3)
        out += [rng.uniform(-bound, bound, n * 64), rng.uniform(-0.1, 0.1, n)]
    b = out[-1]
    b[1::4] += 1.0                                    # raw concentration
    b[2::4] += rng.uniform(0.0, math.pi, 8)           # theta
    b[3::4] += rng.uniform(0.0, 2.0 * math.pi, 8)     # phi
    return np.concatenate(out).astype(np.float32)


def _guide_samples(case, seed):
    """Training samples as a render records them: positions in the unit box,
    unit normals and directions, positive skewed weights."""
    n, g = case["samples"], _generator(seed)

    def unit(k):
        v = torch.randn((k, 3), generator=g, device="cuda")
        return v / v.norm(dim=1, keepdim=True)

    s = torch.zeros((n, 16), device="cuda", dtype=torch.float32)
    s[:, 0:3] = torch.rand((n, 3), generator=g, device="cuda")
    s[:, 3:6] = unit(n)
    s[:, 6:9] = unit(n)
    s[:, 9:12] = torch.nn.functional.normalize(unit(n) + s[:, 3:6] * 1.2, dim=1)
    s[:, 12] = torch.rand((n,), generator=g, device="cuda").pow(4) * 20.0
    return s


def _config(case, seed):
    return wl.pt_config(case["width"], case["height"], spp=case["spp"],
                        frame_offset=(seed % 4096) << 12, max_depth=case["depth"],
                        rr_depth=4 if case["scene"] == "wave" else 5,
                        strategy=case["strategy"],
                        flags=wl.PT_SORT_BY_MATERIAL if case["sort"] else 0,
                        max_batch_paths=1 << 27)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("closest", "any"):
        return dict(kind=kind, accel=_model(case)[1], rays=_rays(case, seed))
    if kind in ("frames", "render"):
        sc, accel = _scene(case, seed)
        st = dict(kind=kind, pt=wl.PathTracer(_ctx(), accel, sc), cfg=_config(case, seed),
                  spp=case["spp"])
        if kind == "frames":
            n = case["width"] * case["height"]
            st["radiance"] = torch.zeros((n, 4), device="cuda", dtype=torch.float32)
            st["color"] = torch.zeros((n, 4), device="cuda", dtype=torch.uint8)
        return st
    if kind == "serve":
        # the same job sizes for every seed; the seed gives the samples drawn
        rng = np.random.default_rng(5)
        reqs = scenes.serving_requests(rng, case["requests"], case["res_lo"], case["res_hi"],
                                       case["spp"], 256 * (seed % 128))
        tracers = [wl.PathTracer(_ctx(), a, sc) for sc, a in _serving_models()]
        pixels = sum(r["width"] * r["height"] for r in reqs)
        films = torch.zeros((pixels, 6), device="cuda", dtype=torch.float32)
        at = 0
        for r in reqs:
            r["pt"] = tracers[r.pop("scene")]
            r["film"] = films[at:at + r["width"] * r["height"]]
            at += r["width"] * r["height"]
        server = wl.Server(_ctx(), batch_paths=1 << 26, lanes=case["lanes"])
        return dict(kind=kind, server=server, reqs=reqs, films=films)
    if kind == "guided":
        c = dict(case, scene="caustic", strategy=2, sort=False)
        base, accel = _model(c)
        sc = scenes.glossy_caustic(case["width"], case["height"], 0, 1)  # for its camera
        pt = wl.PathTracer(_ctx(), accel, scenes.Scene(base.meshes, sc.camera, base.bg))
        guide = wl.Guide(_ctx())
        guide.set_params(_guide_params(seed))
        pt.set_guide(guide, wl.GUIDE_SAMPLE)
        return dict(kind="render", pt=pt, cfg=_config(c, seed), spp=case["spp"], guide=guide)
    guide = wl.Guide(_ctx(), batch_size=case["batch"])
    guide.set_params(_guide_params(seed))
    return dict(kind=kind, guide=guide, samples=_guide_samples(case, seed), steps=case["steps"])


@functools.lru_cache(maxsize=1)
def _serving_models():
    return [(sc, wl.Accel(_ctx(), sc)) for sc in scenes.serving_scenes()]


# ---- one pass ------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "closest":
        hits = state["accel"].trace_closest(state["rays"])
        return {"t": hits[:, 0], "prim": hits.view(torch.int32)[:, 1], "b1": hits[:, 2],
                "b2": hits[:, 3]}
    if kind == "any":
        return {"bits": state["accel"].trace_any(state["rays"])}
    if kind == "frames":
        for frame in range(state["spp"]):
            state["pt"].launch_frame(state["cfg"], frame, state["radiance"], state["color"])
        return {"radiance": state["radiance"], "color": state["color"]}
    if kind == "render":
        film, _ = state["pt"].render(state["cfg"], stats=False)
        return {"film": film, "image": state["pt"].resolve(film, state["spp"])}
    if kind == "serve":
        state["films"].zero_()
        state["server"].render(state["reqs"])
        return {"films": state["films"]}
    state["guide"].train(state["samples"], state["steps"])
    return {"params": state["guide"].get_params()}


# ---- work ------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("closest", "any"):
        tris = 36 if case["scene"] == "cornell" else case["count"] * 20 * 4 ** case["subdiv"]
        out = 16 if kind == "closest" else 0.125
        return {"bytes": case["rays"] * (32 + out) + min(tris * 36, case["rays"] * 48),
                "flops": case["rays"] * RAY_FLOPS}
    if kind == "serve":
        res = 0.5 * (case["res_lo"] + case["res_hi"])
        pixels = case["requests"] * res * res
        paths = pixels * 0.5 * (1 + case["spp"])
        return {"bytes": 48 * pixels, "flops": paths * 4 * (2 * RAY_FLOPS + VERTEX_FLOPS)}
    if kind == "train":
        per = 2 * (3 * 4 * 64 * 64 + 3 * 64 * 32)  # forward, deltas, weight gradients
        n = min(case["steps"] * case["batch"], case["samples"])
        return {"bytes": 64 * n + 6 * 4 * 18720 * case["steps"],
                "flops": case["steps"] * case["batch"] * per}
    pixels = case["width"] * case["height"]
    paths = pixels * case["spp"]
    # vertices per path: a closed box keeps paths alive to roulette, the open
    # scenes lose them to the background
    vertices = 1 if case.get("scene") == "wave" or kind == "guided" else min(8, case["depth"])
    return {"bytes": (24 + 12) * pixels,
            "flops": paths * vertices * (2 * RAY_FLOPS + VERTEX_FLOPS)}


# ---- the same in 64 bits -----------------------------------------------------------
def exact(case, seed):
    if case["kind"] == "closest":
        return _exact_closest(case, seed)
    if case["kind"] == "train":
        return {"params": _exact_train(case, seed)}
    return None  # renders: a path's branches have no 64-bit counterpart; occlusion bits


def _exact_closest(case, seed):
    sc, _ = _model(case)
    if sc.num_triangles * case["rays"] > 2e10:
        return None
    tri = torch.from_numpy(sc.triangles()).cuda().double().view(-1, 3, 3)
    rays = _rays(case, seed).double()
    v0, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    n = rays.shape[0]
    t = torch.full((n,), INF, device="cuda", dtype=torch.float64)
    b1, b2 = torch.zeros_like(t), torch.zeros_like(t)
    # blocks of rays x triangles as matrix products: with n = e1 x e2,
    # det = -d.n and m = o x d, t = (o - v0).n / det,
    # u = (o - v0).(d x e2) / det and v = d.((o - v0) x e1) / det
    nrm = torch.linalg.cross(e1, e2)
    step = max(1, int(4e7 // tri.shape[0]))
    a1, a2 = torch.linalg.cross(v0, e1), torch.linalg.cross(v0, e2)
    for k in range(0, n, step):
        o, d = rays[k:k + step, 0:3], rays[k:k + step, 4:7]
        m = torch.linalg.cross(o, d)
        det = -(d @ nrm.T)
        u = ((m @ e2.T) + (d @ a2.T)) / det
        v = -((m @ e1.T) + (d @ a1.T)) / det
        s = ((o @ nrm.T) - (v0 * nrm).sum(1)) / det
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (s >= 0)
        s = torch.where(ok, s, torch.full_like(s, INF))
        best, at = s.min(1)
        hit = torch.isfinite(best)
        rows = torch.arange(best.shape[0], device="cuda")
        t[k:k + step] = best
        b1[k:k + step] = torch.where(hit, u[rows, at], torch.zeros_like(best))
        b2[k:k + step] = torch.where(hit, v[rows, at], torch.zeros_like(best))
    return {"t": t, "prim": None, "b1": b1, "b2": b2}


def _encode(q):
    """The network's 64 inputs: lane group g of each 16-feature block holds
    axis g's sine and cosine pairs, then the normal and the direction."""
    x = torch.zeros((q.shape[0], 64), device=q.device, dtype=torch.float64)
    for g in range(3):
        for p in range(7):
            e = 16 * (p // 2) + 4 * g + 2 * (p % 2)
            if p < 6:
                a = (2.0 ** p) * math.pi * q[:, g]
                x[:, e], x[:, e + 1] = a.sin(), a.cos()
            else:
                x[:, e], x[:, e + 1] = q[:, 3 + g], q[:, 6 + g]
    return x


def _exact_train(case, seed):
    """`steps` Adam steps on the mixture's weighted log likelihood, in 64 bits."""
    theta = torch.from_numpy(_guide_params(seed)).cuda().double().requires_grad_(True)
    s = _guide_samples(case, seed).double()
    m, v = torch.zeros_like(theta), torch.zeros_like(theta)
    n, batch = case["samples"], case["batch"]
    for k in range(case["steps"]):
        lo = (k * batch) % n
        part = s[lo:lo + min(batch, n - lo)]
        x, at = _encode(part), 0
        for layer in range(5):
            rows = 64 if layer < 4 else 32
            w = theta[at:at + rows * 64].view(rows, 64)
            b = theta[at + rows * 64:at + rows * 65]
            at += rows * 65
            x = x @ w.T + b
            if layer < 4:
                x = x.relu()
        o = x.view(-1, 8, 4)  # order of the lobes does not matter to the loss
        kappa = torch.nn.functional.softplus(o[..., 1])
        st, ct = o[..., 2].sin(), o[..., 2].cos()
        mu = torch.stack([st * o[..., 3].cos(), st * o[..., 3].sin(), ct], -1)
        cos = (mu * part[:, None, 9:12]).sum(-1)
        norm = kappa.log() - math.log(2 * math.pi) - (-torch.expm1(-2 * kappa)).log()
        logq = torch.logsumexp(o[..., 0].log_softmax(1) + norm + kappa * (cos - 1), 1)
        loss = -(part[:, 12] * logq).mean()
        (g,) = torch.autograd.grad(loss, theta)
        m = 0.9 * m + (1 - 0.9) * g
        v = 0.99 * v + (1 - 0.99) * g * g
        c1, c2 = 1 - 0.9 ** (k + 1), 1 - 0.99 ** (k + 1)
        theta = (theta - 5e-3 * (m / c1) / ((v / c2).sqrt() + 1e-8)).detach().requires_grad_(True)
    return theta.detach().cpu().numpy()
