"""The traversal kernels at the edges of their dispatch: the deep-BVH kernels
(32-entry stack, 64-bit addresses), the change of the raw traces' chunk size
and ray counts around a chunk and an XCD's share."""
import numpy as np
import pytest

import oracle_bind as ob
from wayland_amd import scenes

pytestmark = pytest.mark.gpu


def _deep_scene():
    """Triangles shrinking by 0.55 each towards the origin: a BVH8 deeper than
    the 16-entry stack's kernels take."""
    rng = np.random.default_rng(1)
    n = 160
    s = (0.55 ** np.arange(n))[:, None, None]
    t = ((rng.uniform(-1, 1, (n, 3, 3)) * 0.4 + np.array([1.0, 0.3, -0.2])) * s)
    mesh = scenes.soup_mesh(t.astype(np.float32), scenes.matte_material((0.7, 0.6, 0.5)))
    light = scenes.soup_mesh(np.float32([[[-2, 2.5, -2], [2, 2.5, -2], [2, 2.5, 2]],
                                         [[-2, 2.5, -2], [2, 2.5, 2], [-2, 2.5, 2]]]),
                             scenes.matte_material((0, 0, 0)))
    light.light_L, light.two_sided = (4.0, 4.0, 4.0), True
    cam = scenes.pinhole_camera([0.3, 0.2, 3.0], [0, 0, -1], [0, 1, 0], 40.0, 64, 48)
    return scenes.Scene([mesh, light], cam, (0.2, 0.2, 0.2), "deep")


def _hits(accel, rays_np):
    import torch
    import wayland_amd as wl
    rays = torch.from_numpy(np.ascontiguousarray(rays_np)).cuda()
    hits, bits = accel.trace_closest(rays), accel.trace_any(rays)
    torch.cuda.synchronize()
    return wl.hits_to_numpy(hits), wl.unpack_bits(bits, rays_np.shape[0])


def _same(h, ref):
    hit = ref["prim"] != 0xFFFFFFFF
    assert np.array_equal(h["prim"], ref["prim"])
    assert np.array_equal(h["t"].view(np.uint32), ref["t"].view(np.uint32))
    for b in ("b1", "b2"):
        assert np.array_equal(h[b][hit].view(np.uint32), ref[b][hit].view(np.uint32))


def test_deep_bvh_traces_and_render(gpu_ctx):
    import wayland_amd as wl
    sc = _deep_scene()
    accel = wl.Accel(gpu_ctx, sc)
    assert accel.info()["depth"] > 16
    print(f"case: deep BVH {accel.info()}", flush=True)
    rng = np.random.default_rng(3)
    rays = scenes.traversal_rays(20000, seed=3)
    # half the rays aim at the origin, where the small triangles are
    rays[:, 0:3] = rays[:, 0:3] * 3 - 1
    aim = rng.uniform(-1, 1, (10000, 3)) * (0.55 ** rng.uniform(0, 60, 10000))[:, None]
    rays[:10000, 4:7] = aim - rays[:10000, 0:3]
    tris = sc.triangles()
    h, occ = _hits(accel, rays)
    _same(h, ob.closest_brute(tris, rays))
    assert np.array_equal(occ, ob.any_brute(tris, rays))
    pt, opt = wl.PathTracer(gpu_ctx, accel, sc), ob.OraclePT(sc)
    g = pt.render_samples(wl.pt_config(64, 48, max_depth=8), 1).cpu().numpy()
    o, _ = opt.render_frame(opt.config(64, 48, max_depth=8), 1)
    err = np.abs(g - o) / np.maximum(np.abs(o), 1e-6)
    assert (err.reshape(-1, 3).max(1) <= 1e-5).mean() >= 0.995


@pytest.mark.parametrize("n", [1, 63, 64, 65, 511, 512, 513, 8 * 64 * 3 + 1,
                               786_431, 786_432, 786_433, 1_000_003])
def test_ray_counts_around_the_chunk_sizes(gpu_ctx, n):
    """Chunks of 64 rays below 128 per resident wave (786,432 rays on 256 CUs
    with 24 waves each), 128 from there on: every ray's result equals that of
    the same ray in a trace of another length, and the oracle's."""
    import wayland_amd as wl
    print(f"case: {n} rays", flush=True)
    sc = scenes.icosphere_scene(6, 3, seed=2)
    accel = wl.Accel(gpu_ctx, sc)
    rays = scenes.traversal_rays(n + 4096, seed=9)
    h, occ = _hits(accel, rays[:n])
    whole, occ_whole = _hits(accel, rays)
    _same(h, whole[:n])
    assert np.array_equal(occ, occ_whole[:n])
    _same(h[::41], ob.OracleBVH(sc.triangles()).closest(rays[:n:41]))


@pytest.mark.parametrize("width", [1, 63, 255, 256, 257, 2047, 2048, 2049, 4100])
@pytest.mark.parametrize("sort", [0, 1])
def test_batch_sizes_around_the_queue_segments(gpu_ctx, width, sort):
    """A batch of `width` paths against the same paths in batches of at most
    64: the films are bit-identical, whatever queue segment a path is in."""
    import torch
    import wayland_amd as wl
    print(f"case: {width} x 1, sort {sort}", flush=True)
    sc = scenes.wavefront_scene(4, 2, width=width, height=1)
    pt = wl.PathTracer(gpu_ctx, wl.Accel(gpu_ctx, sc), sc)
    kw = dict(spp=1, max_depth=6, rr_depth=2, flags=wl.PT_SORT_BY_MATERIAL if sort else 0)
    a, _ = pt.render(wl.pt_config(width, 1, **kw), stats=False)
    b, _ = pt.render(wl.pt_config(width, 1, max_batch_paths=64, **kw), stats=False)
    assert torch.equal(a, b)
    assert (a[:, 0:3] != 0).any()


@pytest.mark.parametrize("strategy", [0, 1, 2])
def test_plain_materials_keep_every_bit(gpu_ctx, strategy):
    """Materials without transmission, clearcoat, sheen, tint or subsurface are
    shaded without those terms.  The same materials with a clearcoat gloss
    outside [0, 1] (which a clearcoat of 0 multiplies away) take the general
    expressions: the films are bit-identical, at the ends of the accepted
    ranges too, and beside glass."""
    import torch
    import wayland_amd as wl
    films = []
    for gloss in (1.0, 1.5):
        sc = scenes.wavefront_scene(12, 3, width=160, height=120)
        rng = np.random.default_rng(4)
        k = 0
        for m in sc.meshes:
            if m.light_L is not None:
                continue
            m.material = scenes.disney_material(
                color=rng.uniform(0, 1, 3) * (k % 5 > 0), metallic=(0.0, 1.0, 0.3)[k % 3],
                roughness=(0.01, 0.5, 1.0, 10.0)[k % 4], specular=(0.0, 0.5, 2.0)[k % 3],
                eta=(0.99, 1.01, 1.5, 0.02, 50.0)[k % 5], trans=1.0 if k % 6 == 5 else 0.0,
                clearcoatgloss=gloss if k % 6 != 5 else 1.0)
            k += 1
        pt = wl.PathTracer(gpu_ctx, wl.Accel(gpu_ctx, sc), sc)
        film, _ = pt.render(wl.pt_config(160, 120, spp=16, max_depth=10, strategy=strategy),
                            stats=False)
        films.append(film)
    assert torch.equal(films[0].view(torch.int32), films[1].view(torch.int32))
    assert (films[0][:, 0:3] != 0).any()


@pytest.mark.parametrize("name", ["wave", "textured", "deep"])
@pytest.mark.parametrize("w,h,depth", [(1, 1, 25), (64, 1, 3), (64, 1, 4), (257, 3, 25),
                                       (300, 217, 16), (1031, 777, 16)])
def test_finished_batches_equal_launched_bounces(gpu_ctx, name, w, h, depth):
    """Small batches run all but their first bounces in one kernel
    (render_samples); the traced render of the same frame launches every
    bounce: the same radiance, bit for bit."""
    import torch
    import wayland_amd as wl
    print(f"case: {name} {w} x {h} depth {depth}", flush=True)
    if name == "wave":
        sc = scenes.wavefront_scene(6, 3, width=w, height=h)
    elif name == "textured":
        sc = scenes.textured_cornell_box(w, h)
    else:
        sc = _deep_scene()
    pt = wl.PathTracer(gpu_ctx, wl.Accel(gpu_ctx, sc), sc)
    cfg = wl.pt_config(w, h, max_depth=depth, rr_depth=3)
    for frame in (0, 5):
        a = pt.render_samples(cfg, frame)
        b, _ = pt.trace_samples(cfg, frame, max_vertices=2)
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))


def test_finished_batches_count_their_rays(gpu_ctx):
    """The ray statistics of a small batch equal those of the same paths in a
    batch of two lanes (launched bounces)."""
    import wayland_amd as wl
    sc = scenes.wavefront_scene(4, 3, width=512, height=512)
    pt = wl.PathTracer(gpu_ctx, wl.Accel(gpu_ctx, sc), sc)
    _, big = pt.render(wl.pt_config(512, 512, spp=16, max_depth=8))
    small = [pt.render(wl.pt_config(512, 512, spp=4, max_depth=8, frame_offset=4 * k))[1]
             for k in range(4)]
    for key in ("paths", "extension_rays", "shadow_rays"):
        assert big[key] == sum(s[key] for s in small), key


def _variant(accel, variant):
    """The accel's rays take that variant's kernels from here on."""
    import ctypes as C
    from wayland_amd import _lib
    f = _lib.load().wl_accel_test_variant
    f.restype, f.argtypes = C.c_uint32, [C.c_void_p, C.c_uint32]
    assert f(accel.h, variant) == variant


@pytest.mark.parametrize("name", ["cornell", "ico"])
def test_traversal_variants_agree(gpu_ctx, name):
    """The kernels of a shallow BVH past 4 GB (1) and of a deep one (2), on one
    that is small: the same hits and films, bit for bit, from the raw traces, a
    finished batch, a batch of two lanes and a server."""
    import torch
    import wayland_amd as wl
    print(f"case: variants {name}", flush=True)
    if name == "cornell":
        sc = scenes.textured_cornell_box(256, 256)  # fewer nodes than the LDS copy holds
    else:
        sc = scenes.wavefront_scene(6, 3, width=256, height=256)
    rays = scenes.traversal_rays(100_003, seed=17)
    if name == "cornell":
        rays[:, 0:3] = rays[:, 0:3] * 2 - np.float32([1, 0, 1])

    def results(variant):
        accel = wl.Accel(gpu_ctx, sc)
        _variant(accel, variant)
        pt = wl.PathTracer(gpu_ctx, accel, sc)
        h, occ = _hits(accel, rays)
        out = [h[k].view(np.uint32) for k in ("t", "prim", "b1", "b2")] + [occ]
        for spp in (2, 72):  # 131,072 and 4,718,592 paths
            film, _ = pt.render(wl.pt_config(256, 256, spp=spp, max_depth=6), stats=False)
            out.append(film.view(torch.int32).cpu().numpy())
        server = wl.Server(gpu_ctx, batch_paths=1 << 20)
        films = [torch.zeros((256 * 256, 6), device="cuda") for _ in range(2)]
        server.render([dict(pt=pt, width=256, height=256, spp=2, frame_offset=8 * k, film=f)
                       for k, f in enumerate(films)])
        torch.cuda.synchronize()
        return out + [f.view(torch.int32).cpu().numpy() for f in films]

    short = results(0)
    for variant in (1, 2):
        for a, b in zip(short, results(variant)):
            assert np.array_equal(a, b), variant
