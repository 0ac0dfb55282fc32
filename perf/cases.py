"""Performance cases of the renderer: what a program does with it, through its public calls.

Kinds of cases:

  render  a whole render: begin, `passes` passes, the image.  The radius shrinks from pass to pass, unless alpha is 1 (the
          setting for comparisons against a reference image).  With `graph` the passes are captured and replayed, with
          `guided` photon emission is steered by the learned proposal, which starts anew and trains as the render goes.
  batch   several scenes of uneven size in progress at a fixed radius: `passes` more passes, one launch for all scenes
          each, then their images.
  trace   closest hits of a host array of rays; `static` is the form that does not allocate.
  shadow  occlusion of a host array of rays through alpha-textured screens.
  train   the gradient of the emission proposal's network on a given deposit histogram, then `passes` Adam steps.

Every case starts from its own photon and camera sample streams (the seed picks them), so another seed gives other
photons, pixels, rays or histograms in the same scene.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "friendsrender-r-public_amd"))

import scenes  # noqa: E402
import sppm_amd  # noqa: E402

FLT_MAX = 3.4028234663852886e38


def _case(kind, scene="box", size=0, width=0, height=0, photons=0, passes=1, bvh=8, alpha=1.0, radius=0.01, lens=False,
          halton=False, nee=0, shared=False, graph=False, guided=False, wide=False, scenes=0, rays=0, static=False):
    return dict(kind=kind, scene=scene, size=size, width=width, height=height, photons=photons, passes=passes, bvh=bvh,
                alpha=alpha, radius=radius, lens=lens, halton=halton, nee=nee, shared=shared, graph=graph, guided=guided,
                wide=wide, scenes=scenes, rays=rays, static=static)


def listed():
    return [
        # a thumbnail refreshed while a scene is edited: few pixels, few photons, the time of the launches themselves
        dict(_case("render", "box", width=64, height=64, photons=5_000, passes=8, bvh=4, alpha=0.9), name="thumbnail_64"),
        # the plain box workload, whole: 256^2, 100k photons, 16 passes, BVH4; the estimate is kept besides the image so
        # that renders of several machines can be merged
        dict(_case("render", "box", width=256, height=256, photons=100_000, passes=16, bvh=4, alpha=0.9, radius=0.0087,
                   shared=True), name="box_256"),
        # a small textured scene with every material at sizes that divide nothing
        dict(_case("render", "full", size=20, width=333, height=217, photons=77_777, passes=8, alpha=0.7, radius=0.02,
                   lens=True, shared=True), name="full_333x217"),
        # the main scene's transmitting surfaces under a sky, with next-event estimation and the Halton camera sampler
        dict(_case("render", "sky", width=400, height=300, photons=150_001, passes=8, alpha=0.9, radius=0.01, halton=True,
                   nee=2, shared=True), name="sky_nee_400x300"),
        # the headline: full-material scene with 203k triangles, 1024^2, 1M photons per pass
        dict(_case("render", "full", size=100, width=1024, height=1024, photons=1_000_000, passes=32, alpha=0.7,
                   radius=0.02, lens=True, shared=True), name="full_1024"),
        # the same scene at 512^2 with captured passes, as a progressive viewer runs it
        dict(_case("render", "full", size=100, width=512, height=512, photons=250_000, passes=16, radius=0.01, lens=True,
                   shared=True, graph=True), name="full_512_graph"),
        # occluded light, plain and guided (64x4 bf16 network trained every 4th pass) as the time-to-error comparison
        # runs them: 298k triangles, 1024^2, 1M photons
        dict(_case("render", "occluded", size=61, width=1024, height=1024, photons=1_000_000, passes=16, radius=0.02,
                   guided=True), name="occluded_1024_guided"),
        # caustics: 500k triangles of rough glass, 4M photons per pass, 128x6 fp16 network trained every pass
        dict(_case("render", "caustic", size=500_000, width=1024, height=1024, photons=4_000_000, passes=8, alpha=0.7,
                   radius=0.01, lens=True, guided=True, wide=True), name="caustic_4m_guided"),
        # a dozen uneven scenes in one batch
        dict(_case("batch", scenes=12, photons=1, passes=2, radius=0.02), name="batch_12"),
        # a million rays through the 203k-triangle scene (picking, ambient occlusion, radiosity of another program)
        dict(_case("trace", "full", size=100, rays=1_000_000), name="rays_1m"),
        # shadow rays through screens, as a direct-light integrator asks for them, few enough to be latency
        dict(_case("shadow", "screens", rays=20_000, bvh=4), name="shadow_20k"),
        # training of the wide proposal network
        dict(_case("train", wide=True, size=50), name="train_128x6"),
    ]


def draw(rng):
    def log(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(["render"] * 6 + ["batch", "trace", "shadow", "train"])
    if kind == "render":
        scene = rng.choice(["box", "full", "full", "sky", "occluded", "caustic", "transmit"])
        size = {"full": log(10, 100), "occluded": log(8, 61), "caustic": log(5_000, 500_000)}.get(scene, 0)
        w = log(48, 1100)
        h = max(32, min(1100, int(w * rng.uniform(0.5, 1.5))))
        photons = max(2_000, min(1_500_000, int(w * h * rng.uniform(0.3, 2.5))))
        guided = scene in ("box", "full", "occluded", "caustic") and rng.random() < 0.4
        graph = rng.random() < 0.3
        return _case(kind, scene, size, w, h, photons, passes=rng.randint(4, 16), bvh=rng.choice([2, 4, 8, 8]),
                     alpha=rng.choice([0.7, 0.9, 1.0]), radius=rng.uniform(0.005, 0.02),
                     lens=scene in ("full", "caustic"), halton=not graph and rng.random() < 0.2,
                     nee=rng.choice([0, 0, 1, 2]), shared=not guided and rng.random() < 0.6, graph=graph, guided=guided,
                     wide=guided and rng.random() < 0.4)
    if kind == "batch":
        return _case("batch", scenes=rng.randint(2, 16), photons=rng.randint(1, 1000), passes=rng.randint(1, 3),
                     radius=rng.uniform(0.01, 0.02), bvh=rng.choice([4, 8]))
    if kind == "train":
        return _case("train", size=log(2, 1000), passes=rng.randint(1, 4), wide=rng.random() < 0.5)
    static = kind == "trace" and rng.random() < 0.4
    rays = log(1, 65_536 if static else 1_000_000)
    scene = "screens" if kind == "shadow" else rng.choice(["box", "full", "occluded", "transmit"])
    return _case(kind, scene, {"full": log(10, 60), "occluded": log(8, 40)}.get(scene, 0), rays=rays,
                 bvh=rng.choice([2, 4, 8]), static=static)


# ---- inputs -------------------------------------------------------------------
@functools.lru_cache(maxsize=24)
def _scene(name, size):
    if name == "box":
        return scenes.box_scene()
    if name == "full":
        return scenes.full_scene(freq=size, tex_size=512 if size > 40 else 128)
    if name == "occluded":
        return scenes.occluded_scene(clutter_freq=size)
    if name == "caustic":
        return scenes.caustic_scene(tris=size, tex_size=1024 if size > 100_000 else 256)
    if name == "screens":
        return scenes.screens_scene()
    if name == "transmit":
        return scenes.transmit_scene()
    if name == "sky":  # the transmitting surfaces, open to a sky
        sc = scenes.transmit_scene()
        out = scenes.Scene(sc.pos, sc.nrm, sc.uv, sc.attr, sc.attrs, list(sc.textures) + [scenes.sky_texture()])
        out.ibl = len(out.textures) - 1
        return out
    raise ValueError(name)


@functools.lru_cache(maxsize=4)
def _batch(n, seed):
    return scenes.batch_workload(n=n, seed=seed, tri_range=(2_000, 30_000), max_meshes=4, resolutions=(128, 256, 512))


def _camera(case, seed):
    w, h = case["width"], case["height"]
    if case["scene"] == "occluded":
        cam = scenes.occluded_camera(w, h)
    elif case["scene"] == "caustic":
        cam = scenes.caustic_cameras(1, w, h)[0]
    elif case["lens"]:
        cam = scenes.thinlens_camera(w, h)
    else:
        cam = scenes.pinhole_camera(w, h)
    cam = dict(cam, sampler_id=seed % 1_000_003)
    if case["halton"]:
        cam["sampler"] = sppm_amd.SAMPLER_HALTON
    return cam


def _steps(seed):
    """First step of the photon and eye paths' random streams."""
    return (seed * 7919) % 1_000_003


def _rays(case, seed, scene):
    rng = np.random.default_rng(seed)
    n = case["rays"]
    p = scene.pos.reshape(-1, 3)
    lo, hi = p.min(0), p.max(0)
    org = lo + (hi - lo) * rng.uniform(0.05, 0.95, (n, 3))
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return org.astype(np.float32), d.astype(np.float32), rng.uniform(0.1, 1.5, n).astype(np.float32)


def _histogram(case, seed):
    """A deposit histogram: `size` of a thousand cells reach the image, few of them carry most of its light."""
    rng = np.random.default_rng(seed)
    h = rng.gamma(0.3, 1.0, sppm_amd.GUIDE_CELLS) * (rng.random(sppm_amd.GUIDE_CELLS) < 1e-3 * case["size"])
    return h.astype(np.float32)


def _network(case):
    return dict(hidden=128, layers=6, fp16=True) if case["wide"] else dict(hidden=64, layers=4, fp16=False)


def prepare(case, seed):
    kind = case["kind"]
    state = dict(case=case)
    if kind == "batch":
        rs = []
        for w in _batch(case["scenes"], case["photons"]):
            rs.append(sppm_amd.Renderer(w["scene"], dict(w["cam"], sampler_id=seed % 1_000_003), case["alpha"],
                                        case["radius"] * w["scene"].diagonal(), w["photons"], bvh_width=case["bvh"],
                                        step_offset=_steps(seed)))
        state["batch"] = sppm_amd.Batch(rs)
        return state
    if kind == "train":
        r = sppm_amd.Renderer(_scene("box", 0), scenes.pinhole_camera(32, 32), 0.9, 0.015, 2000, bvh_width=4)
        r.guide_set(True, learning_rate=1e-3, train_steps=1, seed=1 + seed % 1_000_003, **_network(case))
        # an output layer as training leaves it (it starts at zero)
        w = r.guide_weights()
        h = _network(case)["hidden"]
        w[-h - 1:] = np.random.default_rng(seed + 1).normal(0.0, 0.05, h + 1)
        r.guide_weights(w)
        state.update(renderer=r, weights=w, hist=_histogram(case, seed))
        return state
    scene = _scene(case["scene"], case["size"])
    if kind in ("trace", "shadow"):
        state["renderer"] = sppm_amd.Renderer(scene, scenes.pinhole_camera(32, 32), 0.9, 0.015, 2000,
                                              bvh_width=case["bvh"])
        state["rays"] = _rays(case, seed, scene)
        return state
    r = sppm_amd.Renderer(scene, _camera(case, seed), case["alpha"], case["radius"] * scene.diagonal(), case["photons"],
                          bvh_width=case["bvh"], nee=case["nee"], step_offset=_steps(seed))
    if case["guided"]:
        every = 4 if not (case["graph"] or case["wide"]) else 1
        state["guide"] = dict(mix_plain=0.5, learning_rate=1e-3, train_steps=2 if every == 4 else 1,
                              seed=1 + seed % 1_000_003, history_decay=0.95, train_interval=every,
                              target=sppm_amd.GUIDE_TARGET_RMS, **_network(case))
    state["renderer"] = r
    return state


# ---- one pass -------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        b = state["batch"]
        for _ in range(case["passes"]):
            b.pass_()
        b.sync()
        return [r.reconstruct() for r in b.renderers]
    r = state["renderer"]
    if kind == "trace":
        org, d, _ = state["rays"]
        return (r.trace_static if case["static"] else r.trace)(org, d)
    if kind == "shadow":
        org, d, far = state["rays"]
        return r.occluded(org, d, 1e-4, far)
    if kind == "train":
        r.guide_weights(state["weights"])
        loss, grad = r.guide_gradient(state["hist"])
        r.guide_train(state["hist"], case["passes"])
        return dict(loss=loss, grad=grad, weights=r.guide_weights())
    if case["guided"]:
        r.guide_set(True, **state["guide"])
    r.begin()
    if case["graph"]:
        r.graph_capture()
    for _ in range(case["passes"]):
        r.pass_(stats=False)
    out = dict(image=r.reconstruct())
    if case["shared"]:
        out.update(r.read_shared())
    return out


# ---- what a pass cannot do without -----------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "train":
        net = _network(case)
        n = sppm_amd.guide_nparams(net["hidden"], net["layers"])
        # a forward (2 per weight and cell) and a backward (4) for the gradient call and for each Adam step; the weights
        # and the histogram in, the weights and the gradient out, Adam's two moments in and out
        return dict(flops=(1 + case["passes"]) * 6.0 * n * sppm_amd.GUIDE_CELLS,
                    bytes=4.0 * (2 * sppm_amd.GUIDE_CELLS + 7 * n))
    if kind in ("trace", "shadow"):
        tris = _triangles(case["scene"], case["size"])
        out = 16 if kind == "trace" else 4
        return dict(bytes=case["rays"] * (28.0 + out) + 48.0 * min(tris, 8 * case["rays"]),
                    flops=case["rays"] * _ray_flops(tris))
    if kind == "batch":
        # 2k-30k triangles and 128^2-512^2 pixels per scene, 0.5-2 photons per pixel
        jobs = [(28_000, 114_000, 143_000)] * case["scenes"]
    else:
        jobs = [(_triangles(case["scene"], case["size"]), case["width"] * case["height"], case["photons"])]
    b = f = 0.0
    for tris, pixels, photons in jobs:
        stored = 1.7 * photons
        # pi r^2 over the surfaces a photon lands on (about 6 diagonals^2 / 3), times the stored photons; the radius of
        # a shrinking render has lost about a third of its square by its middle
        shrink = 0.7 if case["alpha"] < 1.0 else 1.0
        near = stored * math.pi * case["radius"] ** 2 / 2.0 * shrink
        # photons written and read once (44 bytes), the estimate read and written (24 bytes)
        b += case["passes"] * (88.0 * stored + 48.0 * pixels) + 48.0 * tris + 16.0 * pixels
        # 2.3 closest hits per photon path, 1.2 per pixel; per neighbour the distance and a flux term
        f += case["passes"] * ((2.3 * photons + 1.2 * pixels) * _ray_flops(tris) + 0.7 * pixels * near * 20.0)
    return dict(bytes=b, flops=f)


def _triangles(scene, size):
    return {"full": 20 * size * size + 3_100, "occluded": 80 * size * size + 18, "caustic": size + 4, "screens": 80,
            "transmit": 1_600, "sky": 1_600}.get(scene, 3_100)


def _ray_flops(tris):
    """Eight boxes (about 25 operations each) per level of an 8-wide tree, and four triangles."""
    return 200.0 * max(1.0, math.log(max(tris, 8)) / math.log(8.0)) + 4 * 45.0


# ---- how exact ------------------------------------------------------------------------
def tolerance(case):
    kind = case["kind"]
    if kind in ("trace", "shadow"):
        return "exact"  # the nearest hit, ties to the lowest facet: one answer
    if kind == "train":
        # activations and gradients are rounded to 16 bits between the layers, 1e-2 to 4e-2 from the 64-bit gradient
        return {"rel": 1e-2}
    if case["guided"]:
        # the proposal's last bits move a few photons to other cells of the light, and their paths with them: 1e-3 and
        # 0.009 when its weights are off by 1e-7, at 1M photons per pass; less light per pixel at smaller ones
        return {"rel": 1e-2, "max": 0.2}
    # photons, hit points and neighbours are the same ones, and whole numbers too; the flux is summed in float32 (1.5e-7
    # and 3.3e-6 between groups of 32 and of 64 hit points, which sum it in another order)
    return {"rel": 1e-6, "max": 2e-5}


def exact(case, seed):
    if case["kind"] == "train":
        return _exact_train(case, seed)
    if case["kind"] == "trace":
        scene = _scene(case["scene"], case["size"])
        if scene.nfacets * case["rays"] <= 4e9:
            return _exact_trace(case, seed, scene)
    # renders: what a photon path hits and where it ends is decided by float32 comparisons along it, so there is no
    # 64-bit value of an image to compare with
    return None


def _exact_trace(case, seed, scene):
    org, d, _ = (torch.from_numpy(a).cuda().double() for a in _rays(case, seed, scene))
    p = torch.from_numpy(scene.pos).cuda().double().view(-1, 3, 3)
    p0, e1, e2 = p[:, 0], p[:, 1], p[:, 2]
    e1, e2 = e1 - p0, e2 - p0
    n, nt = org.shape[0], p0.shape[0]
    t_out, u_out, v_out = (torch.zeros(n, dtype=torch.float64) for _ in range(3))
    step = max(1, 20_000_000 // nt)
    for a in range(0, n, step):
        o, dd = org[a:a + step, None, :], d[a:a + step, None, :]
        ps = torch.linalg.cross(dd.expand(-1, nt, -1), e2.expand(o.shape[0], -1, -1))
        det = (e1 * ps).sum(-1)
        s = o - p0
        u = (s * ps).sum(-1) / det
        q = torch.linalg.cross(s, e1.expand(o.shape[0], -1, -1))
        v = (dd * q).sum(-1) / det
        t = (e2 * q).sum(-1) / det
        ok = (det != 0) & (u >= 0) & (u <= 1) & (v >= 0) & (u + v <= 1) & (t > 1e-4)
        t = torch.where(ok, t, torch.full_like(t, float("inf")))
        best, k = t.min(1)
        k = k[:, None]
        miss = torch.isinf(best)
        t_out[a:a + step] = torch.where(miss, torch.full_like(best, FLT_MAX), best).cpu()
        u_out[a:a + step] = torch.where(miss, torch.zeros_like(best), u.gather(1, k)[:, 0]).cpu()
        v_out[a:a + step] = torch.where(miss, torch.zeros_like(best), v.gather(1, k)[:, 0]).cpu()
    return None, t_out, u_out, v_out


def _exact_train(case, seed):
    state = prepare(case, seed)  # for the weights that a new network starts with
    theta, hist = state["weights"], state["hist"]
    net = _network(case)
    th = torch.from_numpy(theta).cuda().double().requires_grad_(True)
    c = np.arange(sppm_amd.GUIDE_CELLS)
    it, is_, iv, iu = c % 16, (c // 16) % 16, (c // 256) % 32, c // 8192
    co = np.stack([2 * (iu + 0.5) / 32 - 1, 2 * (iv + 0.5) / 32 - 1, (is_ + 0.5) / 8 - 1, (it + 0.5) / 8 - 1], 1)
    freq = (np.pi * 2.0 ** (np.arange(8) / 2.0)).astype(np.float32).astype(np.float64)
    x = co[:, :, None] * freq
    x = torch.from_numpy(np.stack([np.sin(x), np.cos(x)], -1).reshape(len(c), 64)).cuda()
    o = 0
    for k in range(net["layers"]):
        n = 64 if k == 0 else net["hidden"]
        w = th[o:o + n * net["hidden"]].view(n, net["hidden"])
        o += n * net["hidden"]
        x = torch.relu(x @ w + th[o:o + net["hidden"]])
        o += net["hidden"]
    logit = x @ th[o:o + net["hidden"]] + th[o + net["hidden"]]
    w = torch.from_numpy(hist).cuda().double()
    loss = -(w / w.sum() * torch.log_softmax(logit, 0)).sum()
    loss.backward()
    # Adam's first steps divide the gradient by its own size, so their result has no meaningful 64-bit value
    return dict(loss=float(loss.detach()), grad=th.grad.cpu().numpy(), weights=None)
