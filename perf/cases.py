"""The work that a user of this framework has it do, as timed cases.

A case is one pass of a program's loop through the public entry points of
risltc_amd.Context. Its "kind" says which:

  frame     a renderer's frame: constants, primary visibility, the shading
            pass, accumulation into the running mean
  open      a scene is opened: lights, LTC table and mesh are uploaded, the
            hierarchy is built, and the first frame is shaded
  batch     many views, each with its own mesh and lights, in one call or as
            a hipGraph whose views are updated before each replay
  learned   a frame of the learned pass: proposal tables, shading with the
            visibility cache, one training step on the frame's records
  proposal  the proposal network's inference for one view
  train     one step of the proposal's training on a large batch
  rays      a list of shadow rays against the scene's hierarchy

Scenes are the generators of risltc_amd.synth (a procedural city of up to 4M
triangles, and the small test scene, grid = 0). A mesh is generated once per
process, as a program reads its file once; the camera, the lights' radiance,
the noise seeds, the network's weights and the rays come from the seed.
"""
import copy
import functools
import math

import numpy as np
import torch

import risltc_amd
from risltc_amd import abi, ltcfit, synth

DEV = "cuda"


# ---- the cases ------------------------------------------------------------------

def _frame(name, width, height, grid, lights, candidates, spp, mis="optimal_clamped", technique="ltc_cp",
           sampling="reservoir", sample_count=1, scratch="own", moving=False):
    return dict(name=name, kind="frame", width=width, height=height, grid=grid, lights=lights, candidates=candidates,
                spp=spp, mis=mis, technique=technique, sampling=sampling, sample_count=sample_count, scratch=scratch,
                moving=moving)


def listed():
    return [
        # the smallest workload of the test suite and of an interactive
        # preview: launches and latency decide
        _frame("frame 256x256", 256, 256, 0, 64, 8, 1),
        # an ordinary window of odd size on a medium city with a moving
        # camera and another MIS heuristic
        _frame("frame 853x479", 853, 479, 128, 300, 16, 2, mis="power", moving=True),
        # the headline workload: 1080p, 1M triangles, 1024 lights
        _frame("frame 1080p", 1920, 1080, 270, 1024, 32, 4),
        # the large end: 4.1M triangles, 16384 lights, 16 samples per pixel
        _frame("frame 1080p large", 1920, 1080, 540, 16384, 32, 16),
        # the reference's comparison technique with a sampled target, as its
        # experiments run it
        _frame("frame psa 640x360", 640, 360, 270, 1024, 32, 2, technique="psa"),
        # opening the headline scene: upload, hierarchy, first frame
        dict(name="open city", kind="open", width=1920, height=1080, grid=270, lights=1024, candidates=32, spp=1),
        # views of the batched configuration: each its own mesh, light set,
        # resolution and candidate count
        dict(name="batch of 8", kind="batch", views=8, scale=1.0, graph=False),
        # the same as a graph of small views (thumbnails, probes), cameras
        # and noise updated before each replay
        dict(name="graph of 16 small", kind="batch", views=16, scale=0.125, graph=True),
        # the learned pass's loop at the headline size: inference, shading,
        # one training step per frame
        dict(name="learned 1080p", kind="learned", width=1920, height=1080, grid=270, lights=1024, candidates=24,
             spp=4, clusters=256, hidden=64, outputs=256, batch=8192),
        # the wide network's tables at 1080p, as every view of a learned batch
        # needs them
        dict(name="proposal wide 1080p", kind="proposal", width=1920, height=1080, grid=270, lights=4096,
             clusters=1024, hidden=128, outputs=1024, logits=False),
        # a small view's tables and logits (inspection, other samplers)
        dict(name="proposal 333x187", kind="proposal", width=333, height=187, grid=0, lights=64, clusters=64,
             hidden=64, outputs=256, logits=True),
        # training on the batch that the API takes by default
        dict(name="train 65536", kind="train", width=960, height=540, grid=128, lights=1024, spp=2, clusters=256,
             hidden=64, outputs=256, batch=65536),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame"] * 5 + ["open", "batch", "batch", "learned", "proposal", "train", "rays"])
    width = _log(rng, 96, 1920)
    height = max(33, min(1080, int(width * rng.uniform(0.4, 0.8))))
    grid = rng.choice([0, _log(rng, 40, 270), _log(rng, 40, 270)])
    lights = _log(rng, 24, 4096)
    if kind == "frame":
        technique = rng.choice(["ltc_cp"] * 6 + ["turk", "psa"])
        candidates, spp, count = rng.choice([4, 8, 13, 16, 32, 48]), rng.choice([1, 1, 2, 4, 7]), 1
        if technique == "psa":
            width, height, candidates, spp = min(width, 640), min(height, 360), min(candidates, 16), min(spp, 2)
        elif rng.random() < 0.15:
            count = rng.choice([2, 3])
        fits = width * height * spp * count <= abi.NOALLOC_MAX_SAMPLES
        c = _frame("", width, height, grid, lights, candidates, spp, technique=technique, sample_count=count,
                   mis=rng.choice(["balance", "power", "weighted", "optimal_clamped", "optimal_clamped", "optimal"]),
                   sampling=rng.choice(["reservoir"] * 7 + ["uniform"]),
                   scratch=rng.choice(["own", "fixed"]) if fits else "own", moving=rng.random() < 0.5)
        del c["name"]
        return c
    if kind == "open":
        return dict(kind="open", width=width, height=height, grid=grid, lights=lights, candidates=16, spp=1)
    if kind == "batch":
        return dict(kind="batch", views=rng.randint(2, 10), scale=rng.uniform(0.1, 0.8), graph=rng.random() < 0.5)
    clusters = min(lights, rng.choice([24, 100, 256]))
    hidden = rng.choice([64, 64, 128])
    if kind == "learned":
        return dict(kind="learned", width=width, height=height, grid=grid, lights=lights, candidates=rng.choice([8, 24]),
                    spp=rng.choice([1, 2, 4, 6]), clusters=clusters, hidden=hidden, outputs=256,
                    batch=256 * _log(rng, 4, 64))
    if kind == "proposal":
        if rng.random() < 0.5:
            return dict(kind="proposal", width=min(width, 480), height=min(height, 270), grid=0, lights=64,
                        clusters=rng.choice([40, 64]), hidden=hidden, outputs=rng.choice([256, 1024]), logits=True)
        outputs = rng.choice([256, 1024])
        return dict(kind="proposal", width=width, height=height, grid=grid, lights=lights,
                    clusters=min(lights, outputs) if outputs == 1024 else clusters, hidden=hidden, outputs=outputs,
                    logits=False)
    if kind == "train":
        return dict(kind="train", width=width, height=height, grid=grid, lights=lights, spp=rng.choice([1, 2]),
                    clusters=clusters, hidden=hidden, outputs=rng.choice([256, 1024]), batch=256 * _log(rng, 4, 256))
    return dict(kind="rays", grid=grid, lights=lights, rays=_log(rng, 1000, 4000000))


# ---- scenes ----------------------------------------------------------------------

@functools.lru_cache(maxsize=4)
def _scene(grid, lights):
    if grid == 0:
        return synth.small_scene(seed=0, light_count=lights)
    return synth.city_scene(seed=1, light_count=lights, grid=grid)


_view_scenes, _view_source = [], synth.batch_view_scenes(10)


def _view_scene(v):
    """The v-th scene of the batched configuration (generated in order)."""
    while len(_view_scenes) <= v:
        _view_scenes.append(next(_view_source))
    return _view_scenes[v]


@functools.lru_cache(maxsize=1)
def _table():
    rgba, rg, _ = ltcfit.table(51)
    return rgba, rg


def _camera(scene, rng):
    """A pose near the scene's own: a few metres (the small scene: less) off
    and slightly turned."""
    c, step = scene.camera, (1.0 if scene.name == "small" else 12.0)
    p = np.array(c.position_world_space, np.float64) + rng.uniform(-1.0, 1.0, 3) * (step, step, 0.0)
    p[2] += rng.uniform(0.0, 0.8 * step)
    return synth.make_camera(p, c.rotation_z + rng.uniform(-0.3, 0.3), c.rotation_x + rng.uniform(-0.08, 0.08),
                             fov=c.vertical_fov)


def _lit(scene, rng):
    """The scene with each light's radiance scaled (the records' first three
    floats) and a camera of its own."""
    s = copy.copy(scene)
    rec = np.frombuffer(scene.light_records, np.float32).reshape(scene.light_count, -1).copy()
    rec[:, 0:3] *= rng.uniform(0.5, 2.0, (scene.light_count, 1)).astype(np.float32)
    s.light_records = rec.tobytes()
    s.camera = _camera(scene, rng)
    return s


def _constants(ctx, scene, camera, width, height, noise_seed):
    m = scene.mesh
    return risltc_amd.write_frame_constants(camera, width, height, m.dequantization_factor, m.dequantization_summand,
                                            ctx.ltc_constants, noise_seed=noise_seed, animate=True)


_MIS = dict(balance=abi.MIS_BALANCE, power=abi.MIS_POWER, weighted=abi.MIS_WEIGHTED,
            optimal_clamped=abi.MIS_OPTIMAL_CLAMPED, optimal=abi.MIS_OPTIMAL)
_TECHNIQUE = dict(ltc_cp=abi.SAMPLE_POLYGON_LTC_CP, turk=abi.SAMPLE_POLYGON_AREA_TURK,
                  psa=abi.SAMPLE_POLYGON_PROJECTED_SOLID_ANGLE)


def _open(scene):
    ctx = risltc_amd.Context(0)
    ctx.load_scene(scene, *_table())
    return ctx


def _pixels(n, channels=4):
    return torch.zeros(n * channels, dtype=torch.float32, device=DEV)


def _weights(hidden, outputs, rng):
    """Network parameters in the library's order: each layer's weights [out][in],
    then its biases; the spread of a trained network's logits."""
    parts, shape = [], [(hidden, 96), (hidden, hidden), (hidden, hidden), (outputs, hidden)]
    for k, (o, i) in enumerate(shape):
        lim = math.sqrt(6.0 / i) * (1.5 if k == 3 else 1.0)
        parts += [rng.uniform(-lim, lim, (o, i)), rng.uniform(-0.1, 0.1, o)]
    return [np.asarray(p, np.float32) for p in parts]


# ---- prepare ---------------------------------------------------------------------

def prepare(case, seed):
    rng = np.random.default_rng(seed)
    return dict(frame=_prepare_frame, open=_prepare_open, batch=_prepare_batch, learned=_prepare_learned,
                proposal=_prepare_proposal, train=_prepare_train, rays=_prepare_rays)[case["kind"]](case, rng)


def _prepare_frame(case, rng):
    scene = _lit(_scene(case["grid"], case["lights"]), rng)
    ctx, n = _open(scene), case["width"] * case["height"]
    settings = abi.default_settings(
        sample_count=case["sample_count"], sample_count_light=case["spp"], mis_heuristic=_MIS[case["mis"]],
        light_sampling=abi.LIGHT_RESERVOIR if case["sampling"] == "reservoir" else abi.LIGHT_UNIFORM,
        polygon_sampling_technique=_TECHNIQUE[case["technique"]], ris_candidate_count=case["candidates"])
    return dict(case=case, ctx=ctx, scene=scene, settings=settings, noise=int(rng.integers(1 << 20)), at=0,
                cameras=[scene.camera] + [_camera(scene, rng) for _ in range(15 if case["moving"] else 0)],
                vis=torch.empty(n, dtype=torch.int32, device=DEV), out=_pixels(n), mean=_pixels(n))


def _prepare_open(case, rng):
    scene, n = _lit(_scene(case["grid"], case["lights"]), rng), case["width"] * case["height"]
    return dict(case=case, ctx=risltc_amd.Context(0), scene=scene, noise=int(rng.integers(1 << 20)),
                settings=abi.default_settings(sample_count_light=case["spp"], ris_candidate_count=case["candidates"]),
                vis=torch.empty(n, dtype=torch.int32, device=DEV), out=_pixels(n))


def _prepare_batch(case, rng):
    ctx = risltc_amd.Context(0)
    views, keep = [], []
    for v in range(case["views"]):
        scene = _lit(_view_scene(v % 10), rng)
        w, h = (max(16, int(round(x * case["scale"]))) for x in (scene.width, scene.height))
        if v == 0:
            ctx.load_scene(scene, *_table())
            lights = mesh = 0
        else:
            lights = ctx.add_light_set(scene.light_records, scene.light_count, scene.light_vmax)
            mesh = ctx.add_scene(scene)
        vis, out = torch.empty(w * h, dtype=torch.int32, device=DEV), _pixels(w * h)
        k = _constants(ctx, scene, scene.camera, w, h, int(rng.integers(1 << 20)))
        ctx.render_visibility_scene(mesh, k, vis)
        views.append(ctx.view(k, scene.settings(), vis, out, light_set=lights, scene=mesh))
        keep.append((scene, w, h, vis, out))
    return dict(case=case, ctx=ctx, views=views, keep=keep, at=int(rng.integers(1 << 20)),
                graph=ctx.graph(views) if case["graph"] else None)


def _learn(case, scene, rng):
    """A context with light clusters and a network of given weights."""
    ctx = _open(scene)
    ctx.cluster_lights(case["clusters"])
    ctx.proposal_set_network(case["hidden"], case["outputs"])
    weights = _weights(case["hidden"], case["outputs"], rng)
    ctx.proposal_set_params(np.concatenate([p.ravel() for p in weights]))
    return ctx, weights


def _prepare_learned(case, rng):
    scene = _lit(_scene(case["grid"], case["lights"]), rng)
    ctx, _ = _learn(case, scene, rng)
    ctx.proposal_cache(16, cell_size=1.0, prior_strength=float(np.float32(math.pi)), per_light=True)
    n = case["width"] * case["height"]
    vis = torch.empty(n, dtype=torch.int32, device=DEV)
    ctx.render_visibility(_constants(ctx, scene, scene.camera, case["width"], case["height"], 0), vis)
    settings = abi.default_settings(sample_count_light=case["spp"], ris_candidate_count=case["candidates"],
                                    proposal=abi.PROPOSAL_LEARNED, learned_floor_log2=7)
    return dict(case=case, ctx=ctx, scene=scene, settings=settings, noise=int(rng.integers(1 << 20)), at=0, vis=vis,
                out=_pixels(n))


def _view_directions(camera, width, height):
    """Pixel-to-ray rows (3 x 3, applied to (x, y, 1)) of the first-person
    camera, in 64 bits."""
    cz, sz = math.cos(camera.rotation_z), math.sin(camera.rotation_z)
    cx, sx = math.cos(camera.rotation_x), math.sin(camera.rotation_x)
    r = np.array([[cz, sz, 0.0], [-sz, cz, 0.0], [0.0, 0.0, 1.0]]) @ np.array([[1.0, 0.0, 0.0], [0.0, cx, sx], [0.0, -sx, cx]])
    t = math.tan(0.5 * camera.vertical_fov)
    x, y = -t * width / height * r[:, 0], t * r[:, 1]
    return np.stack([x * (2.0 / width), y * (2.0 / height), x * (1.0 / width - 1.0) + y * (1.0 / height - 1.0) - r[:, 2]], 1)


def _cast(scene, camera, width, height):
    """The visibility buffer of a mesh of few triangles by brute force in 64
    bits, as a host renderer's own raster pass would hand it over."""
    tri = torch.from_numpy(scene.mesh.dequantized().reshape(-1, 3, 3).astype(np.float64)).to(DEV)
    light = torch.from_numpy((scene.mesh.positions[0::3, 1] >> 31).astype(np.int64)).to(DEV)
    rows = torch.from_numpy(_view_directions(camera, width, height)).to(DEV)
    org = torch.tensor(list(camera.position_world_space), dtype=torch.float64, device=DEV)
    i = torch.arange(width * height, device=DEV)
    d = torch.stack([(i % width).double(), (i // width).double(), torch.ones(i.numel(), device=DEV).double()], 1) @ rows.T
    e1, e2, s = tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0], org - tri[:, 0]
    q = torch.linalg.cross(s, e1)
    best = torch.full((i.numel(),), math.inf, dtype=torch.float64, device=DEV)
    prim = torch.full((i.numel(),), -1, dtype=torch.int64, device=DEV)
    for k in range(tri.shape[0]):
        p = torch.linalg.cross(d, e2[k].expand_as(d))
        det = p @ e1[k]
        u, v, t = (p @ s[k]) / det, (d @ q[k]) / det, (e2[k] @ q[k]) / det
        hit = (u >= 0) & (v >= 0) & (u + v <= 1) & (t > 0) & (t < best)
        best = torch.where(hit, t, best)
        prim = torch.where(hit, k + (light[k] << 31), prim)
    return torch.where(prim >= 2 ** 31, prim - 2 ** 32, prim).to(torch.int32)


def _proposal_inputs(case, rng):
    scene = _lit(_scene(case["grid"], case["lights"]), rng)
    return scene, _weights(case["hidden"], case["outputs"], rng)


def _prepare_proposal(case, rng):
    scene, weights = _proposal_inputs(case, rng)
    ctx, n = _open(scene), case["width"] * case["height"]
    ctx.cluster_lights(case["clusters"])
    ctx.proposal_set_network(case["hidden"], case["outputs"])
    ctx.proposal_set_params(np.concatenate([p.ravel() for p in weights]))
    k = _constants(ctx, scene, scene.camera, case["width"], case["height"], 0)
    if case["logits"]:
        vis = _cast(scene, scene.camera, case["width"], case["height"])
    else:
        vis = torch.empty(n, dtype=torch.int32, device=DEV)
        ctx.render_visibility(k, vis)
    return dict(case=case, ctx=ctx, k=k, vis=vis, table=torch.zeros(n * 32, dtype=torch.uint8, device=DEV),
                logits=_pixels(n, case["outputs"]) if case["logits"] else None)


def _prepare_train(case, rng):
    scene = _lit(_scene(case["grid"], case["lights"]), rng)
    ctx, _ = _learn(case, scene, rng)
    n = case["width"] * case["height"]
    vis, out = torch.empty(n, dtype=torch.int32, device=DEV), _pixels(n)
    k = _constants(ctx, scene, scene.camera, case["width"], case["height"], int(rng.integers(1 << 20)))
    ctx.render_visibility(k, vis)
    # the frame whose samples are the training records
    ctx.shade(k, abi.default_settings(sample_count_light=case["spp"], ris_candidate_count=16), vis, out)
    return dict(case=case, ctx=ctx, k=k, vis=vis, out=out, at=int(rng.integers(1 << 20)))


def _prepare_rays(case, rng):
    scene = _lit(_scene(case["grid"], case["lights"]), rng)
    ctx, n = _open(scene), case["rays"]
    g = torch.Generator(device=DEV)
    g.manual_seed(int(rng.integers(1 << 31)))
    # from points above the ground towards lights, in the order of a raster
    # walk over the ground (neighbouring rays start near each other)
    half = 9.0 if case["grid"] == 0 else min(90.0, 2.0 * case["grid"])
    side = int(math.ceil(math.sqrt(n)))
    i = torch.arange(n, device=DEV)
    o = torch.stack([(i % side).float() / side * 2 - 1, (i // side).float() / side * 2 - 1, torch.zeros(n, device=DEV)], 1) * half
    o[:, 2] = 0.1 + 4.0 * torch.rand(n, generator=g, device=DEV)
    to = torch.from_numpy(np.stack([l.world.mean(0) for l in scene.lights])).to(DEV)
    d = to[torch.randint(scene.light_count, (n,), generator=g, device=DEV)] - o
    length = d.norm(dim=1, keepdim=True).clamp_min(1e-3)
    rays = torch.cat([o, torch.full_like(length, 1e-3), d / length, length - 1e-3], 1).contiguous()
    return dict(case=case, ctx=ctx, rays=rays, hits=torch.empty(n, dtype=torch.int32, device=DEV))


# ---- run -------------------------------------------------------------------------

def run(state):
    return dict(frame=_run_frame, open=_run_open, batch=_run_batch, learned=_run_learned, proposal=_run_proposal,
                train=_run_train, rays=_run_rays)[state["case"]["kind"]](state)


def _run_frame(s):
    case, ctx, at = s["case"], s["ctx"], s["at"]
    s["at"] += 1
    k = _constants(ctx, s["scene"], s["cameras"][at % len(s["cameras"])], case["width"], case["height"], s["noise"] + at)
    ctx.render_visibility(k, s["vis"])
    shade = ctx.shade_noalloc if case["scratch"] == "fixed" else ctx.shade
    shade(k, s["settings"], s["vis"], s["out"])
    if case["moving"]:
        return dict(visibility=s["vis"], frame=s["out"])
    ctx.accumulate(s["mean"], s["out"], case["width"] * case["height"], at)
    return dict(visibility=s["vis"], frame=s["out"], mean=s["mean"])


def _run_open(s):
    case, ctx, scene = s["case"], s["ctx"], s["scene"]
    ctx.load_scene(scene, *_table())
    k = _constants(ctx, scene, scene.camera, case["width"], case["height"], s["noise"])
    ctx.render_visibility(k, s["vis"])
    ctx.shade(k, s["settings"], s["vis"], s["out"])
    return dict(visibility=s["vis"], frame=s["out"])


def _run_batch(s):
    ctx = s["ctx"]
    s["at"] += 1
    for v, (scene, w, h, _, _) in zip(s["views"], s["keep"]):
        v.constants = _constants(ctx, scene, scene.camera, w, h, s["at"])
    if s["graph"] is not None:
        s["graph"].update(s["views"])
        s["graph"].launch()
    else:
        ctx.shade_batch(s["views"])
    return [k[4] for k in s["keep"]]


def _run_learned(s):
    case, ctx, at = s["case"], s["ctx"], s["at"]
    s["at"] += 1
    k = _constants(ctx, s["scene"], s["scene"].camera, case["width"], case["height"], s["noise"] + at)
    ctx.proposal_update(k, s["vis"])
    ctx.shade(k, s["settings"], s["vis"], s["out"])
    loss = ctx.proposal_train(k, s["vis"], batch=case["batch"], steps=1, lr=0.02, seed=at)
    params, grad = ctx.proposal_get_params()
    return dict(frame=s["out"], loss=loss, params=params, grad=grad)


def _run_proposal(s):
    s["ctx"].proposal_update(s["k"], s["vis"], table=s["table"], logits=s["logits"])
    return dict(table=s["table"], logits=s["logits"])


def _run_train(s):
    s["at"] += 1
    loss = s["ctx"].proposal_train(s["k"], s["vis"], batch=s["case"]["batch"], steps=1, lr=1e-3, seed=s["at"])
    params, grad = s["ctx"].proposal_get_params()
    return dict(loss=loss, params=params, grad=grad)


def _run_rays(s):
    s["ctx"].trace_shadow_rays(s["rays"], s["hits"])
    return s["hits"]


# ---- work and exact values ---------------------------------------------------------

def _mesh_triangles(grid):
    return 400 if grid == 0 else 14 * grid * grid


def _network_flops(hidden, outputs):
    return 2 * (96 * hidden + 2 * hidden * hidden + hidden * outputs)


def _shading(pixels, spp, count, candidates, lights):
    """A pixel's visibility word, vertices, material and colour, the lights
    and the LTC table; per candidate two plane tests and, for the fraction
    with a part above the horizon, the two clipped-polygon integrals; per
    sample the two prepared polygons and the walk of its shadow rays."""
    return dict(bytes=pixels * 69 + lights * 176 + 64 * 64 * 12,
                flops=pixels * spp * (candidates * 190 + count * 2900))


def work(case):
    kind = case["kind"]
    if kind == "rays":
        # a ray in, a word out, about 60 nodes of 25 operations
        return dict(bytes=36 * case["rays"], flops=1500 * case["rays"])
    if kind == "batch":
        total = dict(bytes=0, flops=0)
        for v in range(case["views"]):
            s = _view_scene(v % 10)
            px = max(16, round(s.width * case["scale"])) * max(16, round(s.height * case["scale"]))
            w = _shading(px, s.spp, 1, s.candidates, s.light_count)
            total = dict(bytes=total["bytes"] + w["bytes"], flops=total["flops"] + w["flops"])
        return total
    pixels = case["width"] * case["height"]
    if kind == "frame":
        w = _shading(pixels, case["spp"], case["sample_count"],
                     case["candidates"] if case["sampling"] == "reservoir" else 0, case["lights"])
        return dict(bytes=w["bytes"] + pixels * (4 + 32), flops=w["flops"] + pixels * 1500)
    if kind == "open":
        w, n = _shading(pixels, case["spp"], 1, case["candidates"], case["lights"]), _mesh_triangles(case["grid"])
        # mesh in, hierarchy out, a box union and a cost per triangle and level
        return dict(bytes=w["bytes"] + n * (49 + 80), flops=w["flops"] + pixels * 1500 + n * math.log2(n) * 30)
    net = _network_flops(case["hidden"], case["outputs"])
    if kind == "learned":
        w = _shading(pixels, case["spp"], 1, case["candidates"], case["lights"])
        return dict(bytes=w["bytes"] + pixels * (32 + 8 * case["spp"]),
                    flops=w["flops"] + pixels * net + 3 * case["batch"] * net)
    if kind == "proposal":
        return dict(bytes=pixels * (53 + 32 + (4 * case["outputs"] if case["logits"] else 0)), flops=pixels * net)
    return dict(bytes=case["batch"] * (57 + 4) + net // 2 * 24, flops=3 * case["batch"] * net)


def _octahedral(q):
    """Unit normals of 16-bit octahedral pairs (.., 2), in 64 bits."""
    f = 2.0 * (65534.0 / 65535.0)
    o = q / 65535.0 * f - (32768.0 / 65535.0) * f
    z = 1.0 - o.abs().sum(-1)
    fold = (1.0 - o.flip(-1).abs()) * torch.where(o >= 0, 1.0, -1.0)
    n = torch.cat([torch.where(z[..., None] < 0, fold, o), z[..., None]], -1)
    return n / n.norm(dim=-1, keepdim=True)


def _features(scene, camera, width, height, vis):
    """The 96 inputs of the network for every pixel, in 64 bits (zeros where
    no mesh triangle is seen)."""
    mesh = scene.mesh
    seen = (vis >= 0).nonzero().squeeze(1)
    prim = vis[seen].long()

    def rows(a, dtype=np.float64):
        return torch.from_numpy(np.asarray(a, dtype)).to(DEV)
    tri = rows(mesh.dequantized().reshape(-1, 3, 3))[prim]
    normals = _octahedral(rows(mesh.normals_uv.reshape(-1, 3, 4)[..., :2]))[prim]
    mat = rows(scene.materials)[rows(mesh.material_index, np.int64)[prim]]
    org = rows(list(camera.position_world_space))
    xy1 = torch.stack([(seen % width).double(), (seen // width).double(), torch.ones_like(seen).double()], 1)
    ray = xy1 @ rows(_view_directions(camera, width, height)).T
    e0, e1, r0 = tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0], org - tri[:, 0]
    c = torch.linalg.cross(ray, e1)
    det = (e0 * c).sum(1)
    by = (r0 * c).sum(1) / det
    bz = -(ray * torch.linalg.cross(e0, r0)).sum(1) / det
    b = torch.stack([1.0 - by - bz, by, bz], 1)[..., None]
    pos, n = (tri * b).sum(1), (normals * b).sum(1)
    n = n / n.norm(dim=1, keepdim=True)
    o = org - pos
    o = o / o.norm(dim=1, keepdim=True)
    no = (n * o).sum(1, keepdim=True)
    n, no = torch.where(no < 0, -n, n), no.abs()
    r = 2.0 * no * n - o
    metal = mat[:, 5:6]
    lum = mat[:, 0:3] @ rows([[0.2126], [0.7152], [0.0722]])
    alpha = (mat[:, 4:5] ** 2).clamp(0.0064, 1.0)
    lo, ext = rows(mesh.dequantization_summand), rows(mesh.dequantization_factor) * 2097151.0
    q = (pos - lo - 0.5 * ext) * (2.0 / ext)

    def waves(v, octaves):
        return [w for j in range(octaves) for a in range(3)
                for x in v for w in (torch.sin(math.pi * 2 ** j * x[:, a:a + 1]), torch.cos(math.pi * 2 ** j * x[:, a:a + 1]))]
    cols = [q] + waves([q], 7) + [n, o, r, alpha, no, lum * (1 - metal), 0.02 * (1 - metal) + lum * metal]
    cols += waves([n, r], 2) + waves([o], 1) + [torch.ones_like(no)]
    X = torch.zeros(vis.numel(), 96, dtype=torch.float64, device=DEV)
    X[seen, :89] = torch.cat(cols, 1)
    return X


def exact(case, seed):
    """Logits of the proposal network by plain torch in 64 bits. The other
    kinds' outputs have no such value: a frame is decided by comparisons of
    32-bit weights with 32-bit noise (which light is taken, which ray is
    traced), the training records are such decisions, and the remaining
    outputs are whole numbers."""
    if case["kind"] != "proposal" or not case["logits"]:
        return None
    scene, w = _proposal_inputs(case, np.random.default_rng(seed))
    vis = _cast(scene, scene.camera, case["width"], case["height"])
    h = _features(scene, scene.camera, case["width"], case["height"], vis)
    for k in range(0, 8, 2):
        h = h @ torch.from_numpy(w[k]).double().to(DEV).T + torch.from_numpy(w[k + 1]).double().to(DEV)
        h = h.clamp_min(0.0) if k < 6 else h
    return dict(table=None, logits=h.reshape(-1))
