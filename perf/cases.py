"""The work a program has this renderer do, as measurable cases.

Each case is a dict of plain sizes and options; its "kind" says which pass it
is.  prepare() sets up what such a program holds before the call (a context
with its cloud, uniforms, shadow volume, network or job list), run() makes the
one pass through the public entry points and returns what the program reads
back: images, trees, data sets, weights.

  pt       path-traced frames of a cloud, then the image
  relight  a new sun direction: shadow volume, first frame, image
  upload   a new cloud from host memory: grid, shadow volume, frame, image
  beams    one photon-beam frame: trace, LBVH, gather, image
  lbvh     an LBVH over beams already on the device, read back
  ppm      one photon-mapping frame: trace, estimate, image
  learned  a learned in-scattering render, then the image
  collect  training data of one cloud, read back
  train    training steps on a device-resident data set, weights read back
  batch    several clouds and views in one batched launch, all images
"""
import ctypes as C
import math

import numpy as np
import torch

import cr_import

pkg = cr_import.package()
cfg = cr_import.configs()
S = pkg.structs

GLOBAL, DDA = S.CR_TRACK_GLOBAL_MAJORANT, S.CR_TRACK_BRICK_DDA
NEE_SV, NEE_RATIO, NEE_NONE = S.CR_NEE_SHADOW_VOLUME, S.CR_NEE_RATIO_TRACKING, S.CR_NEE_NONE
F32, F16 = S.CR_DTYPE_F32, S.CR_DTYPE_F16
DENSE, BRICK4 = S.CR_GRID_DENSE, S.CR_GRID_BRICK4

# The default cloud: the c1 workload's 128^3 FP32 cumulus with its tracker.
C1 = dict(nx=128, ny=128, nz=128, octaves=6, anvil=False, f16=False, brick4=False, dda=False, nee=NEE_SV, sv=256,
          albedo=0.9, bounces=16, camera_z=-0.2)


def listed():
    return [
        # One frame of the reference's interactive loop at its 800x600 window.
        dict(C1, name="preview", kind="pt", width=800, height=600, spp=1, static=False),
        # The c1 workload: a small image, many frames per pixel.
        dict(C1, name="c1", kind="pt", width=256, height=256, spp=64, static=False),
        # The c2 workload, the production render: 1 GiB FP16 anvil, 1080p, 256 spp.
        dict(name="c2", kind="pt", width=1920, height=1080, spp=256, static=False, nx=1024, ny=512, nz=1024, octaves=8,
             anvil=True, f16=True, brick4=True, dda=True, nee=NEE_RATIO, sv=0, albedo=0.999, bounces=256,
             camera_z=-0.15),
        # The interactive loop after the sun was moved: shadow volume again, first frame.
        dict(C1, name="relight", kind="relight", width=800, height=600),
        # A simulation's next time step, ragged, handed over from host memory in .xyz order.
        dict(name="upload", kind="upload", nx=189, ny=131, nz=221, src_f16=False, zfast=True, f16=True, brick4=True,
             dda=True, sv=128, width=800, height=600),
        # The c3 workload as a frame of the technique: 2^22 beams, 1080p gather.
        dict(name="beams", kind="beams", paths=1 << 19, max_beams=1 << 22, radius=0.002, size=128, width=1920,
             height=1080),
        # The beam count the reference allocates for (4096): a build is all launches.
        dict(name="lbvh_4096", kind="lbvh", beams=4096),
        # Photon mapping of the c1 cloud, 12 800 paths into 100^3 cells.
        dict(name="ppm", kind="ppm", paths=12800, cells=100, size=128, width=1920, height=1080),
        # The learned render at the sample count the c5 workload settles on.
        dict(name="learned", kind="learned", spp=32, size=128, width=1920, height=1080),
        # Training data of one cloud (the c5 workload collects 400 of these).
        dict(name="collect", kind="collect", frames=8, spp=256, points=20000, size=128, width=256, height=256),
        # 100 Adam steps of the c5 workload's batch.
        dict(name="train", kind="train", steps=100, batch=8192, points=100000),
        # c4's job statistics (grids, images, spp, suns), a launch of sixteen.
        dict(name="batch", kind="batch", jobs=16, draw_seed=4, grid_hi=256, image_hi=512, spp_hi=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _even(v):
    return v + (v & 1)


def _view(rng, lo, hi, aspect=True):
    """An image of lo..hi pixels on a side; the camera's images have even sides."""
    w = _even(_log_int(rng, lo, hi))
    return w, _even(max(16, int(w * rng.choice([1.0, 0.75, 0.5625])))) if aspect else w


def draw(rng):
    kind = rng.choice(["pt", "pt", "pt", "relight", "upload", "beams", "lbvh", "ppm", "learned", "collect", "train",
                       "batch"])
    if kind == "pt":
        w, h = _view(rng, 64, 1920)
        n = _log_int(rng, 48, 320)
        nee = rng.choice([NEE_SV, NEE_RATIO, NEE_NONE])
        return dict(kind=kind, width=w, height=h, spp=max(1, min(_log_int(rng, 1, 256), (48 << 20) // (w * h))),
                    static=rng.random() < 0.3, nx=n, ny=_log_int(rng, 33, n + 33), nz=_log_int(rng, 33, n + 33),
                    octaves=6, anvil=rng.random() < 0.3, f16=rng.random() < 0.5, brick4=rng.random() < 0.5,
                    dda=rng.random() < 0.6, nee=nee, sv=_log_int(rng, 48, 256) if nee == NEE_SV else 0,
                    albedo=round(rng.uniform(0.8, 1.0), 3), bounces=rng.choice([1, 16, 64, 256]),
                    camera_z=round(rng.uniform(-0.6, -0.1), 3))
    if kind == "relight":
        w, h = _view(rng, 128, 1280)
        return dict(C1, kind=kind, width=w, height=h, nx=_log_int(rng, 48, 300), ny=_log_int(rng, 48, 300),
                    nz=_log_int(rng, 48, 300), f16=rng.random() < 0.5, brick4=rng.random() < 0.5,
                    sv=_log_int(rng, 64, 400))
    if kind == "upload":
        w, h = _view(rng, 128, 1280)
        return dict(kind=kind, nx=_log_int(rng, 31, 300), ny=_log_int(rng, 31, 300), nz=_log_int(rng, 31, 300),
                    src_f16=rng.random() < 0.3, zfast=rng.random() < 0.5, f16=rng.random() < 0.5,
                    brick4=rng.random() < 0.5, dda=rng.random() < 0.5, sv=_log_int(rng, 48, 256), width=w, height=h)
    if kind == "beams":
        w, h = _view(rng, 128, 1920)
        return dict(kind=kind, paths=_log_int(rng, 500, 300000), max_beams=1 << 22,
                    radius=round(rng.uniform(0.002, 0.02), 4), size=_log_int(rng, 48, 256), width=w, height=h)
    if kind == "lbvh":
        return dict(kind=kind, beams=_log_int(rng, 300, 250000))
    if kind == "ppm":
        w, h = _view(rng, 128, 1920)
        return dict(kind=kind, paths=_log_int(rng, 1000, 100000), cells=_log_int(rng, 12, 128),
                    size=_log_int(rng, 48, 256), width=w, height=h)
    if kind == "learned":
        w, h = _view(rng, 128, 1920)
        return dict(kind=kind, spp=_log_int(rng, 1, 32), size=_log_int(rng, 48, 200), width=w, height=h)
    if kind == "collect":
        w, h = _view(rng, 64, 400)
        return dict(kind=kind, frames=rng.randint(1, 8), spp=_log_int(rng, 1, 256), points=_log_int(rng, 500, 20000),
                    size=_log_int(rng, 48, 200), width=w, height=h)
    if kind == "train":
        return dict(kind=kind, steps=_log_int(rng, 1, 100), batch=_log_int(rng, 64, 16384),
                    points=_log_int(rng, 2000, 100000))
    return dict(kind="batch", jobs=rng.randint(2, 16), draw_seed=rng.randint(0, 1 << 20), grid_hi=rng.choice([96, 160]),
                image_hi=rng.choice([192, 320, 512]), spp_hi=rng.choice([32, 64, 128]))


# ------------------------------------------------------------------ prepare

def _sun(seed):
    """A sun above the horizon (light travels downward)."""
    r = np.random.default_rng(seed)
    ct, ph = r.uniform(0.2, 1.0), r.uniform(0.0, 2.0 * math.pi)
    st = math.sqrt(1.0 - ct * ct)
    return (st * math.cos(ph), -ct, st * math.sin(ph))


def _scene(case, seed):
    """The case's cloud as a configs.Scene: the longest axis spans the unit."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    voxel = 1.0 / max(nx, ny, nz)
    shape = S.CR_SHAPE_ANVIL if case["anvil"] else S.CR_SHAPE_CUMULUS
    f = cfg.fbm((nx, ny, nz), voxel, seed=1000 + seed % 100000, octaves=case["octaves"], shape=shape)
    ext = cfg.render_ext(albedo=case["albedo"], bounce_cap=case["bounces"], sky=cfg.SKY, nee=case["nee"],
                         tracking=DDA if case["dda"] else GLOBAL)
    return cfg.Scene("case", f, F16 if case["f16"] else F32, BRICK4 if case["brick4"] else DENSE, 1.0, 64.0,
                     cfg.camera(case["width"], case["height"], position=(0.0, 0.0, case["camera_z"])),
                     cfg.parameters(0.85), ext, case["sv"] or 256, case.get("spp", 1), light_dir=_sun(seed))


def _c1_scene(case, seed, dda):
    """The c1 cloud at the case's sizes, production or reference tracker."""
    n = case["size"]
    return _scene(dict(C1, nx=n, ny=n, nz=n, dda=dda, nee=NEE_RATIO if dda else NEE_SV, width=case["width"],
                       height=case["height"]), seed)


def _frames(n, seed):
    return cfg.frames(n, srand_seed=1 + seed % 100000)


def _prepare_pt(case, seed):
    sc = _scene(case, seed)
    ctx = pkg.Context(0)
    sc.setup(ctx, build_sv=case["nee"] == NEE_SV)
    s = dict(ctx=ctx, frames=_frames(case["spp"], seed), w=sc.width, h=sc.height)
    if case["static"]:
        s["image"] = torch.zeros((sc.height, sc.width, 4), dtype=torch.float32, device="cuda")
        s["array"] = (S.PushConstants * case["spp"])(*s["frames"])
    return s


def _prepare_relight(case, seed):
    sc = _scene(case, seed)
    ctx = pkg.Context(0)
    cloud, _ = sc.setup(ctx)
    return dict(ctx=ctx, cloud=cloud, light=_sun(seed + 7919), sv=case["sv"], frames=_frames(1, seed), w=sc.width,
                h=sc.height)


def _host_cloud(case, seed):
    """A simulation-like density in host memory: noise of several scales under
    a radial envelope, empty outside it."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)
    shape = (case["nz"], case["ny"], case["nx"])
    d = torch.zeros((1, 1) + shape, device="cuda")
    amp = 1.0
    for o in range(5):
        n = [max(2, min(s, (s * (4 << o) + 127) // 128)) for s in shape]
        r = torch.rand((1, 1, *n), device="cuda", generator=g)
        d += amp * torch.nn.functional.interpolate(r, size=shape, mode="trilinear", align_corners=True)
        amp *= 0.5
    ax = [torch.linspace(-1.0, 1.0, s, device="cuda") for s in shape]
    rad = torch.sqrt(ax[0][:, None, None] ** 2 + ax[1][None, :, None] ** 2 + ax[2][None, None, :] ** 2)
    d = ((d[0, 0] / 1.9375) * (1.3 - rad) - 0.35).clamp(0.0, 0.5) * 2.0
    if case["zfast"]:
        d = d.permute(2, 1, 0)
    return d.contiguous().to(torch.float16 if case["src_f16"] else torch.float32).cpu().numpy()


def _prepare_upload(case, seed):
    ctx = pkg.Context(0)
    c = S.CloudProperties()
    ctx.lib.cr_cloud_default(C.byref(c))
    c.baseScaling, c.densityScaling = 1.0, 64.0
    ctx.set_cloud(c)
    ctx.set_grid_layout(BRICK4 if case["brick4"] else DENSE)
    ctx.set_camera(cfg.camera(case["width"], case["height"], position=(0.0, 0.0, -0.2)))
    ctx.set_parameters(cfg.parameters(0.85))
    ctx.set_render_ext(cfg.render_ext(albedo=0.9, bounce_cap=16, sky=cfg.SKY, nee=NEE_SV,
                                      tracking=DDA if case["dda"] else GLOBAL))
    return dict(ctx=ctx, grid=_host_cloud(case, seed), voxel=1.0 / max(case["nx"], case["ny"], case["nz"]),
                layout=S.CR_LAYOUT_Z_FASTEST if case["zfast"] else S.CR_LAYOUT_X_FASTEST,
                storage=F16 if case["f16"] else F32, light=_sun(seed), sv=case["sv"], frames=_frames(1, seed),
                w=case["width"], h=case["height"])


def _prepare_beams(case, seed):
    sc = _c1_scene(case, seed, dda=False)
    ctx = pkg.Context(0)
    cloud, _ = sc.setup(ctx, build_sv=False)
    # camera transmittance of the gather: a shadow volume along the view axis
    ctx.set_shadow_volume(cfg.shadow_volume(cloud, tuple(sc.cam.forward), 256))
    ctx.sv_build()
    ppb = pkg.RenderTechniquePPB(ctx, initialRadius=case["radius"])
    ppb.AllocateResources(cfg.beam_params(case["paths"], seed=38 + seed % 1000, radius=case["radius"], albedo=0.9,
                                          light_dir=sc.light_dir), case["max_beams"])
    return dict(ctx=ctx, ppb=ppb, ext=S.GatherExt(0, 0, 0.9, 0), frame=_frames(1, seed)[0], w=sc.width, h=sc.height)


def _host_beams(case, seed):
    """Beam segments in the unit box: runs of segments along scattered rays."""
    n, r = case["beams"], np.random.default_rng(seed)
    radius = np.float32(0.01)
    runs = -(-n // 16)
    d = r.normal(size=(runs, 3)) + np.array([0.8, -1.2, 0.0])
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    o = r.uniform(0.1, 0.9, (runs, 3)) - np.array([0.5, 0.5, 0.0])
    k = np.arange(16)[None, :, None] * float(radius)
    start = (o[:, None] + d[:, None] * k).reshape(-1, 3)[:n].astype(np.float32)
    end = (o[:, None] + d[:, None] * (k + float(radius))).reshape(-1, 3)[:n].astype(np.float32)
    return start, end, radius


BEAM = np.dtype([("start", "f4", 3), ("morton", "u4"), ("end", "f4", 3), ("radius", "f4"), ("data", "u4"),
                 ("pad", "u4", 3)])
NODE = np.dtype([("parent", "u4"), ("left", "u4"), ("right", "u4"), ("leaf", "u4"), ("bounds", "f4", (2, 4)),
                 ("processed", "u4"), ("pad", "u4", 3)])


def _prepare_lbvh(case, seed):
    ctx = pkg.Context(0)
    sc = _c1_scene(dict(size=32, width=64, height=64), seed, dda=True)
    sc.setup(ctx, build_sv=False)
    start, end, radius = _host_beams(case, seed)
    n = len(start)
    b = np.zeros(n, BEAM)
    b["start"], b["end"], b["radius"], b["data"] = start, end, radius, np.arange(n) // 16
    data = (S.PhotonBeamData * (n // 16 + 1))()
    ctx.upload_beams((S.PhotonBeam * n).from_buffer(b), data)
    return dict(ctx=ctx)


def _prepare_ppm(case, seed):
    sc = _c1_scene(case, seed, dda=False)
    sc.ext = cfg.render_ext(sky=cfg.SKY)
    ctx = pkg.Context(0)
    cloud, _ = sc.setup(ctx)
    pm = S.PhotonMapProperties()
    ctx.lib.cr_photon_map_default(C.byref(pm))
    n = case["cells"]
    pm.voxelCount[:] = (n, n, n)
    ctx.lib.cr_photon_map_set_bounds(C.byref(pm), cloud.bounds[0], cloud.bounds[1])
    pm.stepSize = 0.01
    p = S.PpmParams()
    ctx.lib.cr_ppm_params_default(C.byref(p))
    p.numPaths, p.ambientStep = case["paths"], 0.1
    ppm = pkg.RenderTechniquePPM(ctx, pm, initialRadius=0.01, params=p)
    return dict(ctx=ctx, ppm=ppm, frame=_frames(1, seed)[0], w=sc.width, h=sc.height)


def _set_network(ctx, seed):
    """A network with outputs of a trained one's size (log(1 + radiance))."""
    K, N, wo, bo, total = (C.c_uint32 * 5)(), (C.c_uint32 * 5)(), (C.c_uint32 * 5)(), (C.c_uint32 * 5)(), C.c_uint32()
    ctx.lib.cr_mlp_param_layout(K, N, wo, bo, C.byref(total))
    r = np.random.default_rng(seed)
    p = np.zeros(total.value, np.float32)
    for i in range(5):
        k, n = K[i], (3 if i == 4 else N[i])
        w = np.zeros((K[i], N[i]), np.float32)
        w[:, :n] = r.normal(0.0, math.sqrt(2.0 / k) * (0.2 if i == 4 else 1.0), (k, n))
        p[wo[i]:wo[i] + K[i] * N[i]] = w.ravel()
        p[bo[i]:bo[i] + n] = 0.5 if i == 4 else r.normal(0.0, 0.05, n)
    ctx.check(ctx.lib.cr_mlp_set_params(ctx.h, p.ctypes.data, total.value), "cr_mlp_set_params")
    return total.value


def _prepare_learned(case, seed):
    sc = _c1_scene(case, seed, dda=True)
    ctx = pkg.Context(0)
    sc.setup(ctx, build_sv=False)
    ctx.learn_build_mips()
    _set_network(ctx, seed)
    return dict(ctx=ctx, frames=_frames(case["spp"], seed), w=sc.width, h=sc.height)


def _prepare_collect(case, seed):
    # One cloud and one set of camera paths under another sun: the number of
    # collisions, and so of rows, is the same for every seed.
    sc = _c1_scene(case, 0, dda=True)
    sc.light_dir = _sun(seed)
    ctx = pkg.Context(0)
    sc.setup(ctx, build_sv=False)
    ctx.learn_build_mips()
    return dict(ctx=ctx, frames=_frames(case["frames"], 0), spp=case["spp"], points=case["points"])


def _prepare_train(case, seed):
    ctx = pkg.Context(0)
    sc = _c1_scene(dict(size=64, width=256, height=256), seed, dda=True)
    sc.setup(ctx, build_sv=False)
    ctx.learn_collect(_frames(8, seed), 8, case["points"])
    n = _set_network(ctx, seed)
    return dict(ctx=ctx, steps=case["steps"], batch=case["batch"], seed=3 + seed % 1000, n=n)


def _prepare_batch(case, seed):
    ctx = pkg.Context(0)
    for k, sc in enumerate(cfg.c4(n_jobs=case["jobs"], seed=case["draw_seed"], grid_side=(64, case["grid_hi"]),
                                  image_side=(128, case["image_hi"]), spp=(16, case["spp_hi"]))):
        sc.fbm.seed = 100 + k + 64 * (seed % 100000)
        sc.setup(ctx, build_sv=False)
        ctx.batch_add(_frames(sc.spp, seed + k))
    return dict(ctx=ctx, jobs=case["jobs"])


def prepare(case, seed):
    s = globals()["_prepare_" + case["kind"]](case, int(seed))
    s["kind"] = case["kind"]
    s["ctx"].synchronize()
    return s


# ---------------------------------------------------------------------- run

def _run_pt(s):
    ctx = s["ctx"]
    if "image" in s:
        ctx.check(ctx.lib.cr_pt_render_static(ctx.h, s["array"], len(s["array"]), s["image"].data_ptr()),
                  "cr_pt_render_static")
        return s["image"]
    ctx.pt_render(s["frames"])
    return ctx.download_image(s["h"], s["w"])


def _run_relight(s):
    ctx = s["ctx"]
    ctx.set_shadow_volume(cfg.shadow_volume(s["cloud"], s["light"], s["sv"]))
    ctx.sv_build()
    ctx.pt_render(s["frames"])
    return ctx.download_image(s["h"], s["w"])


def _run_upload(s):
    ctx = s["ctx"]
    ctx.upload_grid(s["grid"], s["voxel"], s["layout"], s["storage"])
    ctx.set_shadow_volume(cfg.shadow_volume(ctx.cloud(), s["light"], s["sv"]))
    ctx.sv_build()
    ctx.pt_render(s["frames"])
    return ctx.download_image(s["h"], s["w"])


def _run_beams(s):
    s["ppb"].RecordDrawCommands(s["frame"], gather_ext=s["ext"])
    return s["ctx"].download_image(s["h"], s["w"])


def _run_lbvh(s):
    ctx = s["ctx"]
    ctx.lbvh_build()
    keys, perm, nodes = ctx.lbvh_download()
    t = np.frombuffer(nodes, NODE)
    links = np.stack([t["parent"], t["left"], t["right"], t["leaf"]]).view(np.int32)
    return {"keys": keys.view(np.int32), "perm": perm.view(np.int32), "links": links, "bounds": t["bounds"][:, :, :3]}


def _run_ppm(s):
    s["ppm"].RecordDrawCommands(s["frame"])
    return s["ctx"].download_image(s["h"], s["w"])


def _run_learned(s):
    s["ctx"].learn_render(s["frames"])
    return s["ctx"].download_image(s["h"], s["w"])


def _run_collect(s):
    ctx = s["ctx"]
    ctx.learn_dataset_clear()
    ctx.learn_collect(s["frames"], s["spp"], s["points"])
    x, t = ctx.learn_dataset()
    return {"features": x.view(np.int16), "targets": t}


def _run_train(s):
    ctx = s["ctx"]
    loss = ctx.learn_train(s["steps"], s["batch"], 1e-3, seed=s["seed"])
    p = np.empty(s["n"], np.float32)
    ctx.check(ctx.lib.cr_mlp_get_params(ctx.h, p.ctypes.data, s["n"]), "cr_mlp_get_params")
    return {"loss": loss, "weights": p}


def _run_batch(s):
    ctx = s["ctx"]
    ctx.batch_render()
    return [ctx.batch_download(j) for j in range(s["jobs"])]


def run(state):
    return globals()["_run_" + state["kind"]](state)


# --------------------------------------------------------------------- work

# Arithmetic one camera path, photon path, march or record cannot do without:
# a trilinear lookup with its coordinates is about 40 operations; a path of
# these clouds makes a dozen lookups and a few bounces (about 1000), a photon
# path with its beams' transmittance samples ten times that.
PATH, PHOTON = 1000.0, 10000.0
ROW = 2.0 * (224 * 128 + 3 * 128 * 128 + 128 * 16)   # network operations of one row, forward
FEATURES = 216 * 40.0


def work(case):
    k = case["kind"]
    px = case.get("width", 0) * case.get("height", 0)
    grid = lambda: case["nx"] * case["ny"] * case["nz"] * (2.0 if case["f16"] else 4.0)  # noqa: E731
    cube = lambda: case["size"] ** 3 * 4.0  # noqa: E731
    if k == "pt":
        return {"bytes": grid() + 4.0 * case["sv"] ** 3 + 16.0 * px, "flops": px * case["spp"] * PATH}
    if k == "relight":
        return {"bytes": grid() + 4.0 * case["sv"] ** 3 + 16.0 * px, "flops": px * PATH + 60.0 * case["sv"] ** 3}
    if k == "upload":
        src = case["nx"] * case["ny"] * case["nz"] * (2.0 if case["src_f16"] else 4.0)
        return {"bytes": src + grid() + 4.0 * case["sv"] ** 3 + 16.0 * px, "flops": px * PATH + 60.0 * case["sv"] ** 3}
    if k == "beams":
        n = min(case["max_beams"], case["paths"] * 200)
        return {"bytes": cube() + n * (48.0 + 80.0 / 50 + 64.0) + 16.0 * px,
                "flops": case["paths"] * PHOTON + px * 10.0 * PATH}
    if k == "lbvh":
        return {"bytes": case["beams"] * (48.0 + 8.0 + 128.0), "flops": case["beams"] * 200.0}
    if k == "ppm":
        return {"bytes": cube() + 4.0 * 256 ** 3 + 16.0 * px + case["paths"] * 5 * 48.0,
                "flops": case["paths"] * PATH + px * 100 * 8 * 40.0}
    if k == "learned":
        rows = px * case["spp"] * 0.2
        return {"bytes": cube() + 16.0 * px, "flops": px * case["spp"] * 0.3 * PATH + rows * (ROW + FEATURES)}
    if k == "collect":
        return {"bytes": cube() + case["points"] * (448.0 + 12.0), "flops": case["points"] * case["spp"] * PATH}
    if k == "train":
        rows = case["steps"] * case["batch"]
        return {"bytes": min(rows, case["points"]) * 460.0 + 320000.0 * 2, "flops": rows * ROW * 3}
    image, grid_side, spp = [(lo + hi) / 2 for lo, hi in ((128, case["image_hi"]), (64, case["grid_hi"]),
                                                          (16, case["spp_hi"]))]
    return {"bytes": case["jobs"] * (2.0 * grid_side ** 3 + 16.0 * image ** 2),
            "flops": case["jobs"] * image ** 2 * spp * 0.6 * PATH}


# -------------------------------------------------------------------- exact

def _clz(v):
    """Leading zeros of 32-bit values (32 for 0)."""
    v = v.astype(np.int64)
    return np.where(v > 0, 31 - np.floor(np.log2(np.maximum(v, 1) + 0.0)).astype(np.int64), 32)


def _exact_lbvh(case, seed):
    """Node boxes in 64 bits: leaf boxes of the capped cylinders in Morton
    order, inner boxes as the union over each Karras node's leaf range."""
    start, end, radius = _host_beams(case, seed)
    n = len(start)
    lo, hi = np.array([-0.5, -0.5, 0.0], np.float32), np.array([0.5, 0.5, 1.0], np.float32)
    q = np.clip(((start + end) / np.float32(2) - lo) / (hi - lo) * np.float32(1024), 0, 1023).astype(np.uint32)
    key = np.zeros(n, np.int64)
    for bit in range(10):
        for a in range(3):
            key |= ((q[:, a].astype(np.int64) >> bit) & 1) << (3 * bit + 2 - a)
    perm = np.argsort(key, kind="stable")
    key = key[perm]
    p, e, r = start[perm].astype(np.float64), end[perm].astype(np.float64), float(radius)
    a = e - p
    ext = r * np.sqrt(np.maximum(0.0, 1.0 - a * a / (a * a).sum(1, keepdims=True)))
    blo, bhi = np.minimum(p, e) - ext, np.maximum(p, e) + ext

    def delta(i, j):
        ok = (j >= 0) & (j < n)
        jj = np.clip(j, 0, n - 1)
        x = key[i] ^ key[jj]
        return np.where(ok, np.where(x == 0, 32 + _clz(i ^ jj), _clz(x)), -1)

    i = np.arange(n - 1)
    d = np.where(delta(i, i + 1) > delta(i, i - 1), 1, -1)
    dmin = delta(i, i - d)
    length = np.zeros(n - 1, np.int64)
    step = 1 << (n - 1).bit_length()
    while step:
        length = np.where(delta(i, i + (length + step) * d) > dmin, length + step, length)
        step >>= 1
    first, last = np.minimum(i, i + length * d), np.maximum(i, i + length * d)
    tlo, thi = [blo], [bhi]   # minima and maxima over runs of 2^k leaves
    while (2 << (len(tlo) - 1)) <= n:
        h = 1 << (len(tlo) - 1)
        tlo.append(np.minimum(tlo[-1][:-h], tlo[-1][h:]))
        thi.append(np.maximum(thi[-1][:-h], thi[-1][h:]))
    ilo, ihi = np.empty((n - 1, 3)), np.empty((n - 1, 3))
    level = np.floor(np.log2(last - first + 1.0)).astype(np.int64)
    for k in np.unique(level):
        m = level == k
        f, l = first[m], last[m] - (1 << k) + 1
        ilo[m], ihi[m] = np.minimum(tlo[k][f], tlo[k][l]), np.maximum(thi[k][f], thi[k][l])
    bounds = np.stack([np.concatenate([ilo, blo]), np.concatenate([ihi, bhi])], axis=1)
    return {"keys": None, "perm": None, "links": None, "bounds": bounds}


def exact(case, seed):
    """Only the LBVH's boxes have a value in 64 bits: the renders, the photon
    maps, the training targets and what is trained on drawn rows are estimates
    whose random walks branch on the 32-bit values themselves."""
    return _exact_lbvh(case, int(seed)) if case["kind"] == "lbvh" else None
