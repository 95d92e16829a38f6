"""The work that a program built on ppmpa_amd has it do, as cases to time.

A case is a dict of plain values; prepare() makes what the program holds
before the call (scene, session, batch, photon set or map), run() makes one
call through the public entry points and returns what it computes, work()
says what that cannot do without, exact() gives 64-bit results where plain
torch can form them.

The kinds:
  render   a session's passes and the mean image (and its variance), from the
           first pass on: a frame, or one step of a program that changes
           scene parameters and renders again.  The image is taken in
           float32, the type the EXR writer stores.
  batch    a few more rounds of many rooms refined together
  fit      a step of recovering albedos from an image: forward render and
           gradients through the autograd pair
  bake     radiance estimates at surface points (a light map's texels) on a
           photon map for any radius
  rt       map build and one eye pass over it (the rt tool)
  pm       one photon pass and its photons in the program's arrays (the pm
           tool)
  classic  one image of the classic ray tracer (the rtc tool)
"""
import ctypes as C
import math
import random

import numpy as np
import torch

import ppmpa_amd as P
from ppmpa_amd import _abi as A
from ppmpa_amd.autograd import Renderer

FILTERS = {"none": A.FILTER_NONE, "cone": A.FILTER_CONE, "gauss": A.FILTER_GAUSS}

_ctx = None


def ctx():
    """The process's one context."""
    global _ctx
    if _ctx is None:
        _ctx = P.Context(0)
    return _ctx


def listed():
    return [
        # an interactive preview: few pixels, few photons, four passes
        dict(name="render_preview", kind="render", scene="caustic", width=160, height=120, photons=20_000, passes=4,
             radius=0.03, depth=10, filter="none", var=False),
        # the two-sphere box's whole schedule
        dict(name="render_box", kind="render", scene="two_spheres", width=256, height=256, photons=200_000, passes=16,
             radius=0.01, depth=8, filter="none", var=True),
        # the production caustic box, part of its schedule
        dict(name="render_caustic", kind="render", scene="caustic", width=1024, height=768, photons=2_000_000,
             passes=64, radius=0.005, depth=16, filter="none", var=False),
        # the same box with the reference's infinite walls, cone filter, odd sizes
        dict(name="render_planes_cone", kind="render", scene="caustic_plane", width=641, height=359, photons=700_001,
             passes=12, radius=0.008, depth=10, filter="cone", var=False),
        # the reference-style room: TS metal and rough glass, Gauss filter, depth of field
        dict(name="render_room_gauss", kind="render", scene="room", width=256, height=256, photons=150_000, passes=8,
             radius=0.05, depth=10, filter="gauss", var=True),
        # the mesh workload at full size
        dict(name="render_mesh", kind="render", scene="mesh7", width=1920, height=1080, photons=8_000_000, passes=4,
             radius=0.005, depth=16, filter="none", var=False),
        # rooms of 2-512 spheres refined together, four rounds at a time
        dict(name="batch_rooms", kind="batch", rooms=24, rounds=4, mix=1, side_min=128, side_max=512,
             photons_min=50_000, photons_max=2_000_000, depth=8),
        # one optimiser step of the inverse workload
        dict(name="fit_step", kind="fit", width=512, height=512, photons=1_000_000, passes=8, radius=0.005, depth=16),
        # a light map: texels of the five walls, row by row
        dict(name="bake_walls", kind="bake", photons=1_000_000, texels=200, radius=0.01, filter="none", refine=False),
        # the rt tool on half a million photons
        dict(name="rt_pass", kind="rt", scene="caustic", width=640, height=480, photons=500_000, radius=0.02, depth=10,
             filter="none"),
        # the pm tool
        dict(name="pm_pass", kind="pm", scene="caustic", photons=1_000_000, depth=10),
        # the rtc tool in a room of 120 spheres
        dict(name="classic_spheres", kind="classic", scene="spheres120", width=800, height=600),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["render", "render", "render", "batch", "fit", "bake", "rt", "pm", "classic"])
    w = _logint(rng, 96, 1280)
    h = max(64, int(w * rng.uniform(0.5, 1.0)))
    if kind == "render":
        scene = rng.choice(["two_spheres", "caustic", "caustic_plane", "room", "mesh%d" % rng.randint(3, 6),
                            "spheres%d" % _logint(rng, 2, 400)])
        n = _logint(rng, 10_000, 2_000_000)
        # the radius shrinks with more photons, as the workloads' do
        r = (0.05 if scene == "room" else 0.01) * math.sqrt(200_000 / n) * rng.uniform(0.7, 1.4)
        return dict(kind="render", scene=scene, width=w, height=h, photons=n, passes=rng.randint(2, 16),
                    radius=min(r, 0.06), depth=rng.randint(6, 16), filter=rng.choice(["none", "none", "cone", "gauss"]),
                    var=rng.random() < 0.5)
    if kind == "batch":
        return dict(kind="batch", rooms=rng.randint(2, 24), rounds=rng.randint(1, 4), mix=rng.randint(1, 1 << 20),
                    side_min=128, side_max=rng.randint(160, 512), photons_min=50_000,
                    photons_max=_logint(rng, 100_000, 2_000_000), depth=8)
    if kind == "fit":
        s = _logint(rng, 96, 512)
        n = _logint(rng, 50_000, 1_000_000)
        return dict(kind="fit", width=s, height=s, photons=n, passes=rng.randint(2, 8),
                    radius=0.005 * math.sqrt(1_000_000 / n), depth=rng.randint(8, 16))
    if kind == "bake":
        n = _logint(rng, 20_000, 1_000_000)
        return dict(kind="bake", photons=n, texels=_logint(rng, 12, 200), radius=0.01 * math.sqrt(1_000_000 / n) *
                    rng.uniform(0.5, 1.0), filter=rng.choice(["none", "cone", "gauss"]), refine=rng.random() < 0.3)
    if kind == "rt":
        n = _logint(rng, 20_000, 500_000)
        return dict(kind="rt", scene=rng.choice(["two_spheres", "caustic", "caustic_plane", "spheres90"]),
                    width=min(w, 640), height=min(h, 480), photons=n, radius=0.02 * math.sqrt(500_000 / n), depth=10,
                    filter=rng.choice(["none", "cone", "gauss"]))
    if kind == "pm":
        return dict(kind="pm", scene=rng.choice(["two_spheres", "caustic", "caustic_plane", "spheres90"]),
                    photons=_logint(rng, 10_000, 1_000_000), depth=10)
    return dict(kind="classic", scene=rng.choice(["caustic", "room", "spheres%d" % _logint(rng, 2, 200)]),
                width=min(w, 800), height=min(h, 600))


# --- inputs ------------------------------------------------------------------

def _spheres_room(k, width, height, rng):
    """A box of random wall albedos with k non-overlapping spheres, each
    diffuse, mirror or glass."""
    sc = P.cornell_box(P.Scene(), left=tuple(rng.uniform(0.1, 0.9, 3)), right=tuple(rng.uniform(0.1, 0.9, 3)),
                       grey=float(rng.uniform(0.4, 0.8)))
    mats = [sc.add_material(P.lambertian(0.75)), sc.add_material(P.mirror()), sc.add_material(P.glass(1.5))]
    rmax = min(0.15, 0.25 * k ** (-1.0 / 3.0))
    at, rad = np.zeros((0, 3)), np.zeros(0)
    for _ in range(k):
        for _try in range(200):
            r = rng.uniform(0.5, 1.0) * rmax
            c = rng.uniform(r + 0.005, 1.0 - r - 0.02, 3)
            if np.all(((at - c) ** 2).sum(1) > (rad + r) ** 2):
                at, rad = np.vstack([at, c]), np.append(rad, r)
                sc.shapes.append(P.sphere(tuple(c), float(r), mats[int(rng.integers(0, 3))]))
                break
    sc.camera = P.pinhole(width, height, (0.5, 0.5, -0.87), (0.5, 0.5, 1.0), 60.0)
    return sc


def _scene(name, width, height, seed):
    rng = np.random.default_rng([seed, 17])
    if name == "two_spheres":
        return P.two_spheres_scene(width, height)
    if name == "caustic":
        return P.caustic_scene(width, height)
    if name == "caustic_plane":
        return P.caustic_scene(width, height, walls="plane")
    if name == "room":
        sc = P.reference_room()
        # the room's own camera at another resolution: the same field of view
        sc.camera.xreso, sc.camera.yreso = width, height
        return sc
    if name.startswith("mesh"):
        return P.mesh_scene(width, height, subdiv=int(name[4:]), seed=1 + seed % 1000)
    return _spheres_room(int(name[7:]), width, height, rng)


def _cfg(case, seed):
    return P.pass_cfg(seed=seed, n_photon=case["photons"], radius0=case["radius"], alpha=2.0 / 3.0,
                      max_depth=case["depth"], pfilter=FILTERS[case.get("filter", "none")])


def _bake_inputs(case, seed):
    """Photons on the five walls of the unit box, a tenth of them in a bright
    spot, and the walls' texel centres with their normals."""
    rng = np.random.default_rng([seed, 5])
    axis = np.array([1, 1, 2, 0, 0])      # floor, ceiling, back, left, right
    side = np.array([0.0, 1.0, 1.0, 0.0, 1.0])
    n = case["photons"]
    f = rng.integers(0, 5, n)
    pos = rng.random((n, 3))
    spot = rng.random(n) < 0.1
    f[spot] = 0
    pos[spot] = 0.5 + 0.08 * rng.standard_normal((int(spot.sum()), 3))
    pos = np.clip(pos, 0.0, 1.0)
    i = np.arange(n)
    pos[i, axis[f]] = side[f]
    inward = np.where(side == 0.0, 1.0, -1.0)
    d = rng.standard_normal((n, 3))
    a = axis[f]
    d[i, a] = -inward[f] * (np.abs(d[i, a]) + 1e-3)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    wl = rng.integers(0, 3, n).astype(np.uint8)
    t = case["texels"]
    uv = (np.stack(np.meshgrid(np.arange(t), np.arange(t), indexing="ij"), -1).reshape(-1, 2) +
          rng.uniform(0.25, 0.75, (t * t, 2))) / t
    q, nrm = [], []
    for w in range(5):
        x, m = np.zeros((t * t, 3)), np.zeros((t * t, 3))
        x[:, [k for k in range(3) if k != axis[w]]] = uv
        x[:, axis[w]] = side[w]
        m[:, axis[w]] = inward[w]
        q.append(x)
        nrm.append(m)
    return pos, d, wl, np.concatenate(q), np.concatenate(nrm)


def prepare(case, seed):
    c, kind = ctx(), case["kind"]
    seed = int(seed) % (1 << 31)
    st = dict(case=case, seed=seed)
    if kind == "render":
        st["scene"] = P.DeviceScene(c, _scene(case["scene"], case["width"], case["height"], seed))
        st["session"] = P.Session(c, st["scene"], _cfg(case, seed))
    elif kind == "batch":
        plan = random.Random(case["mix"])
        rng = np.random.default_rng([seed, 29])
        st["scenes"], cfgs = [], []
        for k in range(case["rooms"]):
            side = plan.randint(case["side_min"], case["side_max"])
            n = _logint(plan, case["photons_min"], case["photons_max"])
            sc = _spheres_room(_logint(plan, 2, 512), side, side, rng)
            st["scenes"].append(P.DeviceScene(c, sc))
            cfgs.append(P.pass_cfg(seed=seed + k, n_photon=n, radius0=0.01 * math.sqrt(200_000 / n), alpha=2.0 / 3.0,
                                   max_depth=case["depth"]))
        # rooms that go on being refined, a few rounds per call, at the launch
        # sizes the batch's tuner mostly settles on
        st["batch"] = P.Batch(c, st["scenes"], cfgs, [1 << 20] * case["rooms"])
        st["batch"].set_launch(eye_waves_per_cu=4, shade_blocks_per_cu=4, tile_width=8)
    elif kind == "fit":
        rng = np.random.default_rng([seed, 41])
        sc = P.inverse_scene(None, case["width"], case["height"], seed=1)
        st["scene"] = P.DeviceScene(c, sc)
        st["render"] = Renderer(c, st["scene"], _cfg(case, seed), case["passes"])
        st["target"] = torch.from_numpy(rng.uniform(0.0, 12.0, (case["height"], case["width"], 3)))
        st["albedo"] = torch.from_numpy(rng.uniform(0.3, 0.7, (32, 3))).requires_grad_()
        st["light"] = torch.tensor(float(rng.uniform(0.8, 1.2)), dtype=torch.float64, requires_grad=True)
    elif kind == "bake":
        pos, d, wl, st["q"], st["n"] = _bake_inputs(case, seed)
        st["photons"] = P.PhotonSet(c, case["photons"])
        st["photons"].upload(pos, d, wl)
        st["map"] = P.build_photonmap(c, st["photons"], 100.0 / case["photons"])
    elif kind == "rt":
        st["scene"] = P.DeviceScene(c, _scene(case["scene"], case["width"], case["height"], seed))
        st["photons"] = P.trace_photons(c, st["scene"], seed, 1, case["photons"], max_depth=case["depth"])
        st["map"] = P.PhotonMap(c, st["photons"].capacity)
    elif kind == "pm":
        st["scene"] = P.DeviceScene(c, _scene(case["scene"], 8, 8, seed))
        st["photons"] = P.trace_photons(c, st["scene"], seed, 2, case["photons"], max_depth=case["depth"])
        # the program's own arrays, with room for three photons stored per
        # photon emitted (rows past the stored ones stay as they are)
        cap = 3 * case["photons"]
        st["pos"], st["dir"] = np.zeros((cap, 3)), np.zeros((cap, 3))
        st["wl"], st["meta"] = np.zeros(cap, np.uint8), np.zeros(cap, np.uint32)
    else:
        st["scene"] = P.DeviceScene(c, _scene(case["scene"], case["width"], case["height"], seed))
    return st


def run(st):
    case, kind, seed = st["case"], st["case"]["kind"], st["seed"]
    c = ctx()
    if kind == "render":
        s = st["session"]
        s.reset()
        s.run(case["passes"])
        mean, var, _ = s.image(with_var=case["var"])
        out = {"mean": mean.astype(np.float32)}
        if case["var"]:
            out["var"] = var.astype(np.float32)
        return out
    if kind == "batch":
        b = st["batch"]
        b.run(case["rounds"])
        return [b.image(k, with_var=False)[0].astype(np.float32) for k in range(case["rooms"])]
    if kind == "fit":
        st["albedo"].grad = st["light"].grad = None
        img = st["render"](st["albedo"], st["light"])
        loss = ((img - st["target"]) ** 2).mean()
        loss.backward()
        return {"image": img.detach().float(), "albedo": st["albedo"].grad, "light": st["light"].grad}
    if kind == "bake":
        return st["map"].estimate_radiance(st["q"], st["n"], case["radius"] ** 2, FILTERS[case["filter"]],
                                           refine64=case["refine"])
    if kind == "rt":
        ph, m = st["photons"], st["map"]
        m.build(ph, ph.power, st["scene"])
        img = P.trace_eye(c, st["scene"], m, seed, 1, case["radius"] ** 2, max_depth=case["depth"],
                          pfilter=FILTERS[case["filter"]])
        return img.astype(np.float32)
    if kind == "pm":
        ph = P.trace_photons(c, st["scene"], seed, 1, case["photons"], max_depth=case["depth"], out=st["photons"])
        n = C.c_uint64()
        c.check(c.lib.ppm_photons_download(c.h, ph.h, len(st["wl"]), st["pos"].ctypes.data_as(A.dp),
                                           st["dir"].ctypes.data_as(A.dp), st["wl"].ctypes.data_as(A.u8p),
                                           st["meta"].ctypes.data_as(A.u32p), C.byref(n)))
        return {"n": n.value, "pos": st["pos"], "dir": st["dir"], "wl": st["wl"], "meta": st["meta"]}
    return P.trace_classic(c, st["scene"], seed, 1, (0.02, 0.02, 0.02)).astype(np.float32)


# --- what a pass cannot do without ---------------------------------------------

def _shapes(name):
    """(shapes tested one by one, shapes that a tree can hold)."""
    if name.startswith("mesh"):
        return 6, 20 * 4 ** int(name[4:]) + 64
    if name.startswith("spheres"):
        k = int(name[7:])
        return (6, k) if k >= 64 else (6 + k, 0)
    return {"two_spheres": (8, 0), "caustic": (9, 0), "caustic_plane": (9, 0), "room": (10, 0)}[name]


def _ray_flops(lin, tree):
    """One ray: about 40 operations per shape tested; a tree of n shapes is
    entered along one path of 2 boxes of 20 operations per level."""
    return 40.0 * lin + (40.0 * math.log2(tree) + 40.0 if tree else 0.0)


def _pass_work(lin, tree, photons, pixels, radius, surface=6.0):
    """One pass: 0.85 photons stored per photon emitted, each of 28 bytes,
    written once and read once; 1.5 queries per pixel, each with 25 shadow
    rays against about a third of a ray's shapes, and the photons of its
    ball (pi r^2 of `surface` square metres) at 20 operations each."""
    ray, s, q = _ray_flops(lin, tree), 0.85 * photons, 1.5 * pixels
    ball = s * min(1.0, math.pi * radius * radius / surface)
    return 56.0 * s, photons * 2.5 * ray + q * ray + q * 25.0 * (ray / 3.0 + 20.0) + q * ball * 20.0


def work(case):
    kind = case["kind"]
    if kind == "batch":
        plan = random.Random(case["mix"])
        b = f = 0.0
        for _ in range(case["rooms"]):
            side = plan.randint(case["side_min"], case["side_max"])
            n = _logint(plan, case["photons_min"], case["photons_max"])
            lin, tree = _shapes("spheres%d" % _logint(plan, 2, 512))
            x, y = _pass_work(lin, tree, n, side * side, 0.01 * math.sqrt(200_000 / n))
            b += case["rounds"] * x + 24.0 * side * side
            f += case["rounds"] * y
        return {"bytes": b, "flops": f}
    if kind == "bake":
        n, q = case["photons"], 5 * case["texels"] ** 2
        ball = n * min(1.0, math.pi * case["radius"] ** 2 / 5.0)
        return {"bytes": 28.0 * n + 72.0 * q, "flops": 20.0 * q * ball}
    if kind == "fit":
        pix = case["width"] * case["height"]
        b, f = _pass_work(40, 0, case["photons"], pix, case["radius"])
        # forward, and the same passes again with their adjoint
        return {"bytes": 2.0 * case["passes"] * b + 48.0 * pix, "flops": 2.0 * case["passes"] * f}
    lin, tree = _shapes(case["scene"])
    scene = 80.0 * (lin + tree)
    if kind == "pm":
        return {"bytes": scene + 0.85 * case["photons"] * 53.0, "flops": 2.5 * case["photons"] * _ray_flops(lin, tree)}
    pix = case["width"] * case["height"]
    if kind == "classic":
        ray = _ray_flops(lin, tree)
        return {"bytes": scene + 24.0 * pix, "flops": 1.5 * pix * (ray + 25.0 * (ray / 3.0 + 20.0))}
    surface = 80.0 if case["scene"] == "room" else 6.0
    b, f = _pass_work(lin, tree, case["photons"], pix, case["radius"], surface)
    if kind == "rt":
        return {"bytes": scene + b + 24.0 * pix, "flops": f - case["photons"] * 2.5 * _ray_flops(lin, tree)}
    return {"bytes": scene + case["passes"] * b + (48.0 if case["var"] else 24.0) * pix, "flops": case["passes"] * f}


# --- 64-bit results --------------------------------------------------------------

def _filter64(name, t):
    """The photon filters as functions of t = d^2 / r^2."""
    if name == "cone":
        d = t.sqrt() / 1.1
        return torch.where(d > 1.0, torch.zeros_like(t), (1.0 - d) / (1.0 - 2.0 / (3.0 * 1.1)))
    if name == "gauss":
        e = 1.0 - torch.exp(-1.953 * t / 2.0)
        eb = 1.0 - 0.14184788965323
        return torch.where(e > eb, torch.zeros_like(t), 0.918 * (1.0 - e / eb) + 0.5)
    return torch.ones_like(t)


def exact(case, seed):
    """The radiance estimates in double, by brute force over the photons whose
    x lies within the radius of a block of queries (sorted by x).  The other
    kinds are Monte Carlo renders with no such form."""
    if case["kind"] != "bake":
        return None
    pos, d, wl, q, nrm = _bake_inputs(case, int(seed) % (1 << 31))
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    order = np.argsort(pos[:, 0], kind="stable")
    pos, d, wl = pos[order], d[order] / np.linalg.norm(d[order], axis=1, keepdims=True), wl[order]
    ps, ds = torch.from_numpy(pos).to(dev), torch.from_numpy(d).to(dev)
    onehot = torch.nn.functional.one_hot(torch.from_numpy(wl.astype(np.int64)), 3).double().to(dev)
    r, r2 = case["radius"], case["radius"] ** 2
    out = torch.zeros((len(q), 3), dtype=torch.float64)
    qo = np.argsort(q[:, 0], kind="stable")
    step = 512
    for b in range(0, len(q), step):
        k = qo[b:b + step]
        lo = np.searchsorted(pos[:, 0], q[k[0], 0] - r - 1e-9)
        hi = np.searchsorted(pos[:, 0], q[k[-1], 0] + r + 1e-9, side="right")
        x, n = torch.from_numpy(q[k]).to(dev), torch.from_numpy(nrm[k]).to(dev)
        got = torch.zeros((len(k), 3), dtype=torch.float64, device=dev)
        for a in range(lo, hi, 32768):
            e = min(hi, a + 32768)
            d2 = (x[:, None, 0] - ps[None, a:e, 0]) ** 2
            d2 += (x[:, None, 1] - ps[None, a:e, 1]) ** 2
            d2 += (x[:, None, 2] - ps[None, a:e, 2]) ** 2
            w = torch.clamp(-(n @ ds[a:e].T), min=0.0) * _filter64(case["filter"], d2 / r2)
            got += torch.where(d2 <= r2, w, torch.zeros_like(w)) @ onehot[a:e]
        out[k] = got.cpu()
    return (out * (100.0 / case["photons"] / (math.pi * r2))).numpy()
