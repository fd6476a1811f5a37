"""What is timed: the calls that programs of this device make.

Each case is one pass through a public entry point: an ANARI frame, a BVH
build or a batched launch of ``include/vrx_hip.h``, or a forward and backward
of ``visrtx_amd.diffvol``.  The listed sizes are those of ``bench.py``, of the
tests and of the example client; ``draw`` gives further ones from the same
ranges, odd and ragged sizes among them.

``exact`` restates the path in 64 bits with torch alone.  It covers the small
sphere frame (every ray against every sphere), the volume frames and the
differentiable volume.  The other scenes have none: every ray against every
primitive takes minutes there, and AO and light samples depend on the
device's own random sequence.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from visrtx_amd import _native as N
from visrtx_amd import anari as A
from visrtx_amd import batch as B
from visrtx_amd import diffvol as D
from visrtx_amd import scenes as S

FOV = math.radians(45.0)
LIGHTS = [S.LightDesc("directional", direction=(0.3, -0.6, 0.8), irradiance=1.5),
          S.LightDesc("point", position=(0.5, 1.5, -0.5), intensity=2.0)]


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: a thumbnail of a small scene, its pixels mapped to
        # the host as ANARI viewers do; launches and synchronisation count
        dict(name="frame_small", kind="spheres", n=20_000, w=96, h=64, renderer="raycast",
             spp=1, aos=0, lights=False, color="f32", host=True),
        # an interactive frame of a mesh (camera moves, scene stays)
        dict(name="frame_heightfield", kind="heightfield", n=257, w=1024, h=768,
             renderer="raycast", spp=1, aos=0, lights=False, color="srgb", rebuild=False),
        # the same mesh deformed each frame: BVH rebuild and frame
        dict(name="frame_deforming", kind="heightfield", n=257, w=1024, h=768,
             renderer="raycast", spp=1, aos=0, lights=False, color="srgb", rebuild=True),
        # particle data, primary rays only
        dict(name="frame_spheres_10m", kind="spheres", n=10_000_000, w=1920, h=1080,
             renderer="raycast", spp=1, aos=0, lights=False, color="srgb", host=False),
        # the same data, final quality with ambient occlusion
        dict(name="frame_ao16_10m", kind="spheres", n=10_000_000, w=1920, h=1080,
             renderer="ao", spp=16, aos=1, lights=False, color="srgb", host=False),
        # lit particles: shadow rays to two lights and one AO ray per sample
        dict(name="frame_lit_1m", kind="spheres", n=1_000_000, w=1920, h=1080,
             renderer="directLight", spp=4, aos=1, lights=True, color="f32", host=False),
        # a million instances of a sphere (glyphs)
        dict(name="frame_instances_1m", kind="instances", n=1_000_000, w=1920, h=1080),
        # a dense scalar field, half-voxel steps
        dict(name="volume_512", kind="volume", nx=512, ny=512, nz=512, w=1920, h=1080,
             rate=1.0, sparse=False),
        # a field that is mostly transparent
        dict(name="volume_sparse_512", kind="volume", nx=512, ny=512, nz=512, w=1920, h=1080,
             rate=1.0, sparse=True),
        # BVH build of streamed particle data
        dict(name="build_spheres_10m", kind="build", prim="sphere", n=10_000_000),
        # many views of an instanced mesh scene (data generation)
        dict(name="batch_64_views", kind="batch", views=64, res=512, instances=256, meshes=16,
             tri_max=2_000_000),
        # one optimisation step of a density grid and its transfer function
        dict(name="diffvol_128", kind="diffvol", nx=128, ny=128, nz=128, views=32, res=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, top=(1920, 1080)):
    w = _log(rng, 64, top[0])
    return w, max(48, min(top[1], int(w * rng.uniform(0.5, 1.0))))


def draw(rng):
    kind = rng.choice(["spheres", "spheres", "heightfield", "heightfield", "instances", "volume",
                       "volume", "build", "build", "batch", "diffvol"])
    if kind in ("spheres", "heightfield"):
        w, h = _size(rng)
        renderer = rng.choice(["raycast", "raycast", "ao", "directLight"])
        c = dict(kind=kind, w=w, h=h, renderer=renderer,
                 spp=1 if renderer == "raycast" else rng.choice([1, 2, 4, 8]),
                 aos=0 if renderer == "raycast" else rng.choice([1, 2]),
                 lights=renderer == "directLight", color=rng.choice(["srgb", "f32"]))
        if kind == "spheres":
            c.update(n=_log(rng, 5_000, 10_000_000), host=w * h < 40_000)
        else:
            c.update(n=_log(rng, 33, 1025), rebuild=rng.random() < 0.4)
        return c
    if kind == "instances":
        w, h = _size(rng)
        return dict(kind=kind, n=_log(rng, 500, 1_000_000), w=w, h=h)
    if kind == "volume":
        w, h = _size(rng)
        return dict(kind=kind, nx=_log(rng, 33, 512), ny=_log(rng, 33, 512),
                    nz=_log(rng, 33, 512), w=w, h=h, rate=rng.choice([0.125, 0.5, 1.0]),
                    sparse=rng.random() < 0.5)
    if kind == "build":
        prim = rng.choice(["sphere", "triangle", "cylinder"])
        return dict(kind=kind, prim=prim, n=_log(rng, 1_000, 10_000_000 if prim == "sphere"
                                                 else 4_000_000))
    if kind == "batch":
        return dict(kind=kind, views=rng.randint(2, 64), res=_log(rng, 48, 512),
                    instances=_log(rng, 4, 256), meshes=rng.randint(1, 16),
                    tri_max=_log(rng, 20_000, 2_000_000))
    return dict(kind=kind, nx=_log(rng, 17, 128), ny=_log(rng, 17, 128), nz=_log(rng, 17, 128),
                views=rng.randint(1, 32), res=_log(rng, 32, 256))


def tolerance(case):
    k = case["kind"]
    if k == "build":
        return "exact"      # topology, boxes and order are integers and copies
    if k == "volume":
        # 32-bit sums over up to 1,800 samples whose transmittances are products
        # of as many factors, hardware exp2 / log2, and the 0.99 cut-off that a
        # rounding moves by one sample: 1e-5 to 4e-5 from the 64-bit image
        return {"rel": 2e-4, "max": 5e-2}
    if k == "diffvol":
        # the cut-off moves a ray's last sample and all that its gradient holds:
        # the image is 6e-5, the gradients 6e-4 to 7e-4 from 64 bits
        return {"rel": 3e-3}
    # surfaces: normals of small spheres at a distance carry 1e-5; identifiers
    # and packed colours are whole numbers and stay the same
    return {"rel": 4e-5}


def work(case):
    k = case["kind"]
    if k in ("spheres", "heightfield", "instances"):
        px = case["w"] * case["h"]
        n, pb = case["n"], 16
        if k == "heightfield":
            n, pb = 2 * (case["n"] - 1) ** 2, 48
        elif k == "instances":
            pb = 112
        spp, aos = case.get("spp", 1), case.get("aos", 0)
        rays = px * spp * (1 + aos + (len(LIGHTS) if case.get("lights") else 0))
        by = px * (16 + (16 if case.get("color") == "f32" else 4)) + min(n, px) * pb
        if case.get("rebuild"):
            by += n * (24 + 48 + 4 + 64)
        # one descent to a leaf: two slab tests a level, one primitive test
        return {"bytes": by, "flops": rays * (math.log2(max(n, 2)) * 24 + 30)}
    if k == "volume":
        px = case["w"] * case["h"]
        vox = case["nx"] * case["ny"] * case["nz"]
        per_ray = 0.27 * max(case["nx"], case["ny"], case["nz"]) * case["rate"]
        if case["sparse"]:
            return {"bytes": 0.03 * vox * 4 + px * 32, "flops": px * per_ray * 0.06 * 40}
        return {"bytes": vox * 4 + px * 32, "flops": px * per_ray * 40}
    if k == "build":
        n = case["n"]
        pin = {"sphere": 16, "triangle": 48, "cylinder": 36}[case["prim"]]
        rec = {"sphere": 16, "triangle": 48, "cylinder": 32}[case["prim"]]
        return {"bytes": n * (pin + rec + 4 + 64), "flops": n * 100}
    if k == "batch":
        px = case["views"] * case["res"] ** 2
        tris = case["meshes"] * 0.3 * case["tri_max"]
        return {"bytes": px * 20 + min(tris, px) * 48,
                "flops": px * (math.log2(tris * case["instances"]) * 24 + 40)}
    rays = case["views"] * case["res"] ** 2
    vox = case["nx"] * case["ny"] * case["nz"]
    per_ray = 0.4 * max(case["nx"], case["ny"], case["nz"])
    return {"bytes": rays * (24 + 16 + 16) + vox * 8, "flops": rays * per_ray * 180}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _spheres(n, seed):
    """n centres in the unit cube, radii log-uniform; radii grow as the count
    falls so that scenes of all sizes cover a similar part of the image."""
    g = _gen(seed)
    c = torch.rand((n, 3), generator=g, device="cuda")
    k = (1e7 / n) ** (1.0 / 3.0)
    u = torch.rand(n, generator=g, device="cuda")
    r = (1e-4 * k) * torch.exp(u * math.log(30.0))
    return c, r.float()


def _noise(nx, ny, nz, seed, octaves=4, freq=4):
    """Fractal value noise in [0, 1], (nz, ny, nx)."""
    g = _gen(seed)
    out = torch.zeros((nz, ny, nx), device="cuda")
    amp, total = 1.0, 0.0
    for o in range(octaves):
        m = (freq << o) + 1
        lat = torch.rand((1, 1, m, m, m), generator=g, device="cuda")
        out += amp * torch.nn.functional.interpolate(lat, size=(nz, ny, nx), mode="trilinear",
                                                     align_corners=True)[0, 0]
        total += amp
        amp *= 0.5
    return (out / total).contiguous()


def _blobs(nx, ny, nz, seed, count=12):
    """A field that is 0 outside ``count`` balls."""
    noise = _noise(nx, ny, nz, seed)
    rng = np.random.default_rng(seed)
    ax = [torch.linspace(0.0, 1.0, m, device="cuda") for m in (nz, ny, nx)]
    data = torch.zeros_like(noise)
    for _ in range(count):
        c, r = rng.uniform(0.15, 0.85, 3), rng.uniform(0.06, 0.14)
        lo = [max(int((c[a] - r) * (m - 1)) - 1, 0) for a, m in enumerate((nz, ny, nx))]
        hi = [min(int((c[a] + r) * (m - 1)) + 2, m) for a, m in enumerate((nz, ny, nx))]
        sl = tuple(slice(a, b) for a, b in zip(lo, hi))
        q = sum(((ax[a][sl[a]] - c[a]) ** 2).reshape([-1 if a == b else 1 for b in range(3)])
                for a in range(3)) / (r * r)
        bump = torch.where(q < 1.0, (1.0 - q) ** 2, torch.zeros_like(q))
        data[sl] = torch.maximum(data[sl], bump * (0.5 + noise[sl]))
    return data


def _nudge(seed, scale=0.05):
    return np.random.default_rng(1000 + seed).uniform(-scale, scale, 3)


def _camera(case, seed):
    """Camera of a case: that of the bench scene, moved a little by the seed."""
    e = _nudge(seed)
    asp = case["w"] / case["h"]
    if case["kind"] == "heightfield":
        p = (0.5 + e[0], -1.5 + e[1], 1.2 + e[2])
        return S.CameraDesc(p, S.look_at(p, (0.5, 0.5, 0.0)), (0, 0, 1), FOV, asp)
    if case["kind"] == "volume":
        p = (1.9 + e[0], 1.5 + e[1], -1.0 + e[2])
        return S.CameraDesc(p, S.look_at(p, (0.5, 0.5, 0.5)), (0, 1, 0), math.radians(35.0), asp)
    p = (0.5 + e[0], 0.5 + e[1], -1.2 + e[2])
    return S.CameraDesc(p, S.look_at(p, (0.5, 0.5, 0.5)), (0, 1, 0), FOV, asp)


def _volume_tf(sparse, sp):
    """(opacity control points, unit distance) of a volume case."""
    if sparse:
        return np.array([0.0, 0.0, 0.4, 0.8], np.float32), 4.0 * sp
    return np.array([0.0, 0.05], np.float32), sp


def _poses(case, seed):
    rng = np.random.default_rng(seed)
    out = []
    for i in range(case["views"]):
        phi = 2.0 * math.pi * (i + rng.uniform(0.0, 0.5)) / case["views"]
        z = rng.uniform(-0.6, 0.6)
        r = math.sqrt(1.0 - z * z)
        out.append((0.5 + 2.0 * r * math.cos(phi), 0.5 + 2.0 * z, 0.5 + 2.0 * r * math.sin(phi)))
    return out


def _rays64(pos, direction, up, fovy, w, h):
    """Pinhole rays through the pixel corners, row 0 at the bottom, in 64 bits."""
    d = np.asarray(direction, np.float64)
    d /= np.linalg.norm(d)
    hh = 2.0 * math.tan(0.5 * fovy)
    du = np.cross(d, np.asarray(up, np.float64))
    du *= hh * (w / h) / np.linalg.norm(du)
    dv = np.cross(du, d)
    dv *= hh / np.linalg.norm(dv)
    t = [torch.tensor(v, device="cuda", dtype=torch.float64)
         for v in (d - 0.5 * du - 0.5 * dv, du, dv)]
    y, x = torch.meshgrid(torch.arange(h, device="cuda", dtype=torch.float64) / h,
                          torch.arange(w, device="cuda", dtype=torch.float64) / w, indexing="ij")
    out = t[0] + x.reshape(-1, 1) * t[1] + y.reshape(-1, 1) * t[2]
    return out / out.norm(dim=1, keepdim=True)


def _diff_inputs(case, seed):
    """Density, colour map and rays of an optimisation step, and the gradient
    of the image that its loss hands back."""
    g = _gen(seed + 77)
    dens = _noise(case["nx"], case["ny"], case["nz"], seed)
    lut = torch.from_numpy(D.colormap_lut(S.COLORMAP5, np.array([0.0, 0.3]))).cuda()
    res = case["res"]
    org, dirs = [], []
    for p in _poses(case, seed):
        d = _rays64(p, np.array([0.5, 0.5, 0.5]) - np.array(p), (0, 1, 0), FOV, res, res)
        dirs.append(d.float())
        org.append(torch.tensor(p, device="cuda", dtype=torch.float32).expand(len(d), 3))
    org, dirs = torch.cat(org).contiguous(), torch.cat(dirs).contiguous()
    up = torch.randn((len(org), 4), generator=g, device="cuda") * (1.0 / len(org))
    return dens, lut, org, dirs, up


def _diff_spec(case):
    sp = tuple(1.0 / (case[k] - 1) for k in ("nx", "ny", "nz"))
    m = min(sp)
    return D.GridSpec(dims=(case["nx"], case["ny"], case["nz"]), spacing=sp, unit_distance=m,
                      step=0.5 * m, early_stop=True, image=(case["res"], case["res"]))


# ---------------------------------------------------------------------------
# the programs
# ---------------------------------------------------------------------------
class _DeviceBuffer:
    """A device pointer handed out by anariMapFrame, as torch reads it.  The
    memory is the frame's, so the buffer keeps the program alive."""

    def __init__(self, app, ptr, shape, typestr):
        self.app = app
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape,
                                         "typestr": typestr, "version": 2}


class _App:
    """One ANARI program: device, scene and frame, and the arrays it shares."""

    def __init__(self):
        self.dev = A.Device()
        self.s = S.AnariScene(self.dev)
        self.shared = []

    def share(self, t, elem):
        self.shared.append(t)
        return self.s.keep(self.dev.shared_array(t.data_ptr(), elem,
                                                 t.shape[0] if t.dim() else 1))

    def surface_world(self, geom, lights):
        dev, s = self.dev, self.s
        dev.commit(geom)
        mat = s.keep(dev.new("Material", "matte"))
        dev.set(mat, "color", (0.8, 0.7, 0.6), A.FLOAT32_VEC3)
        dev.commit(mat)
        surf = s.keep(dev.new("Surface"))
        dev.set(surf, "geometry", geom, A.GEOMETRY)
        dev.set(surf, "material", mat, A.MATERIAL)
        dev.commit(surf)
        self.world = s.keep(dev.new("World"))
        dev.set(self.world, "surface", s.keep(dev.array([surf], A.SURFACE)), A.ARRAY1D)
        if lights:
            hs = [S._light(dev, s, l) for l in LIGHTS]
            dev.set(self.world, "light", s.keep(dev.array(hs, A.LIGHT)), A.ARRAY1D)
        dev.commit(self.world)

    def frame(self, case, cam, kind="raycast", color="srgb", **rp):
        dev, s = self.dev, self.s
        torch.cuda.synchronize()    # shared arrays are filled on torch's stream
        self.w, self.h, self.color = case["w"], case["h"], color
        self.cam = S.make_camera(dev, s, cam)
        self.r = S.make_renderer(dev, s, kind, **rp)
        self.f = S.make_frame(dev, s, self.world, self.cam, self.r, self.w, self.h,
                              color=A.FLOAT32_VEC4 if color == "f32" else A.UFIXED8_RGBA_SRGB)

    def settle(self):
        """Frames until the device has chosen how to launch this frame."""
        for _ in range(12):
            self.render()
            self.dev.ready(self.f)
            if self.dev.get_property(self.f, "tunedNodeWidth", A.INT32):
                break

    def render(self):
        self.dev.commit(self.cam)
        self.dev.render(self.f)

    CHANNELS = ("color", "depth", "primitiveId", "objectId", "instanceId")

    def map_device(self, views):
        """The channels where the device keeps them; ``views`` (of the caller:
        tensors refer to this program) holds those already wrapped."""
        out = {}
        for ch in self.CHANNELS:
            p = self.dev.map_frame_device_ptr(self.f, "channel." + ch)
            v = views.get((ch, p))
            if v is None:
                if ch == "color":
                    f32 = self.color == "f32"
                    shape, ts = (self.h, self.w, 4), "<f4" if f32 else "|u1"
                else:
                    shape, ts = (self.h, self.w), "<f4" if ch == "depth" else "<i4"
                v = torch.as_tensor(_DeviceBuffer(self, p, shape, ts), device="cuda")
                views[(ch, p)] = v
            out[ch] = v
        return out

    def map_host(self):
        # identifiers as signed words, as torch holds them
        out = {ch: self.dev.map_frame(self.f, "channel." + ch)[0] for ch in self.CHANNELS}
        return {k: v.view(np.int32) if v.dtype == np.uint32 else v for k, v in out.items()}

    def __del__(self):
        try:
            torch.cuda.synchronize()
            self.s.release()
            self.dev.close()
        except Exception:
            pass


def prepare(case, seed):
    k = case["kind"]
    if k == "build":
        return _prepare_build(case, seed)
    if k == "batch":
        return _prepare_batch(case, seed)
    if k == "diffvol":
        dens, lut, org, dirs, up = _diff_inputs(case, seed)
        return {"case": case, "spec": _diff_spec(case), "dens": dens.requires_grad_(True),
                "lut": lut.requires_grad_(True), "org": org, "dirs": dirs, "up": up}
    app = _App()
    dev, s = app.dev, app.s
    if k == "instances":
        sc, _ = S.instanced_spheres_workload(case["n"], seed + 21, case["w"], case["h"])
        grow = (1e6 / case["n"]) ** (1.0 / 3.0)
        sc.instances[0].xfm[:, [0, 4, 8]] *= grow
        app.s = S.build_anari(dev, sc)
        app.world = app.s.world
        app.frame(case, _camera(case, seed))
    elif k == "volume":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        data = (_blobs if case["sparse"] else _noise)(nx, ny, nz, seed)
        torch.cuda.synchronize()
        app.shared.append(data)
        arr = s.keep(dev.L.anariNewArray3D(dev.h, C.c_void_p(data.data_ptr()), None, None,
                                           A.FLOAT32, nx, ny, nz))
        sp = [1.0 / (m - 1) for m in (nx, ny, nz)]
        opac, unit = _volume_tf(case["sparse"], min(sp))
        field = s.keep(dev.new("SpatialField", "structuredRegular"))
        dev.set(field, "data", arr, A.ARRAY3D)
        dev.set(field, "spacing", sp, A.FLOAT32_VEC3)
        dev.commit(field)
        vol = s.keep(dev.new("Volume", "transferFunction1D"))
        dev.set(vol, "value", field, A.SPATIAL_FIELD)
        dev.set(vol, "color", s.keep(dev.array(S.COLORMAP5, A.FLOAT32_VEC3)), A.ARRAY1D)
        dev.set(vol, "opacity", s.keep(dev.array(opac, A.FLOAT32)), A.ARRAY1D)
        dev.set(vol, "unitDistance", unit, A.FLOAT32)
        dev.set(vol, "id", 3, A.UINT32)
        dev.commit(vol)
        app.world = s.keep(dev.new("World"))
        dev.set(app.world, "volume", s.keep(dev.array([vol], A.VOLUME)), A.ARRAY1D)
        dev.commit(app.world)
        app.frame(case, _camera(case, seed), color="f32", volumeSamplingRate=case["rate"])
    else:
        if k == "spheres":
            c, r = _spheres(case["n"], seed)
            app.geom = s.keep(dev.new("Geometry", "sphere"))
            dev.set(app.geom, "vertex.position", app.share(c, A.FLOAT32_VEC3), A.ARRAY1D)
            dev.set(app.geom, "vertex.radius", app.share(r, A.FLOAT32), A.ARRAY1D)
        else:
            v, idx = S.gen_heightfield(case["n"], seed + 1)
            v, idx = torch.from_numpy(v).cuda(), torch.from_numpy(idx.view(np.int32)).cuda()
            app.geom = s.keep(dev.new("Geometry", "triangle"))
            dev.set(app.geom, "vertex.position", app.share(v, A.FLOAT32_VEC3), A.ARRAY1D)
            dev.set(app.geom, "primitive.index", app.share(idx, A.UINT32_VEC3), A.ARRAY1D)
        app.surface_world(app.geom, case["lights"])
        rp = {}
        if case["renderer"] != "raycast":
            rp = dict(pixelSamples=case["spp"], ambientSamples=case["aos"],
                      ambientOcclusionDistance=0.5)
            if case["renderer"] == "directLight":
                rp["ambientRadiance"] = 0.3
        app.frame(case, _camera(case, seed), case["renderer"], case["color"], **rp)
    if case.get("rebuild"):
        app.render()
        dev.ready(app.f)
    else:
        app.settle()
    errs = dev.errors()
    if errs:
        raise RuntimeError(str(errs))
    return {"case": case, "app": app, "views": {}}


def _prepare_build(case, seed):
    L = N.hip()
    n, prim = case["n"], case["prim"]
    g = _gen(seed)
    p = N.vrx_prims()
    keep = []
    if prim == "sphere":
        c, r = _spheres(n, seed)
        keep += [c, r]
        p.type, p.n, p.d_position, p.d_radius = N.VRX_SPHERE, n, c.data_ptr(), r.data_ptr()
    elif prim == "triangle":
        c = torch.rand((n, 1, 3), generator=g, device="cuda")
        e = (torch.rand((n, 3, 3), generator=g, device="cuda") - 0.5) * (0.5 / n ** (1.0 / 3.0))
        v = (c + e).reshape(-1, 3).contiguous()
        idx = torch.arange(3 * n, device="cuda", dtype=torch.int32).reshape(n, 3)
        keep += [v, idx]
        p.type, p.n, p.d_position, p.d_index = N.VRX_TRIANGLE, n, v.data_ptr(), idx.data_ptr()
    else:
        c = torch.rand((n, 1, 3), generator=g, device="cuda")
        e = (torch.rand((n, 2, 3), generator=g, device="cuda") - 0.5) * (1.0 / n ** (1.0 / 3.0))
        v = (c + e).reshape(-1, 3).contiguous()
        idx = torch.arange(2 * n, device="cuda", dtype=torch.int32).reshape(n, 2)
        keep += [v, idx]
        p.type, p.n, p.d_position, p.d_index = N.VRX_CYLINDER, n, v.data_ptr(), idx.data_ptr()
        p.global_radius = 0.1 / n ** (1.0 / 3.0)
    sz = N.vrx_bvh_sizes()
    N.check(L.vrx_bvh_query_sizes(p.type, n, C.byref(sz)))
    buf = {k: torch.zeros(getattr(sz, k) // 4, device="cuda", dtype=torch.int32)
           for k in ("nodes", "leaves", "leaf_ids", "header")}
    ws = torch.empty(sz.workspace, device="cuda", dtype=torch.uint8)
    b = N.vrx_bvh()
    b.d_nodes, b.d_leaves = buf["nodes"].data_ptr(), buf["leaves"].data_ptr()
    b.d_leaf_ids, b.d_header = buf["leaf_ids"].data_ptr(), buf["header"].data_ptr()
    return {"case": case, "keep": keep, "prims": p, "bvh": b, "buf": buf, "ws": ws}


def _prepare_batch(case, seed):
    app = _App()
    sc, cams = S.batched_workload(case["views"], case["res"], case["instances"], case["meshes"],
                                  tri_max=case["tri_max"], seed=9 + seed)
    app.s = S.build_anari(app.dev, sc)
    r = S.make_renderer(app.dev, app.s, "raycast")
    scene = B.scene_of(app.dev, app.s.world, wide=True)
    bf = B.BatchFrame(scene, B.renderer_of(app.dev, r), cams, case["res"], case["res"], srgb=True)
    return {"case": case, "app": app, "bf": bf}


def run(state):
    case = state["case"]
    k = case["kind"]
    if k == "build":
        ws = state["ws"]
        N.check(N.hip().vrx_bvh_build(C.byref(state["prims"]), C.byref(state["bvh"]),
                                      ws.data_ptr(), ws.numel(),
                                      torch.cuda.current_stream().cuda_stream), "vrx_bvh_build")
        return state["buf"]
    if k == "batch":
        bf = state["bf"]
        bf.render()
        return {"color": bf.color.view(torch.uint8), "depth": bf.depth,
                "primitiveId": bf.prim_id, "objectId": bf.obj_id, "instanceId": bf.inst_id}
    if k == "diffvol":
        dens, lut = state["dens"], state["lut"]
        dens.grad = lut.grad = None
        rgba = D.render(dens, lut, state["org"], state["dirs"], state["spec"])
        rgba.backward(state["up"])
        return {"rgba": rgba.detach(), "grad_density": dens.grad, "grad_lut": lut.grad}
    app = state["app"]
    if case.get("rebuild"):
        app.dev.commit(app.geom)    # the vertices changed
    app.render()
    app.dev.ready(app.f)
    return app.map_host() if case.get("host") else app.map_device(state["views"])


# ---------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------
def exact(case, seed):
    k = case["kind"]
    if k == "spheres" and case["renderer"] == "raycast" and case["color"] == "f32" \
            and case["n"] * case["w"] * case["h"] <= 200_000_000:
        return _exact_spheres(case, seed)
    if k == "volume":
        return _exact_volume(case, seed)
    if k == "diffvol":
        return _exact_diffvol(case, seed)
    return None


def _exact_spheres(case, seed):
    c, r = _spheres(case["n"], seed)
    c, r = c.double(), r.double()
    cam = _camera(case, seed)
    w, h = case["w"], case["h"]
    o = torch.tensor(np.asarray(cam.position, np.float32), device="cuda").double()
    d = _rays64(cam.position, cam.direction, cam.up, cam.fovy, w, h)
    co = c - o
    t = torch.empty(len(d), device="cuda", dtype=torch.float64)
    who = torch.empty(len(d), device="cuda", dtype=torch.long)
    for a in range(0, len(d), 512):
        dd = d[a:a + 512]
        pj = dd @ co.T
        disc = r * r - ((co * co).sum(1) - pj * pj)
        tt = torch.where((disc >= 0) & (pj - disc.clamp(min=0).sqrt() >= 0),
                         pj - disc.clamp(min=0).sqrt(), torch.inf)
        t[a:a + 512], who[a:a + 512] = tt.min(1)
    hit = torch.isfinite(t)
    p = o + torch.where(hit, t, 0.0)[:, None] * d
    nrm = p - c[who]
    nrm = nrm / nrm.norm(dim=1, keepdim=True)
    base = torch.tensor([0.8, 0.7, 0.6], dtype=torch.float32, device="cuda").double()
    col = torch.zeros((len(d), 4), device="cuda", dtype=torch.float64)
    col[:, :3] = torch.where(hit[:, None], (nrm * d).sum(1).abs()[:, None] * base, 0.0)
    col[:, 3] = 1.0
    depth = torch.where(hit, t, 1e30)
    out = {ch: None for ch in _App.CHANNELS}
    out["color"] = col.reshape(h, w, 4).cpu().numpy()
    out["depth"] = depth.reshape(h, w).cpu().numpy()
    return out


def _lut64(colors, opacities):
    p = np.arange(256) / 255.0
    lut = np.empty((256, 4))
    for k in range(3):
        lut[:, k] = np.interp(p, np.linspace(0, 1, len(colors)), colors[:, k].astype(np.float64))
    lut[:, 3] = np.interp(p, np.linspace(0, 1, len(opacities)), opacities.astype(np.float64))
    return torch.from_numpy(lut).cuda()


class _Field64:
    """Trilinear samples of a field on the unit cube in 64 bits, and rays."""

    def __init__(self, data, lut):
        self.data, self.lut = data.reshape(-1), lut
        nz, ny, nx = data.shape
        self.dims = torch.tensor([nx, ny, nz], device="cuda")
        self.stride = torch.tensor([1, nx, nx * ny], device="cuda")
        self.sp = 1.0 / (self.dims.double() - 1.0)

    def interval(self, o, d):
        a, b = (0.0 - o) / d, (1.0 - o) / d
        t0 = torch.minimum(a, b).amax(1).clamp(min=0.0)
        return t0, torch.maximum(a, b).amin(1)

    def cell(self, p):
        g = torch.minimum((p / self.sp).clamp(min=0.0), self.dims - 1.0)
        i = torch.minimum(g.long(), self.dims - 2)
        return (i * self.stride).sum(1), g - i

    def corners(self, f):
        for q in range(8):
            w = 1.0
            off = 0
            for a in range(3):
                bit = (q >> a) & 1
                w = w * (f[:, a] if bit else 1.0 - f[:, a])
                off = off + bit * int(self.stride[a])
            yield off, w

    def value(self, base, f):
        return sum(w * self.data[base + off].double() for off, w in self.corners(f))

    def classify(self, s):
        xr = s * 256.0 - 0.5
        x = xr.clamp(0.0, 255.0)
        i = x.long().clamp(max=254)
        f = (x - i)[:, None]
        a, b = self.lut[i], self.lut[i + 1]
        return a + (b - a) * f, b - a, i, f[:, 0], (s > 0) & (s < 1) & (xr > 0) & (xr < 255)


def _exact_volume(case, seed):
    nx, ny, nz, w, h = (case[k] for k in ("nx", "ny", "nz", "w", "h"))
    sp = [1.0 / (m - 1) for m in (nx, ny, nz)]
    opac, unit = _volume_tf(case["sparse"], min(sp))
    fld = _Field64((_blobs if case["sparse"] else _noise)(nx, ny, nz, seed),
                   _lut64(S.COLORMAP5, opac))
    cam = _camera(case, seed)
    d = _rays64(cam.position, cam.direction, cam.up, cam.fovy, w, h)
    o = torch.tensor(np.asarray(cam.position, np.float32), device="cuda").double()
    t0, t1 = fld.interval(o, d)
    step = 0.5 * min(sp) / case["rate"]
    depth = torch.where(t0 < t1, t0, 1e30)
    acc = torch.zeros((len(d), 4), device="cuda", dtype=torch.float64)
    live = (t0 < t1).nonzero()[:, 0]
    T = torch.ones(len(live), device="cuda", dtype=torch.float64)
    dl, tl, te, al = d[live], t0[live], t1[live], acc[live]
    k = 0
    while len(live):
        t = tl + k * step
        ok = (t <= te) & (al[:, 3] < 0.99)
        if k % 16 == 0 or k < 2:
            acc[live[~ok]] = al[~ok]
            live, T, dl, tl, te, al, t = (v[ok] for v in (live, T, dl, tl, te, al, t))
            ok = ok[ok]
            if not len(live):
                break
        co = fld.classify(fld.value(*fld.cell(o + t[:, None] * dl)))[0]
        tau = (1.0 - co[:, 3]) ** (step / unit)
        wt = torch.where(ok, T * (1.0 - tau), 0.0)
        al[:, :3] += wt[:, None] * co[:, :3]
        al[:, 3] += wt
        T = torch.where(ok, T * tau, T)
        k += 1
    # the renderer multiplies colour by opacity, then adds the black background
    col = torch.cat([acc[:, :3] * acc[:, 3:], torch.ones_like(acc[:, 3:])], 1)
    out = {ch: None for ch in _App.CHANNELS}
    out["color"], out["depth"] = col.reshape(h, w, 4), depth.reshape(h, w)
    return out


def _exact_diffvol(case, seed):
    dens, lut, org, dirs, up = _diff_inputs(case, seed)
    fld = _Field64(dens, lut.double())
    o, d, G = org.double(), dirs.double(), up.double()
    m = min(1.0 / (case[k] - 1) for k in ("nx", "ny", "nz"))
    step, expo = 0.5 * m, 0.5
    t0, t1 = fld.interval(o, d)
    n = len(o)
    rgba = torch.zeros((n, 4), device="cuda", dtype=torch.float64)
    tot = torch.zeros(n, device="cuda", dtype=torch.float64)
    gd = torch.zeros(dens.numel(), device="cuda", dtype=torch.float64)
    gl = torch.zeros((256, 4), device="cuda", dtype=torch.float64)
    for back in (False, True):
        live = (t0 < t1).nonzero()[:, 0]
        T = torch.ones(len(live), device="cuda", dtype=torch.float64)
        O = torch.zeros_like(T)
        suf = tot[live].clone()
        k = 0
        while True:
            t = t0[live] + k * step
            ok = (t <= t1[live]) & (O < 0.99)
            live, T, O, suf, t = (v[ok] for v in (live, T, O, suf, t))
            if not len(live):
                break
            base, f = fld.cell(o[live] + t[:, None] * d[live])
            co, slope, i, lf, inside = fld.classify(fld.value(base, f))
            tau = (1.0 - co[:, 3]) ** expo
            wt = T * (1.0 - tau)
            g = G[live]
            v = (g[:, :3] * co[:, :3]).sum(1) + g[:, 3]
            if not back:
                rgba[live, :3] += wt[:, None] * co[:, :3]
                rgba[live, 3] += wt
                tot[live] += wt * v
            else:
                suf = suf - wt * v
                da = (suf - T * tau * v) * (-expo) / (1.0 - co[:, 3])
                dc = torch.cat([wt[:, None] * g[:, :3], da[:, None]], 1)
                for c in range(4):
                    gl[:, c] += torch.bincount(i, dc[:, c] * (1.0 - lf), 256)
                    gl[:, c] += torch.bincount(i + 1, dc[:, c] * lf, 256)
                ds = (dc * slope).sum(1) * 256.0 * inside
                for off, wc in fld.corners(f):
                    gd.index_add_(0, base + off, ds * wc)
            O = O + wt
            T = T * tau
            k += 1
    return {"rgba": rgba, "grad_density": gd.reshape(dens.shape), "grad_lut": gl}
