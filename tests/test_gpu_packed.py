"""The packed 64-byte 4-wide nodes (vrx_bvh_pack): their grid planes enclose
the exact child boxes, every leaf is reached once, and frames over them equal
the frames over BVH2 nodes bit for bit (the accepted hits are those of exact
boxes), also for axis-parallel rays, far cameras, flat and tiny or huge
scenes, and over the 128-byte nodes of vrx_bvh_widen."""
import ctypes as C
import math

import numpy as np
import pytest

from tests.test_gpu_render import render_gpu
from visrtx_amd import _native as N
from visrtx_amd import anari as A
from visrtx_amd import scenes as S

pytestmark = pytest.mark.gpu

LEAF, EMPTY = 0x80000000, 0xFFFFFFFE
CHANNELS = ("color", "depth", "primitiveId", "objectId", "instanceId")


def _spheres(n, seed, scale=1.0, flat=False, dup=False):
    rng = np.random.default_rng(seed)
    c = rng.random((n, 3)).astype(np.float32)
    if flat:
        c[:, 1] = 0.5
    if dup:
        c[:] = c[rng.integers(0, max(n // 8, 1), n)]
    r = (rng.uniform(0.02, 0.08, n) * (50.0 / max(n, 50)) ** (1 / 3)).astype(np.float32)
    return (c * scale).astype(np.float32), (r * scale).astype(np.float32)


def _walk(nodes, bvh2):
    """(leaf, planes, steps, exact box) of every leaf slot reachable from the
    root, checking inner slots against the BVH2 subtree's box on the way."""
    f = nodes.view(np.float32)
    raw, rawf = bvh2, bvh2.view(np.float32)

    def box2(i):
        b = rawf[i, :12].reshape(2, 6)
        return np.concatenate([b[:, :3].min(0), b[:, 3:].max(0)])

    parent = {}
    for i in range(len(raw)):
        for j in range(2):
            parent[int(raw[i, 12 + j])] = rawf[i, 6 * j:6 * j + 6]
    todo, leaves = [0], []
    while todo:
        i = todo.pop()
        org, step = f[i, 0:3].astype(np.float64), f[i, 3:6].astype(np.float64)
        lo = nodes[i, 6:9].copy().view(np.uint8).reshape(3, 4)
        hi = nodes[i, 9:12].copy().view(np.uint8).reshape(3, 4)
        for c in range(4):
            link = int(nodes[i, 12 + c])
            if link == EMPTY:
                assert c >= 2 and (lo[:, c] == 255).all() and (hi[:, c] == 0).all()
                continue
            exact = (parent[link] if link & LEAF else box2(link)).astype(np.float64)
            assert (org + lo[:, c] * step <= exact[:3] - step / 128).all(), (i, c)
            assert (org + hi[:, c] * step >= exact[3:] + step / 128).all(), (i, c)
            (leaves if link & LEAF else todo).append(link & ~LEAF if link & LEAF else link)
    return leaves


@pytest.mark.parametrize("n", [2, 3, 4, 5, 6, 17, 513, 3000])
@pytest.mark.parametrize("form", ["plain", "flat", "dup", "big", "far"])
def test_planes_enclose_boxes(require_gpu, n, form):
    from tests.devmem import DeviceBuffer as DB
    c, r = _spheres(n, n, scale=1e6 if form == "big" else 1.0, flat=form == "flat",
                    dup=form == "dup")
    if form == "far":
        c += np.float32(3e4)
    L = N.hip()
    sz = N.vrx_bvh_sizes()
    N.check(L.vrx_bvh_query_sizes(N.VRX_SPHERE, C.c_uint32(n), C.byref(sz)))
    dpos, drad = DB.from_array(c), DB.from_array(r)
    bufs = [DB(sz.nodes), DB(sz.leaves), DB(sz.leaf_ids), DB(sz.header),
            DB(L.vrx_bvh_packed_bytes(N.VRX_SPHERE, n))]
    ws = DB(sz.workspace)
    p = N.vrx_prims(N.VRX_SPHERE, n, dpos.addr, None, drad.addr, 0.0)
    b = N.vrx_bvh(*[x.addr for x in bufs])
    print(f"[packed] {form} {n}", flush=True)
    N.check(L.vrx_bvh_build(C.byref(p), C.byref(b), ws.addr, C.c_size_t(sz.workspace), None))
    N.check(L.vrx_bvh_pack(C.byref(b), N.VRX_SPHERE, n, None), "vrx_bvh_pack")
    N.check(L.vrx_device_sync())
    raw = bufs[0].to_array(np.uint32, 16 * (n - 1)).reshape(-1, 16)
    packed = bufs[4].to_array(np.uint32, 16 * (n - 1)).reshape(-1, 16)
    assert sorted(_walk(packed, raw)) == list(range(n))


def _prims(kind, n, seed):
    c, r = _spheres(n, seed)
    if kind == "sphere":
        return S.GeomDesc("sphere", c, radius=r, surface_id=1)
    rng = np.random.default_rng(seed + 1)
    k = 3 if kind == "triangle" else 2
    v = c[:, None, :] + rng.uniform(-0.1, 0.1, (n, k, 3)).astype(np.float32)
    kw = {}
    if kind in ("cone", "curve"):
        kw["radius"] = rng.uniform(0.01, 0.03, n * k).astype(np.float32)
    elif kind == "cylinder":
        kw["global_radius"], kw["caps"] = 0.02, True
    return S.GeomDesc(kind, v.reshape(-1, 3).astype(np.float32), surface_id=1, **kw)


def _equal(sc, cam, w, h, kind="raycast", **kw):
    a = render_gpu(sc, cam, w, h, kind, nodeWidth=2, **kw)
    b = render_gpu(sc, cam, w, h, kind, nodeWidth=4, **kw)
    assert not a["errors"] and not b["errors"]
    for ch in CHANNELS:
        np.testing.assert_array_equal(b[ch], a[ch], err_msg=ch)
    assert a["rays"] == b["rays"]
    return a


@pytest.mark.parametrize("kind", ["sphere", "triangle", "cylinder", "cone", "curve"])
@pytest.mark.parametrize("n", [2, 3, 5, 40, 2000])
def test_frames_equal_bvh2(require_gpu, kind, n):
    sc = S.SceneDesc(geoms=[_prims(kind, n, n)], world_geoms=[0], world_id=0)
    cam = S.CameraDesc((0.5, 0.5, -1.2), (0, 0, 1), (0, 1, 0), 0.9, 1.25)
    _equal(sc, cam, 80, 64)
    _equal(sc, cam, 80, 64, longRaySteps=2)


@pytest.mark.parametrize("form", ["axis", "far", "big", "small", "flat", "grid"])
def test_extreme_views_equal_bvh2(require_gpu, form):
    scale = {"big": 1e6, "small": 1e-5}.get(form, 1.0)
    if form == "grid":   # rays in the planes of the vertices
        v, idx = S.gen_heightfield(33, 3)
        g = S.GeomDesc("triangle", v, idx, surface_id=0)
        cam = S.CameraDesc((0.5, -1.0, 0.9), (0.0, 1.5, -0.9), (0, 0, 1), 0.8, 1.0)
    else:
        c, r = _spheres(3000, 5, scale, flat=form == "flat")
        if form in ("axis", "flat"):
            c = np.round(c * 16) / np.float32(16)
            r[:] = 1 / 32
        g = S.GeomDesc("sphere", c.astype(np.float32), radius=r, surface_id=0)
        m = 0.5 * scale
        cam = S.CameraDesc((m, m, -1.2 * scale), (0, 0, 1), (0, 1, 0), 0.8, 1.0)
        if form == "far":
            cam = S.CameraDesc((0.5, 0.5, -3e4), (0, 0, 1), (0, 1, 0), 5e-5, 1.0)
    sc = S.SceneDesc(geoms=[g], world_geoms=[0], world_id=0)
    out = _equal(sc, cam, 128, 128)
    assert (out["depth"] < 1e29).any()
    # shadow rays along an axis
    sc.lights = [S.LightDesc("directional", direction=(0.0, 0.0, 1.0)),
                 S.LightDesc("directional", direction=(0.0, -1.0, 0.0))]
    _equal(sc, cam, 64, 64, "directLight", pixelSamples=2, ambientRadiance=0.2)


def test_instances_equal_bvh2(require_gpu):
    rng = np.random.default_rng(8)
    geoms = [_prims("sphere", 300, 2), _prims("sphere", 1, 3)]
    insts = []
    for k in range(200):
        m = np.zeros(12, np.float32)
        m[:9] = (S.random_rotation(rng) * rng.uniform(0.05, 0.3)).T.reshape(-1)
        m[9:] = rng.random(3)
        insts.append(S.InstanceDesc(geoms=[k % 2], xfm=m, id=k))
    sc = S.SceneDesc(geoms=geoms, instances=insts, world_id=0)
    cam = S.CameraDesc((0.6, 0.5, -1.2), (0, 0, 1), (0, 1, 0), 0.9, 1.0)
    _equal(sc, cam, 160, 160)
    _equal(sc, cam, 64, 64, "ao", pixelSamples=2, ambientOcclusionDistance=0.4)


def test_wide_records_of_the_c_abi_render_the_same(require_gpu):
    """A scene whose d_wide holds vrx_bvh_widen's 128-byte records (any
    wide_format but VRX_WIDE_PACKED) gives the same batched frame."""
    import torch
    from visrtx_amd import batch as B
    dev = A.Device()
    n = 900
    s = S.build_anari(dev, S.SceneDesc(geoms=[_prims("triangle", n, 4)], world_geoms=[0],
                                       world_id=0))
    r = S.make_renderer(dev, s, "raycast", nodeWidth=4)
    cams = [S.CameraDesc((0.5, 0.5, -1.2), (0, 0, 1), (0, 1, 0), 0.9, 1.0)]
    scene = B.scene_of(dev, s.world, wide=True)
    got = {}
    L = N.hip()
    for form in ("packed", "wide"):
        if form == "wide":
            # vrx_geom: type, n, then the vrx_bvh (five pointers)
            host = torch.empty(512, dtype=torch.uint8)
            size = 8 + C.sizeof(N.vrx_bvh)
            N.check(L.vrx_memcpy_sync(host.data_ptr(), C.c_void_p(scene.d_geoms),
                                      C.c_size_t(size), N.VRX_D2H))
            b = N.vrx_bvh.from_buffer_copy(host.numpy()[8:size].tobytes())
            wide = torch.empty(L.vrx_bvh_wide_bytes(n), dtype=torch.uint8, device="cuda")
            b.d_wide = wide.data_ptr()
            N.check(L.vrx_bvh_widen(C.byref(b), n, None))
            host[8:size] = torch.frombuffer(bytearray(bytes(b)), dtype=torch.uint8)
            N.check(L.vrx_memcpy_sync(C.c_void_p(scene.d_geoms), host.data_ptr(),
                                      C.c_size_t(size), N.VRX_H2D))
            N.check(L.vrx_device_sync())
            assert scene.wide_format != 0
            scene.wide_format = 0
        print("[packed] batched", form, flush=True)
        bf = B.BatchFrame(scene, B.renderer_of(dev, r), cams, 96, 96)
        assert bf.renderer.node_width == 4
        bf.render()
        torch.cuda.synchronize()
        got[form] = bf.channels()
    for ch in CHANNELS:
        np.testing.assert_array_equal(got["wide"][ch], got["packed"][ch], err_msg=ch)
    assert (got["wide"]["depth"] < 1e29).any()
    s.release()
    dev.close()
