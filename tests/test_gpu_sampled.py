"""AO and directLight frames of the wave-at-a-time kernel with its ray queue
(packed nodes) against the per-pixel kernel (BVH2 nodes): the same draws, rays
and sums, so opaque frames are bit-identical.  Translucent ones differ by the
order in which a shadow ray's surfaces are added, a few 1e-7 per surface; 1e-5
allows for the layers.  Sizes: none to more secondary rays per hit than the
queue holds for one pixel (6), frames of partial tiles, accumulation."""
import ctypes as C
import math

import numpy as np
import pytest

from tests.test_gpu_packed import _prims
from tests.test_gpu_render import render_gpu
from visrtx_amd import _native as N
from visrtx_amd import anari as A
from visrtx_amd import batch as B
from visrtx_amd import scenes as S

pytestmark = pytest.mark.gpu

CAM = S.CameraDesc((0.5, 0.5, -1.2), (0, 0, 1), (0, 1, 0), 0.9, 1.0)
LIGHTS = [S.LightDesc("directional", direction=(0.2, -0.5, 1.0), irradiance=1.2),
          S.LightDesc("point", position=(0.2, 1.4, -0.6), intensity=1.5),
          S.LightDesc("spot", position=(0.5, 0.5, -1.0), direction=(0, 0, 1), intensity=2.0,
                      opening_angle=1.0)]


def _scene(kind, n, lights=(), opacity=1.0, instances=0):
    g = _prims(kind, n, n)
    g.opacity = opacity
    if not instances:
        return S.SceneDesc(geoms=[g], world_geoms=[0], world_id=0, lights=list(lights))
    rng = np.random.default_rng(3)
    insts = []
    for k in range(instances):
        m = np.zeros(12, np.float32)
        m[:9] = (S.random_rotation(rng) * 0.3).T.reshape(-1)
        m[9:] = rng.random(3)
        insts.append(S.InstanceDesc(geoms=[0], xfm=m, id=k))
    return S.SceneDesc(geoms=[g], instances=insts, world_id=0, lights=list(lights))


def _compare(sc, w, h, kind, exact=True, **kw):
    a = render_gpu(sc, CAM, w, h, kind, nodeWidth=2, **kw)
    b = render_gpu(sc, CAM, w, h, kind, nodeWidth=4, **kw)
    assert not a["errors"] and not b["errors"]
    for ch in ("depth", "primitiveId", "objectId", "instanceId"):
        np.testing.assert_array_equal(b[ch], a[ch], err_msg=ch)
    if exact:
        np.testing.assert_array_equal(b["color"], a["color"])
    else:
        np.testing.assert_allclose(b["color"], a["color"], rtol=1e-5, atol=1e-5)
    assert a["rays"] == b["rays"]


@pytest.mark.parametrize("aos", [0, 1, 2, 6, 7, 13])
@pytest.mark.parametrize("spp", [1, 3, 8])
def test_ao(require_gpu, aos, spp):
    _compare(_scene("sphere", 500), 75, 50, "ao", pixelSamples=spp, ambientSamples=aos,
             ambientOcclusionDistance=0.4)


@pytest.mark.parametrize("kind", ["sphere", "triangle", "cylinder"])
@pytest.mark.parametrize("lights,aos", [(0, 0), (0, 1), (1, 0), (2, 1), (3, 3), (3, 4), (3, 9)])
def test_direct_light(require_gpu, kind, lights, aos):
    _compare(_scene(kind, 400, LIGHTS[:lights]), 41, 33, "directLight", pixelSamples=3,
             ambientSamples=aos, ambientRadiance=0.3)


@pytest.mark.parametrize("size", [(1, 1), (8, 8), (9, 7), (64, 3)])
def test_partial_tiles(require_gpu, size):
    _compare(_scene("sphere", 3), *size, "ao", pixelSamples=2, ambientSamples=1)


@pytest.mark.parametrize("kind", ["ao", "directLight"])
@pytest.mark.parametrize("opacity", [0.3, 0.98, 0.995])
def test_translucent(require_gpu, kind, opacity):
    _compare(_scene("sphere", 300, LIGHTS[:2], opacity), 48, 40, kind, exact=False,
             pixelSamples=4, ambientSamples=2)


def test_instances(require_gpu):
    sc = _scene("triangle", 60, LIGHTS, instances=40)
    _compare(sc, 64, 64, "ao", pixelSamples=5, ambientSamples=1)
    _compare(sc, 64, 64, "directLight", pixelSamples=2, ambientSamples=1, ambientRadiance=0.2)


def test_accumulation(require_gpu):
    """Frames after the first continue the running sums."""
    out = {}
    for width in (2, 4):
        dev = A.Device()
        s = S.build_anari(dev, _scene("sphere", 400, LIGHTS))
        c = S.make_camera(dev, s, CAM)
        r = S.make_renderer(dev, s, "directLight", nodeWidth=width, pixelSamples=3)
        f = S.make_frame(dev, s, s.world, c, r, 50, 30)
        for i in range(4):
            print(f"[sampled] width {width} frame {i}", flush=True)
            dev.render(f)
            dev.ready(f)
        out[width] = [dev.map_frame(f, "channel." + ch)[0]
                      for ch in ("color", "depth", "primitiveId")]
        assert not dev.errors() and dev.get_property(f, "numSamples", A.INT32) == 9
        s.release()
        dev.close()
    for a, b in zip(out[2], out[4]):
        np.testing.assert_array_equal(a, b)


def test_opacity_above_one(require_gpu):
    """An opacity above 1 does not end a pixel's layers the way 1 does."""
    sc = _scene("sphere", 300, LIGHTS[:1], 1.5)
    assert math.isfinite(sc.geoms[0].opacity)
    _compare(sc, 32, 32, "directLight", exact=False, pixelSamples=2, ambientSamples=1)


def test_queues_are_those_of_the_resident_waves(require_gpu):
    """The frame scratch grows by a queue (16 words a ray, six rays a lane) for
    each wave that can be resident, 20 per compute unit at the kernel's
    registers, or for each wave of a small frame."""
    dev = A.Device()
    s = S.build_anari(dev, _scene("sphere", 100))
    scene = B.scene_of(dev, s.world, wide=True)
    got = {}
    for kind in ("raycast", "ao"):
        r = B.renderer_of(dev, S.make_renderer(dev, s, kind, nodeWidth=4))
        r.defer_steps = 0
        got[kind] = {wh: N.hip().vrx_render_scratch_bytes(C.byref(scene), C.byref(r), *wh)
                     for wh in ((1920, 1080), (64, 48), (1, 1))}
    s.release()
    dev.close()
    cus, queue = C.c_int(), 16 * 4 * 6 * 64
    N.check(N.hip().vrx_device_info(0, None, 0, C.byref(cus), None))
    extra = {wh: got["ao"][wh] - got["raycast"][wh] for wh in got["ao"]}
    print(f"[sampled] queues {extra}, {cus.value} compute units", flush=True)
    for wh, blocks in (((1920, 1080), 5 * cus.value), ((64, 48), 12), ((1, 1), 1)):
        assert 0 < extra[wh] <= 4 * blocks * queue


@pytest.mark.parametrize("size", [(1003, 701), (3001, 17), (8, 20_011), (512, 641)])
def test_more_tiles_than_waves(require_gpu, size):
    """Every tile is rendered once: frames of up to 11,088 tiles (at most 5120
    waves), some of them partial, in rows that are and are not multiples of the
    32 tiles the waves' groups share."""
    sc = _scene("sphere", 40, LIGHTS[:1])
    _compare(sc, *size, "ao", pixelSamples=1, ambientSamples=1)
    _compare(sc, *size, "directLight", pixelSamples=1, ambientSamples=0)


def test_small_scenes_are_not_bound_by_the_tiles(require_gpu):
    """A scene of few primitives at one sample costs little per tile; with one
    counter for all waves its frames took 3 times as long as per-pixel frames
    over BVH2 nodes (0.45 and 0.15 ms), now 1.15 times."""
    w, h = 1920, 1080
    dev = A.Device()
    s = S.build_anari(dev, _scene("sphere", 500))
    c = S.make_camera(dev, s, S.CameraDesc((0.5, 0.5, -1.2), (0, 0, 1), (0, 1, 0), 0.8, w / h))
    frames = [S.make_frame(dev, s, s.world, c, S.make_renderer(dev, s, "ao", nodeWidth=k,
                                                               stackDepthLDS=16), w, h)
              for k in (2, 4)]
    ms = [[], []]
    for i in range(40):
        for f, t in zip(frames, ms):
            dev.commit(c)
            dev.render(f)
            dev.ready(f)
            if i >= 10:
                t.append(dev.get_property(f, "duration", A.FLOAT32) * 1e3)
    assert not dev.errors(), dev.errors()
    s.release()
    dev.close()
    pixel, tiles = (float(np.median(t)) for t in ms)
    print(f"[sampled] per pixel {pixel:.4f} ms, by tiles {tiles:.4f} ms", flush=True)
    assert tiles < 1.5 * pixel
