"""The frame autotuner on worlds that are rebuilt: a choice is kept while the
scene's shape and its frame times stay, and is made again when either changes.
``tunedNodeWidth`` is 0 while the tuner measures."""
import numpy as np
import pytest

from visrtx_amd import anari as A
from visrtx_amd import scenes as S

pytestmark = pytest.mark.gpu


class _World:
    """Spheres whose arrays are replaced between frames.  AO of many samples:
    a frame's kernel takes long against what a host does beside it."""

    def __init__(self, n, radius, renderer="ao", w=640, h=480):
        self.dev = A.Device()
        dev = self.dev
        g = S.GeomDesc("sphere", *self._arrays(n, radius), surface_id=0)
        self.s = S.build_anari(dev, S.SceneDesc(geoms=[g], world_geoms=[0], world_id=0))
        self.geom = self.s.geoms[0]
        cam = S.CameraDesc((0.5, 0.5, -1.2), (0, 0, 1), (0, 1, 0), 0.8, w / h)
        self.c = S.make_camera(dev, self.s, cam)
        kw = dict(pixelSamples=8, ambientOcclusionDistance=0.5) if renderer == "ao" else {}
        r = S.make_renderer(dev, self.s, renderer, **kw)
        self.f = S.make_frame(dev, self.s, self.s.world, self.c, r, w, h)

    @staticmethod
    def _arrays(n, radius):
        return S.gen_spheres(n, seed=5)[0], None, np.full(n, radius, np.float32)

    def rebuild(self, n, radius):
        pos, _, rad = self._arrays(n, radius)
        dev = self.dev
        for name, data, t in (("vertex.position", pos, A.FLOAT32_VEC3),
                              ("vertex.radius", rad, A.FLOAT32)):
            a = dev.array(data, t)
            dev.set(self.geom, name, a, A.ARRAY1D)
            dev.release(a)
        dev.commit(self.geom)

    def frame(self):
        """Renders; (kernel ms, whether the tuner is measuring)."""
        self.dev.commit(self.c)
        self.dev.render(self.f)
        self.dev.ready(self.f)
        return (self.dev.get_property(self.f, "duration", A.FLOAT32) * 1e3,
                self.dev.get_property(self.f, "tunedNodeWidth", A.INT32) == 0)

    def settle(self):
        for _ in range(8):
            if not self.frame()[1]:
                return
        raise AssertionError("the tuner did not settle")

    def close(self):
        assert not self.dev.errors(), self.dev.errors()
        self.s.release()
        self.dev.close()


@pytest.mark.parametrize("n", [(8, 524_288), (100, 6_553_600), (1000, 3000)])
def test_other_primitive_counts_are_measured_again(require_gpu, n):
    print(f"[tune] {n}", flush=True)
    w = _World(n[0], 0.02, "raycast")
    w.settle()
    w.rebuild(n[1], 0.002)
    assert w.frame()[1]
    w.settle()
    w.close()


def test_other_sizes_are_measured_again(require_gpu):
    """A rebuild with another number of entries and another height at once."""
    dev = A.Device()
    g = S.GeomDesc("sphere", *_World._arrays(500, 0.02), surface_id=0)
    insts = []
    for k in range(993):
        m = np.zeros(12, np.float32)
        m[[0, 4, 8]] = 0.05
        m[9:] = (k % 10 / 10, k // 10 % 10 / 10, k // 100 / 10)
        insts.append(S.InstanceDesc(geoms=[0], xfm=m, id=k))
    s = S.build_anari(dev, S.SceneDesc(geoms=[g], instances=insts[:1], world_id=0))
    cam = S.CameraDesc((0.5, 0.5, -1.2), (0, 0, 1), (0, 1, 0), 0.8, 1.0)
    c, r = S.make_camera(dev, s, cam), S.make_renderer(dev, s, "raycast")
    f = S.make_frame(dev, s, s.world, c, r, 640, 480)

    def render():
        dev.commit(c)
        dev.render(f)
        dev.ready(f)
        return dev.get_property(f, "tunedNodeWidth", A.INT32)

    for _ in range(8):
        render()
    assert render()
    x = np.asarray([i.xfm for i in insts], np.float32).reshape(-1, 4, 3)
    m4 = np.zeros((len(x), 4, 4), np.float32)
    m4[:, :, :3], m4[:, 3, 3] = x, 1.0
    grp = s.keep(dev.new("Group"))
    surf = S._surface(dev, s, g)
    dev.set(grp, "surface", s.keep(dev.array([surf], A.SURFACE)), A.ARRAY1D)
    dev.commit(grp)
    ih = s.keep(dev.new("Instance", "transform"))
    dev.set(ih, "group", grp, A.GROUP)
    dev.set(ih, "transform", s.keep(dev.array(m4, A.FLOAT32_MAT4)), A.ARRAY1D)
    dev.commit(ih)
    dev.set(s.world, "instance", s.keep(dev.array([ih], A.INSTANCE)), A.ARRAY1D)
    dev.commit(s.world)
    dev.set(f, "size", (640, 512), A.UINT32_VEC2)
    dev.commit(f)
    assert not render()
    assert not dev.errors(), dev.errors()
    s.release()
    dev.close()


@pytest.mark.parametrize("radii", [(0.0003, 0.05), (0.05, 0.0003)])
def test_other_content_of_the_same_shape_is_measured_again(require_gpu, radii):
    n = 100_000
    w = _World(n, radii[0])
    w.settle()
    before = [w.frame()[0] for _ in range(4)]
    w.rebuild(n, radii[1])
    frames = []
    for _ in range(5):
        frames.append(w.frame())
        w.rebuild(n, radii[1])
    print(f"[tune] {radii}: {before} -> {frames}", flush=True)
    after = np.median([t for t, _ in frames])
    assert not 0.6 < after / np.median(before) < 1.7, "the two contents are too alike"
    assert any(m for _, m in frames[:4])
    for _ in range(8):
        w.frame()
    w.settle()
    w.close()


def test_like_content_keeps_the_choice(require_gpu):
    n = 100_000
    w = _World(n, 0.01)
    w.settle()
    for k in range(12):
        w.rebuild(n, 0.01 + 1e-5 * k)
        ms, measuring = w.frame()
        assert not measuring, (k, ms)
    w.close()


def test_alternating_content_settles(require_gpu):
    """Two contents in turn fit no choice: after some attempts the first
    candidate stays, which has no long-ray pass."""
    n = 20_000
    w = _World(n, 0.0003)
    states = []
    for k in range(100):
        w.rebuild(n, 0.08 if k & 1 else 0.0003)
        states.append(w.frame()[1])
    assert any(states[:12]) and not any(states[-40:])
    assert w.dev.get_property(w.f, "tunedLongRaySteps", A.INT32) == 0
    assert w.dev.get_property(w.f, "tunedStackDepth", A.INT32) == 16
    w.close()


def _instances(renderer, w, h, lights=(), opacity=1.0):
    """300 small instanced spheres: few pixels hit, so the ray queues of AO and
    directLight do not pay."""
    dev = A.Device()
    sc, _ = S.instanced_spheres_workload(300)
    sc.lights, sc.geoms[0].opacity = list(lights), opacity
    s = S.build_anari(dev, sc)
    cam = S.CameraDesc((0.5, 0.5, -1.2), (0, 0, 1), (0, 1, 0), 0.8, w / h)
    c = S.make_camera(dev, s, cam)
    kw = dict(ambientRadiance=0.2, ambientOcclusionDistance=0.5)
    frames = [S.make_frame(dev, s, s.world, c, S.make_renderer(dev, s, renderer, **kw, **k), w, h)
              for k in ({}, dict(nodeWidth=4, stackDepthLDS=16))]

    def render(f):
        dev.commit(c)
        dev.render(f)
        dev.ready(f)
        return dev.get_property(f, "duration", A.FLOAT32) * 1e6

    return dev, s, frames, render


def test_launches_that_do_not_pay_are_left(require_gpu):
    """AO of small instanced spheres: 155 us with ray queues, 130 without, 116
    on BVH2 nodes."""
    dev, s, frames, render = _instances("ao", 1920, 1080)
    us = [[], []]
    for i in range(40):
        for f, t in zip(frames, us):
            t.append(render(f))
    assert not dev.errors(), dev.errors()
    s.release()
    dev.close()
    tuned, queues = (float(np.median(t[12:])) for t in us)
    print(f"[tune] tuned {tuned:.1f} us, with ray queues {queues:.1f}", flush=True)
    assert tuned < 0.9 * queues


@pytest.mark.parametrize("renderer", ["ao", "directLight"])
@pytest.mark.parametrize("opacity", [1.0, 0.4])
def test_all_candidates_of_the_sampled_renderers_give_one_frame(require_gpu, renderer, opacity):
    lights = [S.LightDesc("directional", direction=(0.2, -0.5, 1.0), irradiance=1.2)]
    dev, s, frames, render = _instances(renderer, 203, 150, lights, opacity)
    out = []
    for i in range(8):
        render(frames[0])
        out.append([dev.map_frame(frames[0], "channel." + ch)[0]
                    for ch in ("color", "depth", "primitiveId", "instanceId")])
    width = dev.get_property(frames[0], "tunedNodeWidth", A.INT32)
    assert width in ((2, 4) if opacity == 1.0 else (4,))
    assert not dev.errors(), dev.errors()
    for o in out[1:]:
        for a, b in zip(out[0], o):
            np.testing.assert_array_equal(a, b)
    assert (out[0][1] < 1e29).any()
    s.release()
    dev.close()
