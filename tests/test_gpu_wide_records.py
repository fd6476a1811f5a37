"""The C ABI's frames and batches over each BVH form: BVH2 nodes, the 128-byte
records of vrx_bvh_widen (any wide_format but VRX_WIDE_PACKED) and the packed
ones; AO and directLight on packed nodes also without the ray queues.  The
scenes are opaque, so all forms give the same bits."""
import ctypes as C

import numpy as np
import pytest
import torch

from tests.test_gpu_packed import _prims
from tests.test_gpu_sampled import LIGHTS
from visrtx_amd import _native as N
from visrtx_amd import anari as A
from visrtx_amd import batch as B
from visrtx_amd import scenes as S

pytestmark = pytest.mark.gpu

CAM = S.CameraDesc((0.5, 0.5, -1.2), (0, 0, 1), (0, 1, 0), 0.9, 1.0)
W, H = 75, 50
PACKED_MAGIC = 0x34503634


def _scene(kinds, n, instances):
    geoms = [_prims(k, n, n + i) for i, k in enumerate(kinds)]
    if not instances:
        return S.SceneDesc(geoms=geoms, world_geoms=list(range(len(geoms))), world_id=0,
                           lights=LIGHTS)
    # the cap, cone and curve tests take the ray's direction as a unit vector,
    # as the reference's do: in a scaled instance they report hits off the
    # primitive, and the closest of those depends on the order of the walk
    scale = 0.3 if set(kinds) <= {"sphere", "triangle"} else 1.0
    rng = np.random.default_rng(3)
    insts = []
    for k in range(instances):
        m = np.zeros(12, np.float32)
        m[:9] = (S.random_rotation(rng) * scale).T.reshape(-1)
        m[9:] = rng.random(3)
        insts.append(S.InstanceDesc(geoms=[k % len(geoms)], xfm=m, id=k))
    return S.SceneDesc(geoms=geoms, instances=insts, world_id=0, lights=LIGHTS)


def _widened(scene, keep):
    """A copy of ``scene`` whose d_wide hold vrx_bvh_widen's records."""
    L = N.hip()
    geoms = (N.vrx_geom * scene.num_geoms)()
    size = C.sizeof(geoms)
    N.check(L.vrx_memcpy_sync(C.addressof(geoms), scene.d_geoms, size, N.VRX_D2H))

    def widen(bvh, n):
        buf = torch.empty(max(L.vrx_bvh_wide_bytes(n), 128), dtype=torch.uint8, device="cuda")
        keep.append(buf)
        bvh.d_wide = buf.data_ptr()
        N.check(L.vrx_bvh_widen(C.byref(bvh), n, None), "vrx_bvh_widen")

    for g in geoms:
        widen(g.bvh, g.n)
    out = N.vrx_scene.from_buffer_copy(scene)
    dev = torch.empty(size, dtype=torch.uint8, device="cuda")
    keep.append(dev)
    N.check(L.vrx_memcpy_sync(dev.data_ptr(), C.addressof(geoms), size, N.VRX_H2D))
    out.d_geoms = dev.data_ptr()
    if out.num_entries > 1:
        widen(out.tlas, out.num_entries)
    out.wide_format = 0
    N.check(L.vrx_device_sync())
    return out


def _frame(scene, r, short=0):
    """One frame's channels; ``short``: scratch that much below the query's size."""
    L = N.hip()
    nbytes = L.vrx_render_scratch_bytes(C.byref(scene), C.byref(r), W, H) - short
    scratch = torch.zeros(nbytes, dtype=torch.uint8, device="cuda")
    ch = {k: torch.zeros((H, W) + ((4,) if k in ("accum", "color") else ()), device="cuda",
                         dtype=torch.int32 if k.endswith("id") else torch.float32)
          for k in ("accum", "color", "depth", "prim_id", "obj_id", "inst_id")}
    counters = torch.zeros(64 * 16, dtype=torch.int64, device="cuda")
    f = N.vrx_frame()
    f.width, f.height = W, H
    f.d_accum, f.d_color_f32 = ch["accum"].data_ptr(), ch["color"].data_ptr()
    f.d_depth, f.d_prim_id = ch["depth"].data_ptr(), ch["prim_id"].data_ptr()
    f.d_obj_id, f.d_inst_id = ch["obj_id"].data_ptr(), ch["inst_id"].data_ptr()
    f.d_scratch, f.scratch_bytes = scratch.data_ptr(), nbytes
    f.d_counters = counters.data_ptr()
    cam = B.camera_struct(CAM)
    N.check(L.vrx_render(C.byref(scene), C.byref(cam), C.byref(r), C.byref(f), None), "vrx_render")
    torch.cuda.synchronize()
    assert not scratch[:4].any(), "stack overflow"
    ch["rays"] = counters.view(64, 16)[:, 0].sum()
    return ch


def _same(got, want, what):
    for k, v in want.items():
        assert torch.equal(got[k], v), (what, k)


RENDERERS = [("raycast", {}), ("ao", dict(pixelSamples=3, ambientSamples=2,
                                          ambientOcclusionDistance=0.4)),
             ("directLight", dict(pixelSamples=2, ambientSamples=1, ambientRadiance=0.3))]


@pytest.mark.parametrize("kinds", [("sphere",), ("triangle",), ("cylinder",), ("cone",), ("curve",),
                                   ("sphere", "triangle", "cone")])
@pytest.mark.parametrize("n,instances", [(2, 0), (600, 0), (1, 30), (60, 40)])
def test_forms_give_the_same_frames(require_gpu, kinds, n, instances):
    dev = A.Device()
    s = S.build_anari(dev, _scene(kinds, n, instances))
    packed = B.scene_of(dev, s.world, wide=True)
    assert packed.wide and packed.wide_format == PACKED_MAGIC
    assert (packed.num_entries > 1) == (instances > 0 or len(kinds) > 1)
    keep = []
    wide = _widened(packed, keep)
    one_level = packed.num_entries == 1 and kinds[0] in ("sphere", "triangle", "cylinder")
    for kind, kw in RENDERERS:
        r = B.renderer_of(dev, S.make_renderer(dev, s, kind, **kw))
        for steps in (0, 2) if kind == "raycast" and one_level else (0,):
            r.defer_steps = steps
            print(f"[forms] {kinds} {n} {instances} {kind} long-ray steps {steps}", flush=True)
            r.node_width = 2
            want = _frame(packed, r)
            r.node_width = 4
            _same(_frame(wide, r), want, (kind, steps, "128-byte records"))
            _same(_frame(packed, r), want, (kind, steps, "packed"))
            if kind != "raycast" and packed.single_type in (0, 1, 2):
                # one byte less than the queues need: the per-pixel kernel
                _same(_frame(packed, r, short=1), want, (kind, "without queues"))
        if instances or kind == "raycast":
            r.defer_steps = 0
            out = {}
            for form, sc, width in (("BVH2", packed, 2), ("128-byte records", wide, 4),
                                    ("packed", packed, 4)):
                r.node_width = width
                bf = B.BatchFrame(sc, r, [CAM], W, H)
                bf.render()
                torch.cuda.synchronize()
                out[form] = bf.channels()
            for form in ("128-byte records", "packed"):
                for k, v in out["BVH2"].items():
                    np.testing.assert_array_equal(out[form][k], v, err_msg=f"{kind} {form} {k}")
    assert (want["depth"] < 1e29).any()
    assert not dev.errors(), dev.errors()
    s.release()
    dev.close()
