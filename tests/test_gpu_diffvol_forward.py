"""The forward with and without the image hint, on all rays and on parts of
them, and its y-pair gathers.  All sample the same positions in the same order,
so a ray's colour and opacity are bit-identical; the gradients of a loss over
all rays differ by the order of their 32-bit sums."""
import ctypes as C

import numpy as np
import pytest
import torch

from visrtx_amd import _native as N
from visrtx_amd import diffvol as D
from visrtx_amd import scenes as S

pytestmark = pytest.mark.gpu


def _setup(dims, image):
    nx, ny, nz = dims
    sp = tuple(1.0 / (m - 1) for m in dims)
    m = min(sp)
    dens = torch.from_numpy(S.gen_noise_volume(nx, ny, nz, seed=4)).cuda()
    lut = torch.from_numpy(D.colormap_lut(S.COLORMAP5, np.array([0.0, 0.4]))).cuda()
    views = -(-66_000 // (image[0] * image[1]))
    org, dirs = D.make_rays(D.orbit_cameras(views, seed=3, fovy=45.0), *image)
    spec = dict(dims=dims, spacing=sp, unit_distance=m, step=0.5 * m)
    return dens, lut, org, dirs, spec


@pytest.mark.parametrize("dims", [(2, 2, 2), (17, 9, 33), (64, 64, 64), (65, 2, 31)])
@pytest.mark.parametrize("image", [(255, 263), (23, 17), (64, 64)])
def test_layouts_give_the_same_rays(require_gpu, dims, image):
    dens, lut, org, dirs, spec = _setup(dims, image)
    print(f"[forward] {dims} {image} {len(org)} rays", flush=True)
    with torch.no_grad():
        whole = D.render(dens, lut, org, dirs, D.GridSpec(**spec, image=image))
        loose = D.render(dens, lut, org, dirs, D.GridSpec(**spec))
        parts = torch.cat([D.render(dens, lut, o.contiguous(), d.contiguous(), D.GridSpec(**spec))
                           for o, d in zip(org.split(30_011), dirs.split(30_011))])
        # an image size that does not divide the rays is a hint that does not apply
        odd = D.render(dens, lut, org, dirs, D.GridSpec(**spec, image=(image[0] + 1, image[1] + 2)))
    torch.cuda.synchronize()
    for other in (loose, parts, odd):
        assert torch.equal(whole, other)
    assert (whole[:, 3] > 0).any()


def test_gradients_of_many_rays(require_gpu):
    dens, lut, org, dirs, spec = _setup((33, 20, 27), (64, 64))
    up = torch.randn((len(org), 4), device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    got = []
    for n in (len(org), 20_480):
        d, l = dens.clone().requires_grad_(True), lut.clone().requires_grad_(True)
        for o, v, g in zip(org.split(n), dirs.split(n), up.split(n)):
            D.render(d, l, o.contiguous(), v.contiguous(),
                     D.GridSpec(**spec, image=(64, 64))).backward(g.contiguous())
        got.append((d.grad, l.grad))
    for a, b in zip(*got):
        assert float((a - b).norm() / b.norm()) < 2e-5


@pytest.mark.parametrize("dims", [(2, 2, 2), (17, 9, 33), (64, 64, 64), (65, 2, 31)])
def test_work_space_does_not_change_the_rays(require_gpu, dims):
    """The y-pair gathers, with work space, against the density's, with too
    little of it and through the entry point that takes none; the checkpoints
    hold exactly what the size query says."""
    dens, lut, org, dirs, spec = _setup(dims, (255, 263))
    org, dirs = org.repeat(2, 1), dirs.repeat(2, 1)
    spec["step"] = 1 / 512      # 512 samples a ray along the longest side
    s = D.GridSpec(**spec)
    v, n, L = s.struct(dens, lut), len(org), N.hip()
    floats = L.vrx_diffvol_ckpt_floats(C.byref(v), n)
    need = L.vrx_diffvol_workspace_bytes(C.byref(v), n)
    assert need == 8 * dens.numel()
    ws = torch.full((need + 256,), 7, device="cuda", dtype=torch.uint8)
    out = []
    for form, size in (("none", 0), ("short", need - 1), ("whole", need)):
        print(f"[forward] {dims} work space {form}", flush=True)
        rgba = torch.empty((n, 4), device="cuda")
        ck = torch.full((floats + 64,), -7.0, device="cuda")
        args = (C.byref(v), n, org.data_ptr(), dirs.data_ptr(), rgba.data_ptr(), ck.data_ptr())
        if form == "none":
            N.check(L.vrx_diffvol_forward(*args, None))
        else:
            N.check(L.vrx_diffvol_forward_ws(*args, ws.data_ptr(), size, None))
        torch.cuda.synchronize()
        assert (ck[floats:] == -7.0).all() and (ws[need:] == 7).all()
        assert (ws[:need] != 7).any() == (form == "whole")
        out.append((rgba, ck.view(torch.int32)))
    assert (out[0][0][:, 3] > 0).any()
    assert L.vrx_diffvol_forward_ws(*args, ws.data_ptr() + 4, need, None) == -2
    # slots that a ray does not use keep their fill
    for rgba, ck in out[1:]:
        assert torch.equal(rgba, out[0][0]) and torch.equal(ck, out[0][1])


def test_image_hint_does_not_slow_the_forward(require_gpu):
    """The hint is for the backward: pixel tiles made the forward of a large
    grid and few rays 20 to 40 % slower."""
    m = 383
    dens = torch.rand((m + 1,) * 3, device="cuda") * 0.5
    lut = torch.from_numpy(D.colormap_lut(S.COLORMAP5, np.array([0.0, 0.3]))).cuda()
    org, dirs = D.make_rays(D.orbit_cameras(2, seed=3, fovy=45.0), 256, 256)
    kw = dict(dims=(m + 1,) * 3, spacing=(1 / m,) * 3, unit_distance=1 / m, step=0.5 / m)
    specs = [D.GridSpec(**kw), D.GridSpec(**kw, image=(256, 256))]
    us = [[], []]
    with torch.no_grad():
        for i in range(24):
            for spec, t in zip(specs, us):
                a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                a.record()
                for _ in range(4):
                    D.render(dens, lut, org, dirs, spec)
                b.record()
                torch.cuda.synchronize()
                if i >= 4:
                    t.append(a.elapsed_time(b) * 250)
    plain, hint = (float(np.median(t)) for t in us)
    print(f"[forward] 2 views of 256x256, 384^3: {plain:.1f} us, with image {hint:.1f}", flush=True)
    assert hint < 1.1 * plain
