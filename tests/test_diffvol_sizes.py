"""Sizes of the differentiable volume's buffers (host code, no GPU): a
checkpoint buffer sized for the most rays and steps of a program serves every
other call, whatever the grid, as vrx_diffvol_forward takes no size."""
import ctypes as C

import pytest

from visrtx_amd import _native as N

DIMS = [(2, 2, 2), (17, 9, 33), (128, 128, 128), (192, 192, 192), (256, 256, 256), (1024, 512, 512)]


def _vol(dims, max_steps=500, checkpoint=64):
    v = N.vrx_diffvol()
    v.dims[:] = dims
    v.max_steps, v.checkpoint = max_steps, checkpoint
    return v


@pytest.mark.parametrize("n", [1, 65_535, 65_536, 1 << 20, 1 << 23])
@pytest.mark.parametrize("max_steps,checkpoint", [(1, 0), (64, 64), (500, 64), (500, 7)])
def test_checkpoints_do_not_depend_on_the_grid(n, max_steps, checkpoint):
    ck = checkpoint or 64
    want = n * (2 + -(-max_steps // ck) + 8)
    for dims in DIMS:
        v = _vol(dims, max_steps, checkpoint)
        assert N.hip().vrx_diffvol_ckpt_floats(C.byref(v), n) == want, dims


@pytest.mark.parametrize("step", [0.5, 1.0, 0.25])
def test_work_space(step):
    """The y-pair copy: 8 B a voxel where there is a ray for 8 voxels and 36M
    samples along rays that cross the longest side; not for the rays of one or
    two small images, where it only adds a launch."""
    size = N.hip().vrx_diffvol_workspace_bytes
    for dims in DIMS:
        v = _vol(dims)
        m = min(1.0 / (d - 1) for d in dims)
        v.spacing[:] = [1.0 / (d - 1) for d in dims]
        v.step = step * m
        vox = dims[0] * dims[1] * dims[2]
        many = 36e6 * step * m
        for n in (0, 1, 65_536, 131_072, vox // 8, 1 << 18, 1 << 19, 1 << 21, 1 << 24):
            if abs(n - many) < 1e-3 * many:
                continue    # a rounding of the quotient decides
            want = 8 * vox if n >= many and 8 * n >= vox else 0
            assert size(C.byref(v), n) == want, (dims, n)
    v = _vol((64, 64, 64))
    v.spacing[:] = [1 / 63] * 3
    v.step = 0.5 / 63
    assert size(C.byref(v), 2 * 256 * 256) == 0
    assert size(None, 1 << 20) == 0
