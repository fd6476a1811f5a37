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


def test_work_space():
    size = N.hip().vrx_diffvol_workspace_bytes
    for dims in DIMS:
        v = _vol(dims)
        vox = dims[0] * dims[1] * dims[2]
        for n in (0, 1, 65_535, 65_536, vox // 8 - 1, vox // 8, vox // 8 + 1, 1 << 24):
            n = max(n, 0)
            want = 8 * vox if n >= 65_536 and 8 * n >= vox else 0
            assert size(C.byref(v), n) == want, (dims, n)
    assert size(None, 1 << 20) == 0
