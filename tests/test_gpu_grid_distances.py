"""vrx_volume_grid_distances: per macro cell the Chebyshev distance to the
nearest cell whose majorant is above 0 (255 at most), against a brute force;
the majorants stay as they are."""
import ctypes as C

import numpy as np
import pytest

from tests.devmem import DeviceBuffer as DB
from visrtx_amd import _native as N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (16, 17, 33), (200, 40, 90), (4200, 2, 1), (130, 130, 130)])
@pytest.mark.parametrize("share", [0.0, 0.02, 0.5, 1.0])
def test_distances(require_gpu, dims, share):
    m = [(d + 15) // 16 for d in dims]
    rng = np.random.default_rng(1)
    maj = np.where(rng.random(m[::-1]) < share, rng.uniform(0.1, 1.0, m[::-1]), 0.0).astype(np.float32)
    v = N.vrx_volume()
    v.dims[:] = dims
    L = N.hip()
    cells = L.vrx_volume_grid_cells(C.byref(v))
    assert cells == maj.size
    nbytes = L.vrx_volume_grid_bytes(C.byref(v))
    buf = DB.from_array(np.concatenate([maj.reshape(-1).view(np.uint8),
                                        np.full(nbytes - 4 * cells, 7, np.uint8)]))
    print(f"[distances] {dims} {share}", flush=True)
    N.check(L.vrx_volume_grid_distances(C.byref(v), C.c_void_p(buf.addr), None))
    N.check(L.vrx_device_sync())
    out = buf.to_array(np.uint8, 5 * cells)
    np.testing.assert_array_equal(out[:4 * cells].view(np.float32), maj.reshape(-1))
    idx = np.argwhere(maj > 0)
    want = np.full(maj.shape, 255)
    for p in np.ndindex(maj.shape):
        if len(idx):
            want[p] = min(np.abs(idx - np.array(p)).max(1).min(), 255)
    np.testing.assert_array_equal(out[4 * cells:].reshape(maj.shape), want)
