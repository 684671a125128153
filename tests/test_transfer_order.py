"""The batched transfers' paths -- the kernel on the pinned buffer or copies
through the device's, tiles permuted or copied 16 bytes at a time -- around
the sizes where they change and at rows that no 16 bytes divide, for every
host type: exactly the values of a cast, and the per-field calls' bits."""
import ctypes

import numpy as np
import pytest

from cable_amd.fields import BY_NAME

pytestmark = pytest.mark.gpu

NAMES = ["veg%iveg", "canopy%fe", "ssnow%wb", "rad%albedo"]   # 4 and 8 bytes, 1 to 6 rows


@pytest.mark.parametrize("ordered", [False, True])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("mp", [1, 3, 257, 1300, 1601, 140001])
def test_transfers_over_sizes_and_host_types(mp, precision, ordered):
    from cable_amd import gpu
    print(f"[transfer order] {mp} tiles, precision {precision}, ordered {ordered}", flush=True)
    rng = np.random.default_rng(mp + precision)
    L = gpu.lib()
    g = gpu.CableGPU(mp, precision)
    if ordered:
        g.set_tile_order(rng.permutation(mp))
    ids = np.array([BY_NAME[n].fid for n in NAMES], dtype=np.int32)
    for code, dt in ((gpu.HOST_F64, np.float64), (1, np.float32), (2, np.int32)):
        a = [rng.normal(scale=100.0, size=BY_NAME[n].shape(mp)).astype(dt) for n in NAMES]
        b = [np.empty_like(x) for x in a]
        types = np.full(len(NAMES), code, dtype=np.int32)
        for fn, arrs in ((L.cable_gpu_upload_fields, a), (L.cable_gpu_download_fields, b)):
            ptrs = (ctypes.c_void_p * len(NAMES))(*[x.ctypes.data for x in arrs])
            assert fn(g.h, len(NAMES), ids.ctypes.data, ptrs, types.ctypes.data) == 0
        for n, x, y in zip(NAMES, a, b):
            f = BY_NAME[n]
            dev = (np.where(x < 0, -np.floor(np.abs(x) + 0.5), np.floor(np.abs(x) + 0.5)).astype(np.int32)
                   if f.prec == "I" else x.astype(np.float32 if precision == 1 and f.prec == "F" else np.float64))
            back = (np.where(dev < 0, -np.floor(np.abs(dev) + 0.5), np.floor(np.abs(dev) + 0.5))
                    if dt is np.int32 else dev).astype(dt)
            np.testing.assert_array_equal(y, back, err_msg=f"{n} {dt.__name__}")
            np.testing.assert_array_equal(g.download(n), dev.astype(np.float64), err_msg=f"{n} {dt.__name__}")
    g.close()
