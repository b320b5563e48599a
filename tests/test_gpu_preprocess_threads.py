"""icon_preprocess_noalloc called by several threads at once on one device, each
with its own stream and stacks (its scratch array is shared): the results must
be those of icon_preprocess, bit for bit.
"""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_overlapping_noalloc_calls(icon):
    from feilab_amd.icon import DeviceArray
    lib = icon.lib()
    shapes = [(7, 300, 257), (21, 128, 200), (3, 700, 512), (40, 64, 65)]

    def call(fn, d, shape, tilt, stream):
        nz, ny, nx = shape
        modes = np.zeros(nz)
        rc = fn(0, d.ptr, nx, ny, nz, None if tilt is None else tilt.ctypes.data_as(ctypes.c_void_p),
                0 if tilt is None else 200, modes.ctypes.data_as(ctypes.c_void_p), stream)
        assert rc == 0, lib.icon_preprocess_error()
        return d.numpy(), modes

    def worker(k):
        shape, rng = shapes[k], np.random.default_rng(k)
        stream = ctypes.c_void_p()
        assert lib.icon_set_device(0) == 0 and lib.icon_stream_create(ctypes.byref(stream)) == 0
        bad = 0
        for rep in range(12):
            st = rng.gamma(4.0, 30.0, shape).astype(np.float32)
            tilt = np.linspace(-60, 60, shape[0]).astype(np.float32) if rep % 2 else None
            a, ma = call(lib.icon_preprocess, DeviceArray.from_host(st), shape, tilt, stream)
            b, mb = call(lib.icon_preprocess_noalloc, DeviceArray.from_host(st), shape, tilt, stream)
            bad += int(not (np.array_equal(a, b) and np.array_equal(ma, mb)))
        lib.icon_stream_destroy(stream)
        return bad

    print("overlapping noalloc calls", flush=True)
    with ThreadPoolExecutor(len(shapes)) as ex:
        assert list(ex.map(worker, range(len(shapes)))) == [0] * len(shapes)
