"""Tree construction through the standalone entry points at the sizes where its route changes (one leaf,
one workgroup of 4 or 8 leaves per thread up to 8192, the launches beyond, 4, 8 or 16 keys per thread in
the sort, one or three launches per scan): the sorted keys, the permutation, a well-formed hierarchy and its
boxes, and the queries by brute force."""
import ctypes as C

import numpy as np
import pytest

from luisacomputesimulator_amd import LcsxError, _check, hiprt, load_library
from oracle import morton32

pytestmark = pytest.mark.gpu

INVALID = 0xFFFFFFFF


def read(lib, h, name, count, dtype):
    out = np.zeros(count, dtype=dtype)
    _check(lib.lcsx_lbvh_read(h, name.encode(), out.ctypes.data_as(C.c_void_p), out.nbytes))
    return out


@pytest.mark.parametrize("n", [1, 2, 3, 1023, 1024, 1025, 4096, 4097, 8192, 8193, 65536, 65537, 200001, 294912, 294913])
def test_construct_sizes(require_gpu, n):
    lib = load_library()
    rng = np.random.default_rng(n)
    nv = n + 1
    x = np.cumsum(rng.uniform(-0.01, 0.01, size=(nv, 3)), 0).astype(np.float32)
    x[nv // 2:nv // 2 + 4] = x[nv // 2]  # equal keys: ordered by leaf
    e = np.stack([np.arange(n), np.arange(1, n + 1)], 1).astype(np.uint32)
    dx, de = hiprt.DeviceArray(x.reshape(-1)), hiprt.DeviceArray(e.reshape(-1))
    pad = hiprt.DeviceArray(np.full(nv, 1e-3, dtype=np.float32))
    h = C.c_void_p()
    _check(lib.lcsx_lbvh_create(2, de.ptr, n, C.byref(h)))
    try:
        _check(lib.lcsx_lbvh_construct(h, dx.ptr, nv, None))
        _check(lib.lcsx_lbvh_refit(h, dx.ptr, dx.ptr, pad.ptr, None))
        keys = read(lib, h, "morton_sorted", n, np.uint64)
        order = read(lib, h, "sorted_to_orig", n, np.uint32)
        print(f"[gpu-lbvh] construct {n} leaves", flush=True)
        assert np.all(keys[1:] > keys[:-1])  # by (code, leaf), all distinct
        assert np.array_equal((keys & np.uint64(0xFFFFFFFF)).astype(np.uint32), order)
        assert np.array_equal(np.sort(order), np.arange(n, dtype=np.uint32))
        lo = np.minimum(x[e[:, 0]], x[e[:, 1]])
        hi = np.maximum(x[e[:, 0]], x[e[:, 1]])
        cover = min(n, 256 * ((nv + 255) // 256))
        g0 = lo[:cover].min(0)
        inv = np.float32(1.0) / np.maximum(hi[:cover].max(0) - g0, np.float32(1e-6))
        c = (np.float32(0.5) * (x[e[:, 0]] + x[e[:, 1]]) - g0) * inv
        for k in rng.integers(0, n, size=min(n, 200)):
            o = order[k]
            assert int(keys[k] >> np.uint64(32)) == morton32(*[float(t) for t in c[o]])
        if n > 1:
            parent = read(lib, h, "parent", 2 * n - 1, np.uint32)
            children = read(lib, h, "children", 2 * (2 * n - 1), np.uint32).reshape(-1, 2)
            assert np.count_nonzero(parent == INVALID) == 1 and parent[0] == INVALID
            assert np.array_equal(np.bincount(children[:n - 1].reshape(-1), minlength=2 * n - 1)[1:], np.ones(2 * n - 2))
        boxes = np.concatenate([lo[:32] - np.float32(0.01), hi[:32] + np.float32(0.01)], 1).astype(np.float32)
        m = len(boxes)
        db = hiprt.DeviceArray(boxes.reshape(-1))
        plo, phi = lo - np.float32(1e-3), hi + np.float32(1e-3)
        want = np.argwhere(np.all((plo[None] < boxes[:, None, 3:]) & (phi[None] > boxes[:, None, :3]), 2)).astype(np.uint32)
        dp, dc = hiprt.DeviceArray(np.zeros(2 * (len(want) + 64), dtype=np.uint32)), hiprt.DeviceArray(np.zeros(1, np.uint32))
        _check(lib.lcsx_lbvh_query(h, db.ptr, m, 0, dp.ptr, len(want) + 64, dc.ptr, None))
        got = dp.numpy()[:2 * int(dc.numpy()[0])].reshape(-1, 2)
        assert np.array_equal(got[np.lexsort((got[:, 1], got[:, 0]))], want)
    finally:
        lib.lcsx_lbvh_destroy(h)


def test_order_of_calls(require_gpu):
    """A refit before the construction and a query before the refit are refused: they would walk arrays that
    nothing has written."""
    lib = load_library()
    x = hiprt.DeviceArray(np.arange(12, dtype=np.float32))
    e = hiprt.DeviceArray(np.array([0, 1, 1, 2, 2, 3], dtype=np.uint32))
    pad, box = hiprt.DeviceArray(np.full(4, 1e-3, np.float32)), hiprt.DeviceArray(np.array([0, 0, 0, 9, 9, 9], np.float32))
    pairs, count = hiprt.DeviceArray(np.zeros(16, np.uint32)), hiprt.DeviceArray(np.zeros(1, np.uint32))
    h = C.c_void_p()
    _check(lib.lcsx_lbvh_create(2, e.ptr, 3, C.byref(h)))
    try:
        with pytest.raises(LcsxError, match="refit before construct"):
            _check(lib.lcsx_lbvh_refit(h, x.ptr, x.ptr, pad.ptr, None))
        _check(lib.lcsx_lbvh_construct(h, x.ptr, 4, None))
        with pytest.raises(LcsxError, match="query before refit"):
            _check(lib.lcsx_lbvh_query(h, box.ptr, 1, 0, pairs.ptr, 8, count.ptr, None))
        _check(lib.lcsx_lbvh_refit(h, x.ptr, x.ptr, pad.ptr, None))
        _check(lib.lcsx_lbvh_query(h, box.ptr, 1, 0, pairs.ptr, 8, count.ptr, None))
        assert int(count.numpy()[0]) == 3
    finally:
        lib.lcsx_lbvh_destroy(h)
