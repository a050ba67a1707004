"""GPU: the sample sort of pair lists on lists made for it, called by itself."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "libpairs.so")
TRI_BITS = 24


class Bits(C.Structure):
    _fields_ = [("mesh", C.c_uint32), ("tri", C.c_uint32)]


@pytest.fixture(scope="module")
def lib(ctx):
    if not os.path.exists(LIB):
        from oibvh_amd import facade_build

        facade_build.build()
    lib = C.CDLL(LIB)
    lib.oi_pairs_sort_bytes.restype = C.c_uint64
    lib.oi_pairs_sort_bytes.argtypes = [C.c_uint32]
    lib.oi_launch_pairs_sort.argtypes = [C.c_void_p, C.c_void_p, C.c_uint32, Bits, C.c_void_p, C.c_void_p]
    return lib


def sample_places(n):
    """places of a list of n whose keys the sort samples"""
    S = 8 * min(1024, n // 256)
    i = np.arange(S, dtype=np.uint64)
    lo, hi = i * n // S, (i + 1) * n // S
    w = np.uint64(0xFFFFFFFF)
    h = (i + 1) * np.uint64(2654435769) & w
    h = (h ^ (h >> np.uint64(16))) * np.uint64(2654435769) & w
    h ^= h >> np.uint64(15)
    return (lo + (h * (hi - lo) >> np.uint64(32))).astype(np.int64)


def hits_of(keys):
    """pairs of two meshes in the order of their keys (below 2^48)"""
    keys = keys.astype(np.uint64)
    tri = np.uint64((1 << TRI_BITS) - 1)
    return np.stack([np.zeros_like(keys), np.ones_like(keys), keys >> np.uint64(TRI_BITS), keys & tri],
                    1).astype(np.uint32)


@pytest.mark.parametrize("order", ["missed", "missed_high", "stride", "random", "reversed"])
@pytest.mark.parametrize("n", [4096, 9217, 10240, 33000, 65537, 262144 + 5])
def test_sample_sort_orders_any_list(lib, n, order):
    """Lists of which the sample sees only one end of the keys, so that one bucket
    holds nearly all of them and is sorted in memory (missed); lists that repeat with
    the sample's stride; and plain ones: sorted."""
    from oibvh_amd import api

    print(f"pair sort of {n}, {order}", flush=True)
    r = np.random.default_rng(n)
    if order.startswith("missed"):
        keys = r.permutation(n) + (1 << 40)
        seen = sample_places(n)
        assert len(set(seen)) == len(seen) and seen.min() >= 0 and seen.max() < n
        keys[seen] = r.permutation(len(seen)) + (1 << 41 if order == "missed_high" else 0)
    elif order == "stride":
        i = np.arange(n)
        keys = np.where(i % 32 == 0, i, i + (1 << 40))
    else:
        keys = r.permutation(n) * 977 if order == "random" else np.arange(n)[::-1] * 977
    hits = hits_of(keys)
    src, out = api.DeviceBuffer.from_array(hits), api.DeviceBuffer(hits.nbytes)
    scratch = api.DeviceBuffer(lib.oi_pairs_sort_bytes(n))
    assert lib.oi_launch_pairs_sort(None, src.ptr, n, Bits(1, TRI_BITS), scratch.ptr, out.ptr) == 0
    assert np.array_equal(out.download(np.uint32, 4 * n).reshape(n, 4), hits_of(np.sort(keys)))
