"""The device sort against numpy's stable sort: one workgroup (up to 8 192
keys), whole and partial tiles beyond, look-back over many tiles, digits that
are the same in every key (an odd and an even number of moving passes)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = (2, 65, 8191, 8192, 8193, 16384, 100003, 33 * 8192 + 1, 1000003)


def _keys(kind, n, dtype, rng):
    top = np.iinfo(dtype).max
    if kind == "random":
        return rng.integers(0, top, n, dtype=dtype, endpoint=True)
    if kind == "equal":
        return np.full(n, 0x0102030405060708 & int(top), dtype)
    if kind == "one byte":  # one moving pass: the keys end in the scratch buffer
        return (rng.integers(0, 256, n).astype(dtype) << dtype(8)) | dtype(7)
    if kind == "two bytes":
        return rng.integers(0, 1 << 16, n).astype(dtype)
    return np.sort(rng.integers(0, top, n, dtype=dtype, endpoint=True))[::-1].copy()  # descending


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("kind", ("random", "equal", "one byte", "two bytes", "descending"))
@pytest.mark.parametrize("dtype,with_values", ((np.uint64, True), (np.uint32, True), (np.uint64, False),
                                               (np.uint32, False)))
def test_sort_matches_numpy_stable(gpu, n, kind, dtype, with_values):
    keys = _keys(kind, n, dtype, np.random.default_rng(n))
    vals = np.arange(n, dtype=np.uint32)[::-1].copy()
    s = gpu.Stream()
    dk = gpu.DeviceArray.from_numpy(keys, s)
    dv = gpu.DeviceArray.from_numpy(vals, s)
    bits = 8 * np.dtype(dtype).itemsize
    if with_values:
        gpu.check(getattr(gpu.lib(), f"dy_sort_by_key_u{bits}_u32")(s.h, dk.ptr, dv.ptr, n), "sort")
    else:
        gpu.check(getattr(gpu.lib(), f"dy_sort_u{bits}")(s.h, dk.ptr, n), "sort")
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(dk.download(s), keys[order])
    assert np.array_equal(dv.download(s), vals[order] if with_values else vals)
