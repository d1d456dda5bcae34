"""DeviceRadixSort of small inputs (one workgroup, or LDS-sorted runs merged by rank) vs the oracle: the sizes
around a wave, a run of 1,024, the one-workgroup line at 2,048 and the last size of the path (152 KB of
keys), bit-exact with index values so that stability shows."""
import numpy as np
import pytest

from gpu_util import empty_dev, log, to_dev, to_host
from test_gpu_radix_sort import SUFFIX, check_bits, gpu_sort

pytestmark = pytest.mark.gpu

LAST = {4: 38912, 8: 19456}


def make_keys(orc, dtype, n, seed, kind):
    raw = orc.generate(0, n, seed)
    dtype = np.dtype(dtype)
    if kind == "few":  # long runs of equal keys, across runs and tiles
        raw = raw % np.uint64(5) * np.uint64(0x0101010101010101)
    if kind == "low":  # every digit but the lowest the same
        raw = raw & np.uint64(0xFF00000000)
    keys = (raw if dtype.itemsize == 8 else (raw >> np.uint64(32)).astype(np.uint32)).view(dtype).copy()
    if dtype.kind == "f":
        keys[::7] = 0.0
        keys[3::11] = -0.0
        keys[np.isnan(keys)] = 1.5
    return keys


@pytest.mark.parametrize("dtype,vbytes", [(np.uint32, 0), (np.uint32, 4), (np.float32, 8), (np.int32, 4), (np.uint64, 4),
                                          (np.int64, 0), (np.float64, 8)])
@pytest.mark.parametrize("kind", ["uniform", "few", "low"])
def test_small_sizes(hip, orc, dev, dtype, vbytes, kind):
    last = LAST[np.dtype(dtype).itemsize]
    for n in (1, 2, 63, 64, 65, 127, 129, 255, 257, 1023, 1024, 1025, 2047, 2048, 2049, 3071, 3073, 12289, last - 1, last,
              last + 1):
        keys = make_keys(orc, dtype, n, 9000 + n, kind)
        log(f"small sort {np.dtype(dtype).name} v{vbytes} {kind} n={n}")
        for desc in (False, True):
            if not vbytes:
                check_bits(gpu_sort(hip, keys, descending=desc), orc.radix_sort(keys, descending=desc))
                continue
            vals = np.arange(n, dtype=np.uint32 if vbytes == 4 else np.uint64)
            ko, vo = gpu_sort(hip, keys, vals, descending=desc)
            eko, evo = orc.radix_sort(keys, vals, descending=desc)
            check_bits(ko, eko)
            assert np.array_equal(vo, evo)


@pytest.mark.parametrize("begin,end", [(0, 1), (3, 9), (5, 30), (24, 32), (31, 32)])
@pytest.mark.parametrize("n", [100, 2048, 2049, 30001])
def test_small_bit_ranges(hip, orc, dev, begin, end, n):
    """Partial ranges (1 to 4 passes): copy form (one pass has no scratch keys and keeps its onesweep pass above
    one tile) and both DoubleBuffer parities."""
    keys = make_keys(orc, np.int32, n, 31 * begin + end + n, "uniform")
    vals = np.arange(n, dtype=np.uint32)
    eko, evo = orc.radix_sort(keys, vals, begin, end)
    log(f"small bits [{begin},{end}) n={n}")
    ko, vo = gpu_sort(hip, keys, vals, begin, end)
    check_bits(ko, eko)
    assert np.array_equal(vo, evo)
    for start in (0, 1):
        k = [empty_dev(n, 4), empty_dev(n, 4)]
        v = [empty_dev(n, 4), empty_dev(n, 4)]
        k[start], v[start] = to_dev(keys), to_dev(vals)
        sel = hip.sort_pairs_db("i32", 4, k[0], k[1], v[0], v[1], start, n, begin, end)
        assert sel == start ^ (((end - begin + 7) // 8) & 1)
        check_bits(to_host(k[sel], np.int32, n), eko)
        assert np.array_equal(to_host(v[sel], np.uint32, n), evo)
