"""DeviceRadixSort of medium inputs (every tile of a pass resident, two-level sums of the tiles' counts) vs the
oracle, bit-exact: sizes around the path's first and last size, whole and partial tiles of 4,096, the line
between one and two levels (32 tiles), whole and partial groups of 16; both places of the histogram rows,
DoubleBuffer parities, temp storage without room for the path, in-place calls and the forced fallback."""
import numpy as np
import pytest
import torch

from gpu_util import empty_dev, log, to_dev, to_host
from test_gpu_radix_small import LAST, make_keys
from test_gpu_radix_sort import SUFFIX, check_bits, gpu_sort

pytestmark = pytest.mark.gpu

TILE = 4096


@pytest.mark.parametrize("dtype,vbytes", [(np.uint32, 0), (np.uint32, 4), (np.float32, 8), (np.uint64, 4), (np.float64, 0),
                                          (np.uint64, 8), (np.int64, 8)])
@pytest.mark.parametrize("kind", ["uniform", "few"])
def test_mid_sizes(hip, orc, dev, dtype, vbytes, kind):
    last = LAST[np.dtype(dtype).itemsize]
    for n in (last + 1, 10 * TILE, 16 * TILE + 1, 32 * TILE - 1, 32 * TILE, 32 * TILE + 1, 33 * TILE, 47 * TILE + 17,
              64 * TILE, (1 << 21) - 5, 1 << 21, (1 << 21) + 1):
        keys = make_keys(orc, dtype, n, 70 + n, kind)
        desc = n % 2 == 1
        log(f"mid sort {np.dtype(dtype).name} v{vbytes} {kind} n={n} desc={desc}")
        if not vbytes:
            check_bits(gpu_sort(hip, keys, descending=desc), orc.radix_sort(keys, descending=desc))
            continue
        vals = np.arange(n, dtype=np.uint32 if vbytes == 4 else np.uint64)
        ko, vo = gpu_sort(hip, keys, vals, descending=desc)
        eko, evo = orc.radix_sort(keys, vals, descending=desc)
        check_bits(ko, eko)
        assert np.array_equal(vo, evo)


@pytest.mark.parametrize("begin,end", [(0, 8), (3, 17), (2, 24), (0, 30)])
@pytest.mark.parametrize("spin", [None, 0])
def test_mid_bits_and_double_buffer(hip, orc, dev, begin, end, spin):
    """One to four passes; with spin limit 0 every unpublished row (a tile's or a group's) is counted from the keys."""
    n = 300007
    lib = hip.lib()
    keys = make_keys(orc, np.uint32, n, begin + 100 * end, "uniform")
    vals = np.arange(n, dtype=np.uint32)
    eko, evo = orc.radix_sort(keys, vals, begin, end)
    log(f"mid bits [{begin},{end}) spin={spin}")
    old = lib.lcpp_hip_get_lookback_spin_limit()
    try:
        if spin is not None:
            lib.lcpp_hip_set_lookback_spin_limit(spin)
        ko, vo = gpu_sort(hip, keys, vals, begin, end)
        check_bits(ko, eko)
        assert np.array_equal(vo, evo)
        for start in (0, 1):
            k = [empty_dev(n, 4), empty_dev(n, 4)]
            v = [empty_dev(n, 4), empty_dev(n, 4)]
            k[start], v[start] = to_dev(keys), to_dev(vals)
            sel = hip.sort_pairs_db("u32", 4, k[0], k[1], v[0], v[1], start, n, begin, end)
            assert sel == start ^ (((end - begin + 7) // 8) & 1)
            check_bits(to_host(k[sel], np.uint32, n), eko)
            assert np.array_equal(to_host(v[sel], np.uint32, n), evo)
    finally:
        lib.lcpp_hip_set_lookback_spin_limit(old)


@pytest.mark.parametrize("dtype,vbytes", [(np.uint32, 4), (np.uint64, 8)])
def test_mid_smallest_temp_and_in_place(hip, orc, dev, dtype, vbytes):
    """The smallest temp storage the sort accepts (no room for this path's rows), and keys and values sorted in
    place with reference-sized temp storage (no room for the histogram rows either, so not in the output)."""
    n = 100003
    kb = np.dtype(dtype).itemsize
    sfx = SUFFIX[np.dtype(dtype)]
    keys = make_keys(orc, dtype, n, 5, "uniform")
    vals = np.arange(n, dtype=np.uint32 if vbytes == 4 else np.uint64)
    eko, evo = orc.radix_sort(keys, vals)
    need = hip.lib().lcpp_hip_internal_radix_needed_bytes(n, kb, vbytes, 0, 8 * kb, 0)
    small = torch.empty(need // 4, dtype=torch.int32, device=dev)
    kin, vin, kout, vout = to_dev(keys), to_dev(vals), empty_dev(n, kb), empty_dev(n, vbytes)
    log(f"mid smallest temp {need} bytes, {sfx} v{vbytes}")
    hip.sort_pairs(sfx, vbytes, kin, kout, vin, vout, n, temp=small)
    check_bits(to_host(kout, dtype, n), eko)
    assert np.array_equal(to_host(vout, vals.dtype, n), evo)
    hip.sort_pairs(sfx, vbytes, kin, kin, vin, vin, n)
    check_bits(to_host(kin, dtype, n), eko)
    assert np.array_equal(to_host(vin, vals.dtype, n), evo)


@pytest.mark.parametrize("spin", [None, 0])
@pytest.mark.parametrize("dtype", [np.uint64, np.int64, np.float64])
def test_mid_more_tiles_than_run_together(hip, orc, dev, dtype, spin):
    """8-byte keys with 8-byte values, one workgroup per CU: tiles of a second round add up the rows of the first."""
    n = (1 << 20) + 37 * TILE + 11
    keys = make_keys(orc, dtype, n, 91, "uniform")
    vals = np.arange(n, dtype=np.uint64)
    lib = hip.lib()
    old = lib.lcpp_hip_get_lookback_spin_limit()
    try:
        if spin is not None:
            lib.lcpp_hip_set_lookback_spin_limit(spin)
        log(f"mid sort {np.dtype(dtype).name} v8 n={n} spin={spin}")
        ko, vo = gpu_sort(hip, keys, vals, descending=True)
    finally:
        lib.lcpp_hip_set_lookback_spin_limit(old)
    eko, evo = orc.radix_sort(keys, vals, descending=True)
    check_bits(ko, eko)
    assert np.array_equal(vo, evo)
