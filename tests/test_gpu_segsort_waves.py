"""Segmented radix-order sorts whose segments average 64 items or more: a wave or a workgroup per segment.
Lengths at the edges of the items per lane (64, 128, 256, 512) and per thread (1,024, 2,048, 4,096), empty
segments, gaps that stay untouched, partial bit ranges and several segments per wave, against the oracle."""
import numpy as np
import pytest
import torch

from gpu_util import to_dev, to_host
from test_gpu_segsort import NP, check, g_sort

pytestmark = pytest.mark.gpu
EDGES = [0, 1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096, 4097,
         9000]


def words(rng, n, ks):
    k = rng.integers(0, 1 << 64, n, dtype=np.uint64).view(np.uint8)[:n * np.dtype(NP[ks]).itemsize].view(NP[ks]).copy()
    if ks in ("f32", "f64"):
        k = np.where(np.isfinite(k), k, NP[ks](0))
        k[::5] = NP[ks](-0.0)
    else:
        k[::3] &= NP[ks](0x70F)
    return k


def layout(rng, lengths):
    """Segments in random order, some behind a gap."""
    lengths = rng.permutation(lengths)
    gaps = rng.integers(0, 2, lengths.size) * rng.integers(0, 40, lengths.size)
    e = np.cumsum(lengths + gaps)
    return (e - lengths).astype(np.uint32), e.astype(np.uint32), int(e[-1]) + 7


@pytest.mark.parametrize("ks", ["u32", "i32", "f32", "u64", "i64", "f64"])
@pytest.mark.parametrize("vb", [0, 4, 8])
@pytest.mark.parametrize("desc", [False, True])
def test_lengths_at_the_edges(hip, orc, dev, ks, vb, desc):
    rng = np.random.default_rng(vb + desc)
    b, e, n = layout(rng, np.array(EDGES + EDGES[:14]))
    keys = words(rng, n, ks)
    vals = np.arange(n, dtype=np.uint32 if vb == 4 else np.uint64) if vb else None
    for begin, end in [(0, None), (3, 17), (5, 5)]:
        kw = dict(begin_bit=begin, end_bit=end, descending=desc)
        gk, gv = g_sort(hip, keys, b, e, values=vals, **kw)
        kw["end_bit"] = 8 * keys.itemsize if end is None else end
        check(orc, keys, b, e, gk, gv, values=vals, **kw)


@pytest.mark.parametrize("ks,vb", [("u32", 0), ("f32", 4), ("u32", 8), ("i64", 0), ("u64", 4), ("f64", 8)])
@pytest.mark.parametrize("desc", [False, True])
def test_tiny_segments(hip, orc, dev, ks, vb, desc):
    """Segments of 1 to 17 items, a 16-lane row each up to 16, beside longer ones that keep the mean at 64 or more."""
    rng = np.random.default_rng(vb + desc)
    b, e, n = layout(rng, np.concatenate([np.arange(1, 18).repeat(40), np.full(700, 16), np.full(22, 4096), [300, 513, 1024]]))
    assert len(b) <= n // 64
    keys = words(rng, n, ks)
    keys[::2] = keys[0]  # ties
    vals = np.arange(n, dtype=np.uint32 if vb == 4 else np.uint64) if vb else None
    for begin, end in [(0, 8 * keys.itemsize), (3, 17), (5, 5)]:
        kw = dict(begin_bit=begin, end_bit=end, descending=desc)
        gk, gv = g_sort(hip, keys, b, e, values=vals, **kw)
        check(orc, keys, b, e, gk, gv, values=vals, **kw)


def test_several_segments_per_wave(hip, orc, dev):
    rng = np.random.default_rng(3)
    b, e, n = layout(rng, np.concatenate([rng.integers(0, 150, 110_000), [513, 1500, 4096, 4097, 5000]]))
    assert len(b) <= n // 64
    keys = words(rng, n, "u32")
    vals = np.arange(n, dtype=np.uint32)
    gk, gv = g_sort(hip, keys, b, e, values=vals)
    check(orc, keys, b, e, gk, gv, values=vals)


@pytest.mark.parametrize("ks,vb", [("u32", 0), ("f32", 4), ("i32", 4), ("i64", 0)])
@pytest.mark.parametrize("desc", [False, True])
def test_medium_segments_apart(hip, orc, dev, ks, vb, desc):
    """Items of up to 8 bytes, 2^22 of them or more, more than 512 per segment: the block kernel sorts the tiny and the medium
    segments, the wave kernel those between."""
    rng = np.random.default_rng(vb + desc)
    b, e, n = layout(rng, np.concatenate([EDGES * 3, np.arange(1, 18), rng.integers(513, 4097, 1000)]).astype(np.int64))
    n = max(n, 1 << 22)
    assert len(b) < n // 512  # on average
    keys = words(rng, n, ks)
    vals = np.arange(n, dtype=np.uint32) if vb else None
    for begin, end in [(0, 8 * keys.itemsize), (3, 17), (5, 5)]:
        kw = dict(begin_bit=begin, end_bit=end, descending=desc)
        hip.profile_reset()
        hip.profile_enable(True)
        gk, gv = g_sort(hip, keys, b, e, values=vals, **kw)
        hip.profile_enable(False)
        assert [hip.profile_query(f"segsort_{x}")[1] for x in ("block", "waves", "tile")] == [1, 1, 0]
        check(orc, keys, b, e, gk, gv, values=vals, **kw)


@pytest.mark.parametrize("step,longest", [(1000, 1000), (70, 16)])
def test_double_buffer_in_place(hip, orc, dev, step, longest):
    """ceil(log2 n) is even: the result goes where the input is."""
    rng = np.random.default_rng(4)
    n = 60_000
    b = np.arange(0, n, step, dtype=np.uint32)
    e = np.minimum(b + rng.integers(0, longest + 1, b.size), n).astype(np.uint32)
    if step == 1000:
        b, e = b[:60], e[:60]
    keys, vals = words(rng, n, "u32"), np.arange(n, dtype=np.uint32)
    k0, v0 = to_dev(keys), to_dev(vals)
    k1, v1 = torch.zeros_like(k0), torch.zeros_like(v0)
    sel = hip.segmented_sort_db("u32", k0, k1, 0, n, b.size, to_dev(b), to_dev(e), values0=v0, values1=v1)
    wk, wv = orc.segmented_sort(keys, b, e, values=vals, keys_out=keys.copy(), values_out=vals.copy())
    assert sel == (0, 0)
    np.testing.assert_array_equal(to_host(k0, np.uint32, n), wk)
    np.testing.assert_array_equal(to_host(v0, np.uint32, n), wv)


@pytest.mark.parametrize("vb", [4, 8])
def test_segments_on_both_sides_of_2p31(hip, dev, vb):
    """Offsets that a signed 32-bit word does not hold: one segment for each number of items per lane, tiny and medium ones
    (which 12-byte items keep in the wave kernel)."""
    n = (1 << 31) + 20_000
    lengths = [1, 9, 40, 100, 200, 300, 512, 900, 4096]
    v_t = torch.int32 if vb == 4 else torch.int64
    b, e, at = [], [], (1 << 31) - sum(lengths) - 100
    for x in lengths + [333] + lengths:  # the one in the middle straddles 2^31
        b.append(at)
        e.append(at + x)
        at += x + 11
    assert b[len(lengths)] < 1 << 31 < e[len(lengths)] and e[-1] <= n
    first, last = b[0], e[-1]
    rng = np.random.default_rng(5)
    some = rng.integers(0, 1 << 32, last - first, dtype=np.uint64).astype(np.uint32)
    keys = torch.zeros(n, dtype=torch.int32, device=dev)
    keys[first:last] = to_dev(some)
    vals = torch.zeros(n, dtype=v_t, device=dev)
    vals[first:last] = torch.arange(last - first, dtype=v_t, device=dev)
    ko, vo = torch.full_like(keys, -1), torch.full_like(vals, -1)
    hip.segmented_sort("u32", keys, ko, n, len(b), to_dev(np.array(b, np.uint32)), to_dev(np.array(e, np.uint32)),
                       values_in=vals, values_out=vo)
    wk, wv = np.full(last - first, 0xFFFFFFFF, np.uint32), np.full(last - first, -1, np.int64)
    for x, y in zip(b, e):
        order = np.argsort(some[x - first:y - first], kind="stable")
        wk[x - first:y - first] = some[x - first:y - first][order]
        wv[x - first:y - first] = order + (x - first)
    np.testing.assert_array_equal(ko[first:last].cpu().numpy().view(np.uint32), wk)
    np.testing.assert_array_equal(vo[first:last].cpu().numpy(), wv)
    for out in (ko, vo):  # nothing else is written
        assert bool((out[:first] == -1).all()) and bool((out[last:] == -1).all())
    del keys, vals, ko, vo, out
    torch.cuda.empty_cache()
