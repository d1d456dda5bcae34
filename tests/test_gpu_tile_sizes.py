"""Select, partition, by-key and run-length calls at the edges of the tiles they use for small and medium inputs
and of the sizes where the tiles change, with and without the helped look-back, against numpy."""
import numpy as np
import pytest
import torch

from gpu_util import to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[None, 0])
def spin(hip, request):
    lib = hip.lib()
    old = lib.lcpp_hip_get_lookback_spin_limit()
    if request.param is not None:
        lib.lcpp_hip_set_lookback_spin_limit(request.param)
    yield
    lib.lcpp_hip_set_lookback_spin_limit(old)


def around(*edges):
    return [n + d for n in edges for d in (-1, 0, 1)]


SELECT = [1, 63] + around(4096, 64 * 4096, 1536 * 4096, 5120 * 8192)


@pytest.mark.parametrize("n", SELECT)
def test_select_and_partition(hip, dev, spin, n):
    x = np.random.default_rng(n).integers(0, 1 << 32, n, dtype=np.uint32)
    d, num = to_dev(x), torch.zeros(1, dtype=torch.int32, device=dev)
    keep = x < 0x55555555
    for call in (hip.select_if, hip.partition_if):
        out = torch.zeros_like(d)
        call("u32", d, out, num, n, hip.predicate("u32", (hip.PRED_LT, 0x55555555)))
        k = int(keep.sum())
        assert int(num.item()) == k
        got = out.cpu().numpy().view(np.uint32)
        np.testing.assert_array_equal(got[:k], x[keep])
        if call is hip.partition_if:
            np.testing.assert_array_equal(got[k:], x[~keep][::-1])


@pytest.mark.parametrize("t", ["u32", "u64"])
@pytest.mark.parametrize("n", [3 * 4096 + 5, 1536 * 4096 + 4097, 5120 * 8192 + 1])
def test_select_everything(hip, dev, t, n):
    """Rows whose masks fill a word only in part (4 rows of u32, every row count of u64)."""
    np_t = np.uint32 if t == "u32" else np.uint64
    x = np.random.default_rng(n).integers(0, 1 << 31, n).astype(np_t)
    d, num = to_dev(x), torch.zeros(1, dtype=torch.int32, device=dev)
    out = torch.zeros(2 * n, dtype=d.dtype, device=dev)  # room for a count twice too large
    hip.select_if(t, d, out[:n], num, n, hip.predicate(t, (hip.PRED_TRUE,)))
    assert int(num.item()) == n
    np.testing.assert_array_equal(out.cpu().numpy().view(np_t)[:n], x)
    assert not out[n:].any()


FLAGGED = [("u32", n) for n in around(4096, 1536 * 4096) + [5120 * 8192, 5120 * 8192 + 1]] + \
          [("u64", n) for n in around(2048, 1536 * 2048, 3584 * 4096)]


@pytest.mark.parametrize("t,n", FLAGGED)
@pytest.mark.parametrize("fs", ["b8", "u32"])
def test_flagged(hip, dev, spin, t, n, fs):
    """Select and partition by flags, over tiles of 4, 8 and 12 rows."""
    np_t = np.uint32 if t == "u32" else np.uint64
    rng = np.random.default_rng(n)
    x = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np_t)
    keep = rng.random(n, dtype=np.float32) < 0.6
    d, num = to_dev(x), torch.zeros(1, dtype=torch.int32, device=dev)
    flags = to_dev(keep.astype(np.uint8 if fs == "b8" else np.uint32))
    k = int(keep.sum())
    for call in (hip.select_flagged, hip.partition_flagged):
        out = torch.zeros_like(d)
        call(t, fs, d, flags, out, num, n)
        assert int(num.item()) == k
        got = out.cpu().numpy().view(np_t)
        np.testing.assert_array_equal(got[:k], x[keep])
        np.testing.assert_array_equal(got[k:], x[~keep][::-1] if call is hip.partition_flagged else 0)


@pytest.mark.parametrize("n", [5] + around(2048, 1536 * 2048, 3584 * 4096, 5120 * 4096))
def test_select_and_partition_8_byte(hip, dev, spin, n):
    """The 8-byte items' row counts (4, 8, 12) with a predicate that keeps a part."""
    x = np.random.default_rng(n).integers(0, 1 << 63, n, dtype=np.uint64) << np.uint64(1)
    bound = 0xA000000000000000
    d, num = to_dev(x), torch.zeros(1, dtype=torch.int32, device=dev)
    keep = x < np.uint64(bound)
    k = int(keep.sum())
    for call in (hip.select_if, hip.partition_if):
        out = torch.zeros_like(d)
        call("u64", d, out, num, n, hip.predicate("u64", (hip.PRED_LT, bound)))
        assert int(num.item()) == k
        got = out.cpu().numpy().view(np.uint64)
        np.testing.assert_array_equal(got[:k], x[keep])
        np.testing.assert_array_equal(got[k:], x[~keep][::-1] if call is hip.partition_if else 0)


RUNS = [1, 3] + around(4096, 64 * 4096, (32 << 20) // 8, (24 << 20) // 4)


@pytest.mark.parametrize("n", RUNS)
@pytest.mark.parametrize("mean", [1, 9, 100_000])
def test_runs_and_by_key(hip, dev, spin, n, mean):
    rng = np.random.default_rng(n)
    head = rng.random(n) < 1.0 / mean
    head[0] = True
    key = np.cumsum(head).astype(np.int32)
    at = np.flatnonzero(head)
    length = np.diff(np.append(at, n))
    x = rng.integers(0, 1000, n).astype(np.int32)
    dk, dx, num = to_dev(key), to_dev(x), torch.zeros(1, dtype=torch.int32, device=dev)
    # 32-bit sums wrap: differences of a 64-bit running sum, reduced to 32 bits.
    s = np.concatenate([[0], np.cumsum(x.astype(np.int64))])
    for form in ("encode", "reduce"):
        unique, second = torch.zeros_like(dk), torch.zeros_like(dk)
        if form == "encode":
            hip.run_length_encode("u32", dk, unique, second, num, n)
            want = length
        else:
            hip.reduce_by_key("i32", "i32", dk, dx, unique, second, num, n)
            want = s[at + length] - s[at]
        assert int(num.item()) == at.size
        np.testing.assert_array_equal(unique.cpu().numpy()[:at.size], key[at])
        np.testing.assert_array_equal(second.cpu().numpy()[:at.size], want.astype(np.int32))
    want = (s[:-1] - np.repeat(s[at], length)).astype(np.int32)
    for out in (torch.zeros_like(dx), dx):  # the second in place
        hip.scan_by_key("i32", "i32", dk, dx, out, n)
        np.testing.assert_array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("n", [42_000_000, 42_000_001])
def test_scan_by_key_where_the_tiles_change(hip, dev, n):
    x = np.random.default_rng(1).integers(0, 50, n).astype(np.int32)
    key = (np.arange(n) // 1000).astype(np.int32)
    out = torch.zeros(n, dtype=torch.int32, device=dev)
    hip.scan_by_key("i32", "i32", to_dev(key), to_dev(x), out, n)
    s = np.cumsum(x) - x
    np.testing.assert_array_equal(out.cpu().numpy(), (s - s[::1000][key]).astype(np.int32))


@pytest.mark.parametrize("k,t,n", [(k, t, n) for k, t, b in [("i32", "u32", 8), ("i64", "i32", 12), ("u32", "i64", 12),
                                                             ("u64", "u64", 16)]
                                   for n in around((64 << 20) // b, 1400 * 6144)])
def test_scan_by_key_mid_tiles(hip, dev, spin, k, t, n):
    """Above 64 MB of keys and values the tiles have 6 rows (items of 8 and 12 bytes); runs within a tile, over more tiles
    than one look-back step reads, and a single one, out of place and in place."""
    np_t = np.dtype({"u": np.uint32, "i": np.int32}[t[0]] if t[1:] == "32" else {"u": np.uint64, "i": np.int64}[t[0]])
    x = np.random.default_rng(n).integers(0, 50, n).astype(np_t)
    s = np.cumsum(x, dtype=np_t)
    for run in (1000, 700_001, n):
        at = np.arange(n) // run
        start = (s - x)[::run][at]
        dk, dx = to_dev(at.astype(np.int64 if k[1:] == "64" else np.int32)), to_dev(x)
        out = torch.zeros_like(dx)
        hip.scan_by_key(k, t, dk, dx, out, n)
        np.testing.assert_array_equal(out.cpu().numpy().view(np_t), s - x - start)
        hip.scan_by_key(k, t, dk, dx, dx, n, inclusive=True)
        np.testing.assert_array_equal(dx.cpu().numpy().view(np_t), s - start)
