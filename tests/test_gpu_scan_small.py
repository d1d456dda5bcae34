"""Scans of one tile and of the two-launch form, at the edges of their tiles (4 KB per row of 256 threads, 16 KB
of 1,024) and of the number of tiles, aligned and not, in place and not, against numpy."""
import numpy as np
import pytest
import torch

from gpu_util import to_dev

pytestmark = pytest.mark.gpu
NP = {"i32": np.int32, "u32": np.uint32, "f32": np.float32, "u64": np.uint64, "f64": np.float64}


def sizes(itemsize):
    v = 16 // itemsize
    tile, one = 1024 * v, 4096 * v
    return [1, 2, v - 1, v, v + 1, tile - 1, tile, tile + 1, one - 1, one, one + 1, 256 * tile, 257 * tile + 5,
            2048 * tile - 1, 2048 * tile, 2048 * tile + 1]


@pytest.mark.parametrize("t", ["i32", "u32", "f32", "u64", "f64"])
@pytest.mark.parametrize("inclusive", [False, True])
@pytest.mark.parametrize("op", ["sum", "max"])
def test_scan_small(hip, dev, t, inclusive, op):
    rng = np.random.default_rng(5)
    for n in sizes(np.dtype(NP[t]).itemsize):
        # Small whole numbers: float sums stay below 2^24 at every size, so they are exact in any order.
        x = rng.integers(0, 2 if n > 100_000 else 50, n).astype(NP[t])
        for off, in_place in [(0, False), (1, False), (0, True)]:
            src = to_dev(np.concatenate([np.zeros(off, NP[t]), x]))[off:]
            out = src if in_place else torch.zeros_like(src)
            if op == "sum":
                hip.scan_sum(t, src, out, n, inclusive=inclusive)
                want = np.cumsum(x.astype(np.float64 if t[0] == "f" else np.uint64)).astype(NP[t])
                want = want if inclusive else np.concatenate([[NP[t](0)], want[:-1]])
            else:
                hip.scan_minmax("max", t, src, out, n, inclusive=inclusive, init=7)
                want = np.maximum(np.maximum.accumulate(x), NP[t](7))
                want = want if inclusive else np.concatenate([[NP[t](7)], want[:-1]])
            np.testing.assert_array_equal(out.cpu().numpy().view(NP[t]), want.astype(NP[t]), err_msg=f"{t} {n} {off} {in_place}")
