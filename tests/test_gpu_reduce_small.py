"""Sum, Min and Max at the edges of the inputs that one workgroup folds (16 KB and 64 KB) and of alignment."""
import numpy as np
import pytest
import torch

from gpu_util import to_dev

pytestmark = pytest.mark.gpu
NP = {"i32": np.int32, "f32": np.float32, "u64": np.uint64, "f64": np.float64}


@pytest.mark.parametrize("t", list(NP))
def test_one_workgroup(hip, dev, t):
    rng = np.random.default_rng(1)
    v = 16 // np.dtype(NP[t]).itemsize
    for n in [1, v - 1, v, v + 1] + [m * v + d for m in (1024, 4096) for d in (-1, 0, 1, v, 2 * v)]:
        for off in range(min(v, 2)):
            x = rng.integers(1, 100, n).astype(NP[t])  # whole numbers: every order gives the exact sum
            d = to_dev(np.concatenate([np.full(off, 1 << 20, NP[t]), x, np.full(3, 1 << 20, NP[t])]))[off:]
            out = torch.zeros(1, dtype=d.dtype, device=dev)
            hip.reduce_sum(t, d, out, n)
            assert out.cpu().numpy().view(NP[t])[0] == x.sum(dtype=np.float64 if t[0] == "f" else np.int64)
            for fold in ("min", "max"):
                hip.reduce_minmax(fold, t, d, out, n)
                assert out.cpu().numpy().view(NP[t])[0] == getattr(x, fold)()


def pairwise(x):
    while x.shape[-1] > 1:
        x = x[..., 0::2] + x[..., 1::2]
    return x[..., 0]


def two_launch_sum(x):
    """The float32 sum in the order of workgroups of 256 threads, four 16-byte vectors each, and a final kernel: items of a
    vector, a thread's vectors and a workgroup's waves one after the other, lanes and workgroups pairwise."""
    v = np.zeros((-(-x.size // 4096) * 1024, 4), np.float32)
    v.reshape(-1)[:x.size] = x
    s = (v[:, 0] + v[:, 1]) + v[:, 2] + v[:, 3]
    a = s.reshape(-1, 4, 4, 64)  # workgroup, vector, wave, lane
    w = pairwise(a[:, 0] + a[:, 1] + a[:, 2] + a[:, 3])
    partials = np.zeros(64, np.float32)
    partials[:len(w)] = w[:, 0] + w[:, 1] + w[:, 2] + w[:, 3]
    return pairwise(partials)


@pytest.mark.parametrize("n", [4200, 5004, 8192, 12_000, 16_384])
def test_one_workgroup_rounds_no_more_than_two_launches(hip, dev, n):
    """Mean distance from the 64-bit sum over 200 inputs; one workgroup's fold may not lie further off."""
    out = torch.zeros(1, dtype=torch.float32, device=dev)
    one, reduced, two = [], [], []
    for seed in range(200):
        x = np.random.default_rng(seed).random(n, dtype=np.float32)
        d, exact = to_dev(x), x.sum(dtype=np.float64)
        hip.reduce_sum("f32", d, out, n)
        one.append(abs(float(out.item()) - exact))
        hip.reduce_op("sum", "f32", d, out, n)
        reduced.append(abs(float(out.item()) - exact))
        two.append(abs(float(two_launch_sum(x)) - exact))
    assert max(np.mean(one), np.mean(reduced)) <= 1.02 * np.mean(two)
