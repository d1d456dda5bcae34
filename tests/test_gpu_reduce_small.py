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
