"""GPU: the first convolution against 64-bit sums: rows staged in LDS with every remainder of their length, channel counts
from one group to the widest whose weights fit and past it, and small batches of many rows per workgroup."""
import numpy as np
import pytest

from beamz_amd import _native as N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,W,C", [(1, 1, 1, 8), (2, 3, 5, 8), (1, 16, 16, 16), (3, 7, 17, 32), (2, 6, 130, 64),
                                     (1, 25, 31, 128), (5, 16, 18, 256), (600, 16, 16, 32), (1, 2, 19, 1024),
                                     (1, 3, 5, 2048), (1, 4, 9, 24), (1, 3, 4, 5)])
def test_first_layer(hip, B, H, W, C):
    import torch
    rng = np.random.default_rng(H * W + C)
    x = torch.from_numpy(rng.random((B, H, W), dtype=np.float32)).cuda().bfloat16()
    w = torch.from_numpy(rng.standard_normal((C, 9), dtype=np.float32)).cuda()
    b = torch.from_numpy(rng.standard_normal(C, dtype=np.float32)).cuda()
    y = torch.full((B * H * W * C + 1,), 7.0, dtype=torch.bfloat16, device="cuda")
    N.call("bz_nn_conv_first", x.data_ptr(), w.data_ptr(), b.data_ptr(), y.data_ptr(), B, H, W, C,
           torch.cuda.current_stream().cuda_stream)
    assert float(y[-1]) == 7.0
    xp = np.zeros((B, H + 2, W + 2))
    xp[:, 1:-1, 1:-1] = x.double().cpu().numpy()
    w64 = w.bfloat16().double().cpu().numpy()
    taps = np.stack([xp[:, t // 3:t // 3 + H, t % 3:t % 3 + W] for t in range(9)], axis=-1)
    ref = np.maximum(taps @ w64.T + b.double().cpu().numpy(), 0.0)
    size = np.abs(taps) @ np.abs(w64).T + np.abs(b.double().cpu().numpy())
    got = y[:-1].double().cpu().numpy().reshape(B, H, W, C)
    # half a bfloat16 step of the result; nine additions, the bias and the products' roundings
    assert np.all(np.abs(got - ref) <= 2.0 ** -8 * ref + 12 * 2.0 ** -24 * size)
