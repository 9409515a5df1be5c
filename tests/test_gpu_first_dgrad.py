"""GPU: the input gradient of the first convolution at 32 channels against 64-bit sums: bands of 8 rows down to one,
images smaller than a band, a tap or 16 pixels, rows at and past the widest that fit, one and several images."""
import numpy as np
import pytest

from beamz_amd import _native as N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,W", [(1, 1, 1), (2, 1, 5), (3, 3, 16), (2, 7, 17), (2, 16, 64), (1, 24, 128), (1, 6, 130),
                                   (1, 5, 401), (1, 4, 604), (1, 4, 605), (20, 128, 9), (300, 7, 3), (257, 8, 20),
                                   (90, 18, 33)])
def test_first_layer_input_gradient(hip, B, H, W):
    import torch
    C = 32
    rng = np.random.default_rng(H * W)
    x = torch.from_numpy(rng.random((B, H, W), dtype=np.float32)).cuda().bfloat16()
    gz = torch.from_numpy(rng.standard_normal((B, H, W, C), dtype=np.float32)).cuda().bfloat16()
    w = torch.from_numpy(rng.standard_normal((C, 9), dtype=np.float32)).cuda()
    gw, gb = torch.zeros_like(w), torch.zeros(C, device="cuda")
    gx = torch.full((B * H * W + 1,), 7.0, device="cuda")
    N.call("bz_nn_conv_first_bwd", x.data_ptr(), gz.data_ptr(), w.data_ptr(), gw.data_ptr(), gb.data_ptr(),
           gx.data_ptr(), B, H, W, C, None, 0, torch.cuda.current_stream().cuda_stream)
    g64, w64 = gz.double().cpu().numpy(), w.bfloat16().double().cpu().numpy()
    ref, size = np.zeros((B, H, W)), np.zeros((B, H, W))
    for tap in range(9):
        dy, dx = tap // 3 - 1, tap % 3 - 1
        ys, xs = slice(max(dy, 0), H + min(dy, 0)), slice(max(dx, 0), W + min(dx, 0))
        yq, xq = slice(max(-dy, 0), H + min(-dy, 0)), slice(max(-dx, 0), W + min(-dx, 0))
        ref[:, ys, xs] += g64[:, yq, xq] @ w64[:, tap]
        size[:, ys, xs] += np.abs(g64[:, yq, xq]) @ np.abs(w64[:, tap])
    assert float(gx[-1]) == 7.0
    got = gx[:-1].double().cpu().numpy().reshape(B, H, W)
    # exact products (bfloat16 factors); at most 32 + 9 FP32 additions a value
    assert np.all(np.abs(got - ref) <= 41 * 2.0 ** -24 * size)
