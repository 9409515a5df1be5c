"""GPU: the pooled linear head against 64-bit sums, from one pixel and eight channels on, with a few and with many
slices of pixels, and its time where a sample has little to add."""
import time

import numpy as np
import pytest

from beamz_amd import _native as N

pytestmark = pytest.mark.gpu


def head(torch, B, HW, C, nout):
    rng = np.random.default_rng(HW + C)
    mk = lambda *s: torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda()
    a, fw, fb = mk(B, HW, C).bfloat16(), mk(nout, C), mk(nout)
    gap, out = torch.full((B, C), 7.0, device="cuda"), torch.full((B, nout), 7.0, device="cuda")
    call = lambda: N.call("bz_nn_head", a.data_ptr(), fw.data_ptr(), fb.data_ptr(), gap.data_ptr(), out.data_ptr(), B, HW, C,
                          nout, torch.cuda.current_stream().cuda_stream)
    return a, fw, fb, gap, out, call


@pytest.mark.parametrize("B,HW,C,nout", [(1, 1, 8, 1), (3, 2, 8, 33), (2, 255, 8, 1), (2, 256, 8, 2), (1, 1500, 8, 3),
                                         (2, 511, 16, 5), (1, 3, 32, 32), (2, 256, 32, 7), (1, 257, 64, 2),
                                         (2, 127, 64, 40), (1, 5, 256, 8), (1, 33, 256, 1), (2, 4, 2048, 3),
                                         (1, 3, 2048, 64)])
def test_head_against_64_bits(hip, B, HW, C, nout):
    torch = hip
    a, fw, fb, gap, out, call = head(torch, B, HW, C, nout)
    call()
    a64, w64 = a.double().cpu().numpy(), fw.double().cpu().numpy()
    mean, size = a64.mean(axis=1), np.abs(a64).mean(axis=1)
    u = 2.0 ** -24
    # HW additions, a division and a rounding; then C products and additions, the bias, and the pooled values' errors
    egap = (HW + 2) * u * size
    assert np.all(np.abs(gap.double().cpu().numpy() - mean) <= egap)
    ref = mean @ w64.T + fb.double().cpu().numpy()
    bound = egap @ np.abs(w64).T + (C + 2) * u * (np.abs(mean) @ np.abs(w64).T + np.abs(fb.double().cpu().numpy()))
    assert np.all(np.abs(out.double().cpu().numpy() - ref) <= bound * (1 + 1e-3))


def test_a_head_with_little_to_add_is_not_slow(hip):
    """One pixel of 8 channels takes no longer than 64 pixels of 64 channels (once it took three times as long: a slice
    per thread, added one after the other)."""
    torch = hip
    best = []
    for shape in ((16, 1, 8, 1), (16, 1500, 8, 1), (16, 64, 64, 8)):
        call = head(torch, *shape)[-1]
        times = []
        for _ in range(8):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(100):
                call()
            torch.cuda.synchronize()
            times.append(time.perf_counter() - t0)
        best.append(min(times))
    assert best[0] < 2 * best[2] and best[1] < 3 * best[2], best
