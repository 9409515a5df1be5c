"""GPU: the tiled 3x3 convolution (16-byte accesses, 64-channel slices) gives the bits of the general one, which serves
a tensor that is not aligned to 16 bytes: both add the same products in the same order. Sizes at the edges of every
tile shape (pixels past a tile, one pixel, images narrower than a tap), each output-channel remainder, with and
without ReLU, bias and mask."""
import pytest

from beamz_amd import _native as N

pytestmark = pytest.mark.gpu

# B, H, W, Ci, Co
SHAPES = [(1, 1, 1, 64, 64), (1, 1, 2, 128, 32), (1, 2, 1, 64, 96), (3, 7, 11, 64, 64), (2, 9, 13, 192, 32),
          (5, 5, 26, 128, 192),                                   # 64 x 64 tiles
          (1, 181, 91, 64, 64), (1, 182, 91, 64, 128),            # 128.7 and 129.4 tiles of 128 pixels: 64 x 64
          (1, 181, 181, 64, 64), (2, 128, 64, 64, 128),           # at least 256 tiles of 128 x 64
          (1, 181, 182, 64, 128), (2, 91, 91, 64, 256),           # at least 256 tiles of 128 x 128
          (1, 16, 64, 64, 32),                                    # 64-pixel rows too few for the row march
          (3, 40, 30, 64, 96), (5, 26, 26, 64, 160), (2, 33, 31, 128, 352)]      # several tiles of odd channel blocks


@pytest.mark.parametrize("shape", SHAPES)
def test_tiled_convolution_gives_the_bits_of_the_general_one(hip, shape):
    import torch
    B, H, W, Ci, Co = shape
    gen = torch.Generator(device="cuda").manual_seed(H * W + Ci)
    rnd = lambda *s: torch.randn(s, generator=gen, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    x, w, b = rnd(B, H, W, Ci).bfloat16(), (rnd(Co, 3, 3, Ci) / (3 * Ci ** 0.5)).bfloat16(), rnd(Co)
    n = B * H * W * Co
    masks = [torch.zeros(n + 1, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    m = torch.relu(rnd(n)).bfloat16()
    masks[0][:n], masks[1][1:] = m, m
    got = []
    for off in (0, 1):                       # aligned, and 2 bytes past: the general kernel
        mask = masks[off].data_ptr() + 2 * off
        outs = [torch.full((n + 1,), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(4)]
        ptr = [o.data_ptr() + 2 * off for o in outs]
        N.call("bz_nn_conv3x3", x.data_ptr(), w.data_ptr(), b.data_ptr(), ptr[0], B, H, W, Ci, Co, 1, st)
        N.call("bz_nn_conv3x3", x.data_ptr(), w.data_ptr(), None, ptr[1], B, H, W, Ci, Co, 0, st)
        N.call("bz_nn_conv3x3_dgrad", x.data_ptr(), w.data_ptr(), ptr[2], B, H, W, Co, Ci, st)
        N.call("bz_nn_conv3x3_dgrad_relu", x.data_ptr(), w.data_ptr(), mask, ptr[3], B, H, W, Co, Ci, st)
        assert all(float(o[n if off == 0 else 0]) == 7.0 for o in outs)      # nothing past the tensor's ends
        got.append([o[off:n + off].view(torch.int16) for o in outs])
    assert all(torch.equal(p, q) for p, q in zip(*got))
    ref = torch.nn.functional.conv2d(x.double().cpu().permute(0, 3, 1, 2), w.double().cpu().permute(0, 3, 1, 2),
                                     b.double().cpu(), padding=1).relu().permute(0, 2, 3, 1)
    y = got[0][0].view(torch.bfloat16).view(B, H, W, Co).double().cpu()
    # half a bfloat16 step of the result, and the FP32 sums' 9 Ci roundings of the terms' mean size
    assert bool(((y - ref).abs() <= 2.0 ** -8 * ref + 9 * Ci * 2.0 ** -24 * 3).all())


def test_channel_counts_that_are_no_multiple_of_64_keep_their_input_on_chip(hip):
    """256 -> 288 channels take at most 2.5 times as long as 256 -> 256 on an input larger than the second-level caches
    (1.6 times as built; four times when every block of 32 channels read the input from memory)."""
    import torch
    st = torch.cuda.current_stream().cuda_stream
    B, H, W, Ci = 128, 32, 32, 256
    x = torch.randn(B, H, W, Ci, device="cuda").bfloat16()
    best = {}
    for Co in (256, 288):
        w = torch.randn(Co, 3, 3, Ci, device="cuda").bfloat16()
        y = torch.empty(B, H, W, Co, dtype=torch.bfloat16, device="cuda")
        times = []
        for _ in range(10):
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            for _ in range(5):
                N.call("bz_nn_conv3x3", x.data_ptr(), w.data_ptr(), None, y.data_ptr(), B, H, W, Ci, Co, 1, st)
            e[1].record()
            torch.cuda.synchronize()
            times.append(e[0].elapsed_time(e[1]))
        best[Co] = min(times)
    assert best[288] < 2.5 * best[256], best
