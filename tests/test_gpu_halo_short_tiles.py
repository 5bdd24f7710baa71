"""Resident-tile convolution of channel-minor layers whose last rounds of tiles, or all of them, are short (192 positions of 256):
forward and input gradient where a tile ends inside a row, between samples and behind the last one."""
import pytest
import torch
import torch.nn.functional as F

import helpers as hp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# samples, channels in, out, height, width: one round, of short tiles only (one to three blocks of filters, images smaller than a
# tile, a tile that ends with the last position); whole and short rounds
@pytest.mark.parametrize("case", [(1, 64, 128, 12, 15), (3, 64, 128, 14, 14), (1, 128, 128, 30, 11), (70, 64, 256, 9, 9), (2, 128, 384, 44, 44),
                                  (8, 64, 128, 6, 7), (128, 64, 128, 28, 28), (100, 128, 256, 20, 20), (77, 192, 128, 33, 33)])
def test_short_tiles(pkg, gpu, case):
    ns, Ci, Co, H, W = case
    g = torch.Generator(device=DEV).manual_seed(Ci + H)
    x = (torch.rand((ns, Ci, H, W), generator=g, device=DEV) * 2 - 1).half()
    w = ((torch.rand((Co, Ci, 3, 3), generator=g, device=DEV) * 2 - 1) * (6.0 / (9 * Ci)) ** 0.5).half()
    dy = (torch.rand((ns, Co, H, W), generator=g, device=DEV) * 2 - 1).half()
    ref = F.conv2d(x.float(), w.float(), padding=1)
    grad = F.conv_transpose2d(dy.float(), w.float(), padding=1)
    x, w, dy, ref, grad = (t.permute(0, 2, 3, 1).contiguous() for t in (x, w, dy, ref, grad))
    y, dx = torch.empty_like(ref, dtype=torch.float16), torch.empty_like(grad, dtype=torch.float16)
    fw, keep = hp.conv2d_args(pkg, x, None, w, None, y, y, Ci, H, W, Co, 3, 3, H, W, (1,) * 4, (1, 1), 1)
    bw, keep2 = hp.conv2d_args(pkg, x, dx, w, None, y, dy, Ci, H, W, Co, 3, 3, H, W, (1,) * 4, (1, 1), 1)
    gpu.ptl_set_gemm_path(5)
    try:
        for call, a, got, want, n in (("ptl_conv2d_fp16_fw_batched", fw, y, ref, 9 * Ci), ("ptl_conv2d_fp16_ig_batched", bw, dx, grad, 9 * Co)):
            for _ in range(2):
                got.fill_(7)
                torch.cuda.synchronize()
                pkg.call(call, a, ns)
                assert gpu.ptl_sync() == 0 and gpu.ptl_last_conv_resident() == 1
                # half a unit in the last place of the result, and n rounded fp32 additions of terms below 1 on either side
                assert bool(((got.float() - want).abs() <= 2.0 ** -11 * want.abs() + 2.0 ** -23 * n).all()), call
    finally:
        gpu.ptl_set_gemm_path(0)
