"""Resident-tile convolution with 32- and 64-filter tiles on layers whose workgroups walk over many tiles and channel slabs: a
tile that is multiplied before all of its pieces have landed shows as single wrong elements, now and then."""
import pytest
import torch
import torch.nn.functional as F

import helpers as hp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("hwc,case", [(0, (60, 192, 32, 40, 1)), (0, (62, 128, 32, 53, 0)), (0, (100, 448, 96, 26, 0)), (0, (100, 448, 64, 26, 0)),
                                      (0, (40, 64, 64, 56, 1)), (1, (40, 192, 64, 40, 1)), (0, (40, 192, 128, 26, 0))])
def test_many_tiles(pkg, gpu, hwc, case):
    ns, Ci, Co, H, p = case
    Ho = H + 2 * p - 2
    g = torch.Generator(device=DEV).manual_seed(Ci + H)
    x = (torch.rand((ns, Ci, H, H), generator=g, device=DEV) * 2 - 1).half()
    w = ((torch.rand((Co, Ci, 3, 3), generator=g, device=DEV) * 2 - 1) * (6.0 / (9 * Ci)) ** 0.5).half()
    ref = F.conv2d(x.float(), w.float(), padding=p)
    if hwc:
        x, w, ref = (t.permute(0, 2, 3, 1).contiguous() for t in (x, w, ref))
    y = torch.empty_like(ref, dtype=torch.float16)
    a, keep = hp.conv2d_args(pkg, x, None, w, None, y, y, Ci, H, H, Co, 3, 3, Ho, Ho, (p,) * 4, (1, 1), hwc)
    gpu.ptl_set_gemm_path(5)
    try:
        for _ in range(4):
            y.fill_(7)
            torch.cuda.synchronize()
            pkg.call("ptl_conv2d_fp16_fw_batched", a, ns)
            assert gpu.ptl_sync() == 0 and gpu.ptl_last_conv_resident() == 1
            # half a unit in the last place of the result, and 9 Ci rounded fp32 additions on either side
            assert bool(((y.float() - ref).abs() <= 2.0 ** -11 * ref.abs() + 1e-4).all())
    finally:
        gpu.ptl_set_gemm_path(0)
