"""Shallow pointwise products over a batch, a resident panel and streamed column tiles: depths that end anywhere in their
slabs, rows that end anywhere in their panels, images that end anywhere in their tiles, against fp32 products."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("b,c,co,h,w", [(90, 5, 9, 11, 17), (43, 31, 64, 17, 19), (44, 33, 65, 17, 19), (30, 65, 130, 19, 31),
                                        (60, 97, 63, 16, 17), (52, 129, 24, 17, 19), (45, 193, 31, 17, 19), (2, 256, 66, 93, 95),
                                        (300, 32, 257, 3, 3)])
def test_pointwise_stream(pkg, gpu, dt, b, c, co, h, w):
    tdt = torch.float32 if dt == "fp32" else torch.float16
    r = lambda *s: (torch.rand(*s, device=DEV) - 0.5).to(tdt)
    # (one element into their buffers: rows start anywhere)
    place = lambda t: torch.cat([torch.full((1,), float("nan"), device=DEV, dtype=tdt), t.flatten()])[1:].view(t.shape)
    x, wt, dy = place(r(b, c, h, w)), place(r(co, c)), place(r(b, co, h, w))
    y, dx = place(torch.zeros_like(dy)), place(torch.zeros_like(x))
    a = pkg.PointWiseConvArgs()
    keep = [pkg.blob(x, dx, c, h, w), pkg.blob(wt, None, c, 1, 1, co * c), pkg.blob(y, dy, co, h, w)]
    a.input, a.coeff, a.output = [pkg.structs.C.pointer(k) for k in keep]
    pkg.call("ptl_conv_pw_%s_fw_batched" % dt, a, b)
    pkg.call("ptl_conv_pw_%s_ig_batched" % dt, a, b)
    assert gpu.ptl_sync() == 0
    want_y = torch.matmul(wt.double(), x.double().view(b, c, -1)).view(dy.shape)
    want_dx = torch.matmul(wt.double().t().contiguous(), dy.double().view(b, co, -1)).view(x.shape)
    for got, want in ((y, want_y), (dx, want_dx)):
        assert float((got.double() - want).abs().max()) <= (2e-3 if dt == "fp16" else 1e-5) * float(want.abs().max())
