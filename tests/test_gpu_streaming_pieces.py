"""Copies, fills, sums and casts in pieces of 16 bytes: exact at any size and start, with nothing written beside the result."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def room(n, off, dtype, seed):
    """A tensor of n values that starts `off` elements behind an aligned place, with sixteen guards behind it; values of all kinds."""
    g = torch.Generator().manual_seed(seed)
    t = ((torch.rand(off + n + 16, generator=g) - 0.5) * 8).to(dtype)
    special = torch.tensor([float("inf"), -float("inf"), float("nan"), 0.0, -0.0, 6e-8, 65504.0, -1e-5]).to(dtype)
    t[off:off + n:5] = special.repeat((n + 39) // 40)[:len(t[off:off + n:5])]
    return t.cuda()


@pytest.mark.parametrize("n", [1, 3, 4, 7, 8, 9, 15, 2047, 2048, 4099, 1210367])
@pytest.mark.parametrize("offs", [(0, 0, 0), (1, 1, 1), (2, 0, 3), (0, 5, 1)])
def test_streaming(pkg, gpu, n, offs):
    for name, src, dst, args in (("copy", 32, 32, "CopyArgs"), ("set_to_value", 32, 32, "SetToValueArgs"), ("set_to_value_fp16", 16, 16, "SetToValueArgsFp16"),
                                 ("vect_sum", 32, 32, "VectSumArgs"), ("vect_sum_fp16", 16, 16, "VectSumArgs"), ("cast_fp16_tensor_to_fp32", 16, 32, "CastArgs"),
                                 ("cast_fp32_tensor_to_fp16", 32, 16, "CastArgs")):
        kind = {16: torch.float16, 32: torch.float32}
        x, y, z = room(n, offs[0], kind[src], n), room(n, offs[1], kind[src], n + 1), room(n, offs[2], kind[dst], n + 2)
        want, (xs, ys) = z.clone(), (t[o:o + n] for t, o in ((x, offs[0]), (y, offs[1])))
        a = getattr(pkg, args)()
        at = lambda t, o: t.data_ptr() + o * t.element_size()
        if args == "CopyArgs":
            a.from_, a.to, a.size, res = at(x, offs[0]), at(z, offs[2]), n, xs
        elif args.startswith("SetToValue"):
            res = torch.full((n,), 0.1, device="cuda", dtype=kind[dst])
            a.to, a.size = at(z, offs[2]), n
            a.value = 0.1 if dst == 32 else int(np.float16(0.1).view(np.uint16))
        elif args == "VectSumArgs":
            a.op_1, a.op_2, a.dest, a.size, res = at(x, offs[0]), at(y, offs[1]), at(z, offs[2]), n, xs + ys
        else:
            a.source, a.destination, a.size, res = at(x, offs[0]), at(z, offs[2]), n, xs.to(kind[dst])
        want[offs[2]:offs[2] + n] = res
        torch.cuda.synchronize()
        pkg.call(name, a)
        assert gpu.ptl_sync() == 0
        np.testing.assert_array_equal(z.cpu().numpy(), want.cpu().numpy(), err_msg=name)
        if args == "VectSumArgs":  # onto an operand, as gradients are added up
            a.dest = at(y, offs[1])
            pkg.call(name, a)
            assert gpu.ptl_sync() == 0
            np.testing.assert_array_equal(ys.cpu().numpy(), res.cpu().numpy(), err_msg=name)
