"""The 64 -> 64 convolution with tiles of 4, of 8 and, forward, of 16 rows
(chosen by the number of tiles): images one row and column beside multiples of
the tiles, and batches on either side of the choice, against a plain FP32 convolution of the
same BF16 operands on the CPU."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# tiles of 4 rows x 32 columns: one; one and a remainder; 256 and 264 of them
# (a round of the card's 256 CUs and one more), then several rounds; 256
# full tiles of 16 rows, forward in one round of them, and as many with a row
# and two columns missing in each image
SHAPES = [(1, 3, 5), (1, 4, 32), (1, 5, 33), (2, 9, 65), (1, 128, 256), (1, 132, 256),
          (5, 129, 129), (32, 64, 64), (32, 63, 62)]


@pytest.mark.parametrize("shape", SHAPES)
def test_conv64_tile_heights(shape):
    import torch

    from pararealml_amd import _native as nat

    b, h, w = shape
    print(f"case: conv64 rows {shape}", flush=True)
    gen = torch.Generator().manual_seed(h * w)
    bf = lambda *s: torch.randn(*s, generator=gen).bfloat16()  # noqa: E731
    x, wk, zp = bf(b, h, w, 64), bf(9, 64, 64) * 0.05, bf(b, h, w, 64)
    bias = torch.randn(64, generator=gen)
    # wk[tap][n][k]: output channel n from input channel k
    kernel = wk.float().reshape(3, 3, 64, 64).permute(2, 3, 0, 1)
    ref = torch.nn.functional.conv2d(x.float().permute(0, 3, 1, 2), kernel, padding=1)
    ref = ref.permute(0, 2, 3, 1)
    lib, st = nat.device_lib(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    xd, wd, zd, bd = x.cuda(), wk.contiguous().cuda(), zp.cuda(), bias.cuda()
    z, a = torch.empty_like(xd), torch.empty_like(xd)
    nat.check(lib.pml_conv64(0, xd.data_ptr(), wd.data_ptr(), bd.data_ptr(), None, z.data_ptr(),
                             a.data_ptr(), b, h, w, st))
    # one BF16 rounding (2^-9) of the result and the FP32 sum of 576 products
    scale = float(ref.abs().max())
    close = dict(rtol=2.0**-8, atol=576 * 2.0**-23 * scale)
    want = ref + bias
    np.testing.assert_allclose(z.float().cpu(), want, **close)
    gelu = torch.nn.functional.gelu(want, approximate="tanh")
    np.testing.assert_allclose(a.float().cpu(), gelu, rtol=2.0**-7, atol=1e-5 * scale)
    nat.check(lib.pml_conv64(1, xd.data_ptr(), wd.data_ptr(), None, zd.data_ptr(), None,
                             a.data_ptr(), b, h, w, st))
    zr = zp.float().requires_grad_(True)
    torch.nn.functional.gelu(zr, approximate="tanh").backward(ref)
    np.testing.assert_allclose(a.float().cpu(), zr.grad, rtol=2.0**-7, atol=1e-4 * scale)
