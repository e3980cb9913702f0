"""Channels-last convolution through the 64-deep persistent 256 x 256 kernel: 64-channel K tiles, pixel and tap
indexes by multiplication, edges, strides, dilations, biases and chunked workspaces."""

import pytest
import torch
import torch.nn.functional as F

from ntops_amd import _lib
from ntops_amd.torch import conv2d

gpu = pytest.mark.gpu


def exact_image(x, w, b, stride, pad, dil, p, q):
    cols = F.unfold(x[None].double(), w.shape[2:], padding=pad, stride=stride, dilation=dil)[0]
    out = w.double().flatten(1) @ cols
    if b is not None:
        out = out + b.double()[:, None]
    return out.view(-1, p, q)


def small_ints(g, *shape):
    """Whole numbers in -2 .. 2: products and their sums are exact in fp32, so only the output's rounding is left."""
    return torch.randint(-2, 3, shape, generator=g).float()


# (n, c, h, w, k, (r, s), stride, padding, dilation, bias): each reaches 240 tiles, or 512 small ones
CASES = [
    (240, 64, 16, 16, 256, (3, 3), 1, 1, 1, True),     # even; 9 K tiles (the last pair half empty)
    (128, 320, 18, 18, 256, (1, 1), 1, 0, 1, False),   # 1 x 1: 5 K tiles, the fewest; 324 pixels: two tiles an image
    (62, 64, 64, 48, 130, (3, 3), (2, 1), (1, 1), 1, True),  # ragged rows, stride 2 down, 1536 pixels
    (2, 64, 180, 180, 256, (3, 5), 1, (2, 4), 2, True),      # many pixels, unequal taps, dilation
    (40, 64, 28, 28, 256, (3, 3), 1, 1, 1, True),      # 160 tiles, the last of each image 16 pixels
    (128, 128, 20, 17, 256, (5, 1), 1, (2, 0), 1, False),    # element copy of the input (rows not 16 bytes)
]


@gpu
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize("case", CASES)
def test_conv_large(case, dtype):
    n, c, h, w, k, (r, s), stride, pad, dil, has_bias = case
    g = torch.Generator().manual_seed(n + c + k)
    x = small_ints(g, n, c, h, w).to(dtype)
    wt = small_ints(g, k, c, r, s).to(dtype)
    b = small_ints(g, k).to(dtype) if has_bias else None
    got = conv2d(x.cuda(), wt.cuda(), b if b is None else b.cuda(), stride=stride, padding=pad, dilation=dil)
    assert _lib.last_kernel() == "gemm_large A:K B:K conv_cl", _lib.last_kernel()
    for img in sorted({0, n // 2, n - 1}):
        exp = exact_image(x[img], wt, b, stride, pad, dil, *got.shape[2:])
        assert torch.equal(got[img].cpu(), exp.to(dtype)), f"image {img}"


@gpu
def test_conv_large_bias_forms_and_chunks():
    """A bias that is not contiguous keeps the 32-channel blocks, and a workspace that holds 120 of 241 images (two
    full chunks of the large kernel's size or not, and one image left) keeps one order of the weights for all."""
    g = torch.Generator().manual_seed(5)
    n, c, h, k = 241, 64, 16, 512
    x, wt = small_ints(g, n, c, h, h).bfloat16(), small_ints(g, k, c, 3, 3).bfloat16()
    bias = small_ints(g, 2 * k).bfloat16()
    xg, wg, bg = x.cuda(), wt.cuda(), bias.cuda()
    exp = {img: exact_image(x[img], wt, bias[::2], 1, 1, 1, h, h).bfloat16() for img in (0, 119, 120, 239, 240)}
    got = conv2d(xg, wg, bg[::2], padding=1)
    assert _lib.last_kernel() == "gemm_mfma 256x256 s4 A:K B:K even conv_cl", _lib.last_kernel()
    out = torch.full((n, k, h, h), float("nan"), dtype=torch.bfloat16, device="cuda")
    lib = _lib.load()
    geo = (c, h, h, k, 3, 3, h, h, 1, 1, 1, 1, 1, 1)
    st = lambda t: _lib.i64_array(t.stride())  # noqa: E731
    fits = lib.ntops_conv2d_workspace(_lib.BF16, 120, *geo, st(wg), st(out))
    ws = torch.empty(fits, dtype=torch.uint8, device="cuda")
    even = bg[::2].contiguous()
    rc = lib.ntops_conv2d(_lib.BF16, n, *geo, xg.data_ptr(), st(xg), wg.data_ptr(), st(wg), even.data_ptr(), 1,
                          out.data_ptr(), st(out), ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.ntops_last_error()
    assert _lib.last_kernel() == "gemm_large A:K B:K conv_cl", _lib.last_kernel()
    for img, e in exp.items():
        assert torch.equal(got[img].cpu(), e), f"strided bias, image {img}"
        assert torch.equal(out[img].cpu(), e), f"chunks, image {img}"


def test_index_division_by_multiplication():
    """The quotients the kernel takes by multiplication, over the sizes its rule accepts."""
    for q in (2, 3, 7, 56, 57, 224, 1000, 4095, 65535):
        most = ((1 << 32) - 1) // q  # pixels * q < 2^32
        m = ((1 << 32) + q - 1) // q
        assert m < 1 << 32
        n = torch.cat([torch.arange(0, min(most, 1 << 16)), most - torch.arange(1, 1 << 12),
                       torch.arange(1, most // q + 1, max(1, most // q // 4096)) * q - 1])
        n = n[(n >= 0) & (n < most)].tolist()
        assert all(v * m >> 32 == v // q for v in n)
    for r in range(1, 12):
        for s in range(1, 12):
            rs = r * s
            for d, most in ((rs, (65536 - 1) // rs), (s, rs)):
                m = (65536 + d - 1) // d
                assert all(t * m >> 16 == t // d for t in range(most)), (r, s)
