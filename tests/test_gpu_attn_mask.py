"""GPU parity: masked attention on the matrix cores over the mask's load paths
-- interior tiles by wide loads at any alignment, the partial last tile by runs
or elements, tiles the mask leaves open -- and the scale's sign."""

import pytest
import torch

import ntops_amd
from ntops_amd import _lib
from oracle import ops as O
from tests.helpers import DT_NAME, assert_close, from_np, to_np

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]

sdpa = ntops_amd.torch.scaled_dot_product_attention


def oracle(q, k, v, mask, scale=None):
    dt = DT_NAME[q.dtype]
    m = None if mask is None else to_np(mask.contiguous())
    return from_np(O.scaled_dot_product_attention(to_np(q), to_np(k), to_np(v), dt, m,
                                                  None if mask is None else DT_NAME[mask.dtype], 0, scale,
                                                  round_p=True), dt)


# one tile exactly, one key past and short of a tile, several tiles with odd
# remainders; rows of a wider mask starting at an odd element
@pytest.mark.parametrize("skv", (1, 63, 64, 65, 130, 191, 256, 333))
@pytest.mark.parametrize("mask_dtype", (torch.bool, torch.float16, torch.bfloat16, torch.float32))
@pytest.mark.parametrize("offset", (0, 1, 4))
def test_mask_loads(skv, mask_dtype, offset):
    g = torch.Generator().manual_seed(skv + offset)
    dtype, b, h, sq, d = torch.float16 if skv % 2 else torch.bfloat16, 2, 3, 70, 64
    q, k, v = (torch.randn(b, h, s, d, generator=g).to(dtype) for s in (sq, skv, skv))
    keep = torch.rand(b, 1, sq, skv + offset + 3, generator=g) > 0.3
    keep[:, :, :40, :128] = True   # open tiles beside mixed ones
    keep[0, :, 5] = False          # a row with no key
    keep[1, :, 7, 64:] = False
    mask = keep if mask_dtype == torch.bool else torch.where(keep, 0.25 * torch.rand(keep.shape, generator=g).round(),
                                                             float("-inf")).to(mask_dtype)
    mask = mask[..., offset:offset + skv]
    wide = torch.zeros(b, 1, sq, skv + offset + 3).to(mask_dtype).cuda()
    wide[..., offset:offset + skv] = mask.cuda()
    got = sdpa(q.cuda(), k.cuda(), v.cuda(), attn_mask=wide[..., offset:offset + skv])
    assert _lib.last_kernel().startswith("sdpa_fwd d64 mask"), _lib.last_kernel()
    full = mask.expand(b, h, sq, skv)
    assert_close(got, oracle(q, k, v, full), 1.6e-2, 1.6e-2, "mask")
    assert (got[0, :, 5] == 0).all()
    # the same under a padding mask that no query row moves
    pad = mask[:, :, 9:10]
    got = sdpa(q.cuda(), k.cuda(), v.cuda(), attn_mask=wide[:, :, 9:10, offset:offset + skv])
    assert_close(got, oracle(q, k, v, pad.expand(b, h, sq, skv)), 1.6e-2, 1.6e-2, "padding")


@pytest.mark.parametrize("scale", (-0.2, 0.0, 3.0))
@pytest.mark.parametrize("masked", (False, True))
def test_scale_signs(scale, masked):
    g = torch.Generator().manual_seed(7)
    q, k, v = (torch.randn(1, 2, s, 128, generator=g).bfloat16() for s in (20, 150, 150))
    mask = None
    if masked:
        mask = torch.where(torch.rand(20, 150, generator=g) > 0.5, 0.0, -1.5)
        mask[:, 30:40] = float("-inf")
    got = sdpa(q.cuda(), k.cuda(), v.cuda(), attn_mask=None if mask is None else mask.cuda(), scale=scale)
    exp = oracle(q, k, v, None if mask is None else mask.expand(1, 2, 20, 150), scale)
    assert_close(got, exp, 1.6e-2, 1.6e-2, f"scale {scale}")


# the large finite values that programs close keys with; tiles of 64 keys
@pytest.mark.parametrize("value, mask_dtype", [(-65504.0, torch.float16)] + [
    (value, dt) for value in (-65504.0, -1e6, -1e9, -1e10, -1e30) for dt in (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
@pytest.mark.parametrize("d", (64, 80, 128))
def test_large_finite_mask_values(value, mask_dtype, dtype, d):
    """Rows whose first or middle tile is closed by a finite value are as if it
    were closed altogether (exp(-65504 + a few tens) is 0 in 64 bits too).  A
    row closed throughout has all its scores at the value: with a zero query
    they are equal, so the row is the mean of V; with any other the values are
    too coarse for the scores (half a unit and more from 1e6 on), but P still
    sums to 1 and the row lies among V's."""
    g = torch.Generator().manual_seed(d)
    b, h, sq, skv = 2, 2, 72, 200
    q, k, v = (torch.randn(b, h, s, d, generator=g).to(dtype) for s in (sq, skv, skv))
    mask = torch.zeros(b, 1, sq, skv)
    mask[:, :, 0:24, :64] = value      # left padding of a tile
    mask[:, :, 24:40, 64:128] = value  # a tile in the middle
    mask[:, :, 20:32, 192:] = value    # the last, partial one
    mask[:, :, 56:] = value            # rows closed throughout
    q[:, :, 56:64] = 0
    mask = mask.to(mask_dtype)
    got = sdpa(q.cuda(), k.cuda(), v.cuda(), attn_mask=mask.cuda()).cpu()
    assert _lib.last_kernel().startswith("sdpa_fwd"), _lib.last_kernel()
    exp = oracle(q, k, v, mask.expand(b, h, sq, skv))
    assert_close(got[:, :, :56], exp[:, :, :56], 1.6e-2, 1.6e-2, "some tiles closed")
    mean = v.double().mean(2, keepdim=True)
    # the sum of 200 equal P is exact and so is each P V product; what is left
    # is the fp32 sums (far below) and one rounding of the result
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert_close(got[:, :, 56:64], mean.expand(b, h, 8, d), ulp, 1e-5, "equal scores")
    # P is rounded (half an ulp of it each way), its sum is not
    lo, hi = v.amin(2, keepdim=True).double(), v.amax(2, keepdim=True).double()
    slack = 2 * ulp * v.abs().amax().double()
    rest = got[:, :, 64:].double()
    assert ((rest >= lo - slack) & (rest <= hi + slack)).all()


@pytest.mark.parametrize("sq, skv, d, causal", ((20, 150, 128, 0), (300, 190, 64, 2), (190, 300, 80, 1)))
@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
def test_zero_scale_stays_on_the_matrix_cores(sq, skv, d, causal, dtype):
    """A zero scale without a mask: equal scores over the keys a row sees, none
    for a row that sees no key, NaN where a query or key is not finite."""
    g = torch.Generator().manual_seed(sq)
    q, k, v = (torch.randn(1, 2, s, d, generator=g).to(dtype) for s in (sq, skv, skv))
    args = dict(scale=0.0, is_causal=causal > 0, causal_variant=causal or None)
    got = sdpa(q.cuda(), k.cuda(), v.cuda(), **args)
    assert _lib.last_kernel().startswith("sdpa_fwd"), _lib.last_kernel()
    i, j = torch.arange(sq)[:, None], torch.arange(skv)[None]
    seen = (j <= i + (skv - sq if causal == 2 else 0)) if causal else torch.ones(sq, skv, dtype=torch.bool)
    p = seen.double() / seen.sum(1, keepdim=True).clamp_min(1)
    # P = 1 exactly: the fp32 sums and one rounding of the result
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert_close(got, p @ v.double(), ulp, 1e-5, "zero scale")
    q[0, 0, 7, 5] = float("-inf")
    k[0, 1, skv // 2, 3] = float("nan")
    bad = sdpa(q.cuda(), k.cuda(), v.cuda(), **args).cpu()
    rows = torch.zeros(1, 2, sq, dtype=torch.bool)
    rows[0, 0, 7] = seen[7].any()
    rows[0, 1] = seen[:, skv // 2]
    assert bad[rows].isnan().all() and torch.equal(bad[~rows], got.cpu()[~rows])
