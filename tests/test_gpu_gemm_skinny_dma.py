"""GPU parity: products of up to 16 rows that stream a large K-major B by DMA
-- column slices of 16, 32 and 64, K tails of a step and of the waves' turns,
partial column slices, a bias or C, alpha, column-major outputs, batches, a
padded weight.  Small-integer operands make every fp32 sum exact, so each
output equals the double-precision product rounded once."""

import pytest
import torch

import ntops_amd
from ntops_amd import _lib

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]

T = ntops_amd.torch


def ints(*shape, seed, dtype):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-8, 9, shape, generator=g, device="cuda").to(dtype)


# (n, k, slice): n one past, one short of and equal to whole slices; k one
# chunk past and one short of whole steps, and steps the four waves do not
# share evenly.  96 MiB of 16-bit B are 50.4 M elements, of fp32 25.2 M.
@pytest.mark.parametrize("m", (1, 7, 16))
@pytest.mark.parametrize("dtype, n, k, cols", (
    (torch.bfloat16, 3009, 16776, 16), (torch.float16, 16, 3146000, 16), (torch.bfloat16, 6145, 8200, 32),
    (torch.float16, 12287, 4104, 64), (torch.bfloat16, 50257, 1016, 64), (torch.float32, 3001, 8396, 16),
    (torch.float32, 6144, 4100, 32), (torch.float32, 50257, 508, 64)))
def test_skinny_dma_exact(m, dtype, n, k, cols):
    x, w, bias = ints(m, k, seed=1, dtype=dtype), ints(n, k, seed=2, dtype=dtype).t(), ints(n, seed=3, dtype=dtype)
    exp = x.double() @ w.double()
    assert exp.abs().max() < 1 << 24
    got = T.mm(x, w)
    assert _lib.last_kernel() in (f"gemm_skinny m16 n{cols} B:K dma", f"gemm_skinny_f32 m16 n{cols} B:K dma")
    assert torch.equal(got, exp.float().to(dtype))
    assert torch.equal(T.addmm(bias, x, w, beta=0.5, alpha=2.0), (2 * exp + 0.5 * bias.double()).float().to(dtype))
    out = torch.full((n, m + 3), 7.0, dtype=dtype, device="cuda")
    T.mm(x, w, out=out.t()[1:1 + m])
    assert torch.equal(out.t()[1:1 + m], exp.float().to(dtype)) and bool((out[:, m + 1:] == 7).all())


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float32))
def test_skinny_dma_batch_and_padded_weight(dtype):
    b, m, n, k = 3, 5, 4099, 4104
    x = ints(b, m, k, seed=4, dtype=dtype)
    room = ints(b, n + 2, k + 24, seed=5, dtype=dtype)
    room[:, n:], room[:, :, k:] = float("nan"), float("nan")  # what lies past the weight is not read into a sum
    w = room[:, :n, :k].transpose(1, 2)
    exp = torch.stack([x[i].double() @ w[i].double() for i in range(b)])
    got = T.bmm(x, w)
    assert _lib.last_kernel().endswith("B:K dma"), _lib.last_kernel()
    assert torch.equal(got, exp.float().to(dtype))
