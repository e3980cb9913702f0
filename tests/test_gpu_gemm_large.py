"""GPU parity: the persistent 256 x 256 GEMM kernel over its edges -- operand
layouts, K tails of a 128-deep pair of K tiles, partial tiles, output rows at
any 2-byte offset, column-major outputs, a bias row, alpha, batches.
Small-integer operands make every fp32 sum exact, so each output equals the
double-precision product rounded once."""

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


def major(t, layout):
    """t with its last (N) or first (T) axis contiguous."""
    return t if layout == "N" else t.transpose(-1, -2).contiguous().transpose(-1, -2)


# even tiles with three pairs of K tiles; K one chunk past a pair and one
# short of one; one row and column past a tile; a single row and column of
# tiles; odd N (K-major B runs as it is, an N-major B is padded)
@pytest.mark.parametrize("m, n, k", ((4096, 3840, 384), (4104, 4112, 264), (3848, 4096, 504), (65288, 256, 328),
                                     (256, 61448, 296), (4097, 4099, 512), (2048, 16387, 776)))
@pytest.mark.parametrize("layout", ("NN", "NT", "TN", "TT"))
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
def test_large_tiles_exact(m, n, k, layout, dtype):
    a, b, bias = ints(m, k, seed=1, dtype=dtype), ints(k, n, seed=2, dtype=dtype), ints(n, seed=3, dtype=dtype)
    exp = a.double() @ b.double()
    ag, bg = major(a, layout[0]), major(b, layout[1])
    got = T.mm(ag, bg)
    assert _lib.last_kernel().startswith("gemm_large "), _lib.last_kernel()
    assert torch.equal(got, exp.float().to(dtype))
    assert torch.equal(T.addmm(bias, ag, bg), (exp + bias.double()).float().to(dtype))
    got = T.addmm(bias, ag, bg, beta=0.5, alpha=2.0)
    assert torch.equal(got, (2 * exp + 0.5 * bias.double()).float().to(dtype))
    assert torch.equal(T.addmm(bias, ag, bg, beta=0, alpha=0.25), (exp / 4).float().to(dtype))


@pytest.mark.parametrize("form", ("odd stride", "column-major", "offset"))
def test_large_tiles_output_views(form):
    """Outputs inside a larger buffer: what lies between the rows stays."""
    m, n, k = 4000, 4112, 320
    dtype = torch.bfloat16
    a, b = ints(m, k, seed=4, dtype=dtype), ints(k, n, seed=5, dtype=dtype)
    exp = (a.double() @ b.double()).float().to(dtype)
    if form == "column-major":
        big = torch.full((n + 3, m + 5), 7.0, dtype=dtype, device="cuda")
        out = big[1:1 + n, 2:2 + m].t()
    else:
        big = torch.full((m + 2, n + (5 if form == "odd stride" else 8)), 7.0, dtype=dtype, device="cuda")
        out = big[1:1 + m, 3:3 + n]
    T.addmm(torch.zeros(n, dtype=dtype, device="cuda"), a, b, out=out)
    assert _lib.last_kernel().startswith("gemm_large "), _lib.last_kernel()
    assert torch.equal(out, exp)
    kept = big.float().sum() - out.float().sum()
    assert kept.item() == 7.0 * (big.numel() - out.numel())


def test_large_tiles_batch_and_full_c():
    """A batch (tiles of different members on one block), and a full C matrix,
    which takes the kernel that loads it in its epilogue."""
    dtype = torch.float16
    a, b = ints(5, 2000, 264, seed=6, dtype=dtype), ints(5, 264, 2056, seed=7, dtype=dtype)
    exp = torch.stack([x.double() @ y.double() for x, y in zip(a, b)]).float().to(dtype)
    assert torch.equal(T.bmm(a, b), exp)
    assert _lib.last_kernel().startswith("gemm_large "), _lib.last_kernel()
    a, b, c = ints(4096, 512, seed=8, dtype=dtype), ints(512, 4096, seed=9, dtype=dtype), ints(4096, 4096, seed=10, dtype=dtype)
    exp = a.double() @ b.double()
    for cv in (c, c[:, :1]):
        assert torch.equal(T.addmm(cv, a, b), (exp + cv.double()).float().to(dtype))
        assert _lib.last_kernel() == "gemm_mfma 256x256 s4 A:K B:N even", _lib.last_kernel()


@pytest.mark.parametrize("m, n, k, layout, large", (
    (2560, 3328, 512, "NN", True),     # 520 small tiles: past the two a CU holds
    (2553, 3321, 512, "NT", True),     # the same, ragged
    (2560, 3328, 520, "TN", True),
    (2560, 3328, 504, "NT", False),    # too short for it
    (2050, 4096, 512, "NT", True),     # 544, the last row of large tiles nearly empty
    (2050, 4096, 1024, "NN", True),
    (1152, 8192, 520, "TN", True),     # 576, the last row of large tiles half empty
    (2050, 4096, 504, "NN", False),
    (2048, 4096, 1024, "NT", True),    # 512: one full round, K-major B
    (2048, 4096, 1016, "NT", False),
    (2048, 4096, 2048, "NN", True),    # N-major B from K = 2048
    (2048, 4096, 2040, "NN", False),
    (2048, 4096, 2048, "TN", False),   # M-major A
    (1792, 4096, 2048, "NT", False),   # 448: seven eighths of a round, not past it
    (384, 19456, 2048, "NT", False),   # 456, large tiles a quarter empty
))
def test_large_tiles_below_a_round(m, n, k, layout, large):
    """Which products of fewer than 240 tiles take the kernel, and their sums (256 CUs)."""
    dtype = torch.bfloat16
    a, b, bias = ints(m, k, seed=11, dtype=dtype), ints(k, n, seed=12, dtype=dtype), ints(n, seed=13, dtype=dtype)
    exp = a.double() @ b.double()
    ag, bg = major(a, layout[0]), major(b, layout[1])
    got = T.mm(ag, bg)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert _lib.last_kernel().startswith("gemm_large " if large else "gemm_mfma 128x128"), _lib.last_kernel()
    assert torch.equal(got, exp.float().to(dtype))
    assert torch.equal(T.addmm(bias, ag, bg), (exp + bias.double()).float().to(dtype))
