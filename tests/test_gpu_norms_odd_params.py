"""GPU parity: norms on rows that are not 16-byte runs, whose weight and bias
are loaded at any element's address -- over every launch shape (packs per lane
x waves per row), widths one element around a pack, rows shorter than a pack,
fp32 parameters of 16-bit rows, and widths whose parameters are larger than
the LDS a block may take."""

import pytest
import torch

import ntops_amd

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]

T = ntops_amd.torch
TOL = {torch.float32: 2e-5, torch.float16: 2e-3, torch.bfloat16: 1.6e-2}  # of values around 1


@pytest.mark.parametrize("cols", (1, 3, 7, 9, 513, 1025, 2049, 4100, 8191, 16389, 20001, 40003, 65529))
@pytest.mark.parametrize("dtype, pdtype", ((torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32),
                                           (torch.float32, torch.float32)))
def test_norms_with_parameters(cols, dtype, pdtype):
    g = torch.Generator().manual_seed(cols)
    x, res = (torch.randn(5, cols, generator=g).to(dtype).cuda() for _ in range(2))
    w, b = ((1 + 0.5 * torch.randn(cols, generator=g)).to(pdtype).cuda() for _ in range(2))
    tol = TOL[dtype]
    d = x.double()
    rms = d * torch.rsqrt(d.square().mean(-1, keepdim=True) + 1e-6)
    c = d - d.mean(-1, keepdim=True)
    ln = c * torch.rsqrt(c.square().mean(-1, keepdim=True) + 1e-5)
    h = (x + res).double()
    arms = h * torch.rsqrt(h.square().mean(-1, keepdim=True) + 1e-6)
    close = lambda got, exp: torch.testing.assert_close(got.double(), exp, rtol=tol, atol=tol)  # noqa: E731
    close(T.rms_norm(x, (cols,), w, 1e-6), rms * w.double())
    close(T.rms_norm(x, (cols,), None, 1e-6), rms)
    y, r = T.add_rms_norm(x, res, (cols,), w, 1e-6)
    assert torch.equal(r, x + res)
    close(y, arms * w.double())
    close(T.layer_norm(x, (cols,), w, b), ln * w.double() + b.double())
    close(T.layer_norm(x, (cols,), w), ln * w.double())
    close(T.layer_norm(x, (cols,), None, b), ln + b.double())
