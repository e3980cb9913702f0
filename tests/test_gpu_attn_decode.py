"""GPU parity: attention of a few query rows over a long key / value cache
(the decode kernel and its merge of key slices), and the two-copy launch that
writes a step's key and value into the cache."""

import pytest
import torch

import ntops_amd
from ntops_amd import _lib
from ntops_amd.kernels.scaled_dot_product_attention import CausalVariant
from oracle import ops as O
from tests.helpers import DT_NAME, assert_close, from_np, to_np

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]

sdpa = ntops_amd.torch.scaled_dot_product_attention


def oracle(q, k, v, causal=0):
    dt = DT_NAME[q.dtype]
    return from_np(O.scaled_dot_product_attention(to_np(q), to_np(k), to_np(v), dt, None, None, causal, None,
                                                  round_p=True), dt)


# edges: one key past the smallest cache served, tiles of 32 / 64 keys with
# remainders, one and sixteen rows per key head, rows of several positions,
# head dims below the kernel's, enough heads for the one-wave blocks
@pytest.mark.parametrize("b, hq, hkv, sq, skv, d, causal", (
    (1, 2, 2, 1, 257, 128, 0),
    (2, 8, 2, 1, 1000, 128, 0),
    (1, 16, 1, 1, 4097, 128, 0),
    (2, 4, 1, 4, 769, 64, 2),
    (1, 3, 1, 5, 300, 64, 2),
    (1, 2, 1, 8, 300, 128, 1),
    (2, 8, 1, 2, 2047, 80, 2),
    (1, 4, 4, 1, 543, 8, 0),
    (3, 6, 2, 1, 1311, 120, 2),
    (32, 32, 16, 1, 259, 64, 0),
    (32, 16, 16, 1, 290, 128, 0),
))
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
def test_decode(b, hq, hkv, sq, skv, d, causal, dtype):
    g = torch.Generator().manual_seed(skv + d)
    rt = lambda *s: torch.randn(*s, generator=g).to(dtype)  # noqa: E731
    # the cache is a slice of a longer one, its heads inside its positions
    q = rt(b, hq, sq, d)
    k, v = (rt(b, skv + 7, hkv, d).transpose(1, 2)[:, :, :skv] for _ in range(2))
    variant = CausalVariant.LOWER_RIGHT if causal == 2 else None
    kg, vg = (t.transpose(1, 2).cuda().transpose(1, 2) for t in (k, v))
    got = sdpa(q.cuda(), kg, vg, is_causal=causal > 0, enable_gqa=True, causal_variant=variant)
    assert _lib.last_kernel().startswith("sdpa_decode"), _lib.last_kernel()
    assert_close(got, oracle(q, k, v, causal), 1.6e-2, 1.6e-2, "decode")
    # without a workspace the C ABI runs one block per key head: the same up
    # to the slices' fp32 sums and the rounding of P against another maximum
    out = torch.empty_like(got)
    st = lambda t: _lib.i64_array(t.stride())  # noqa: E731
    qg = q.cuda()
    _lib.check(_lib.load().ntops_sdpa(
        _lib.dtype_code(dtype), b, hq, hkv, sq, skv, d, qg.data_ptr(), st(qg), kg.data_ptr(), st(kg), vg.data_ptr(),
        st(vg), None, 0, None, causal, d ** -0.5, out.data_ptr(), st(out), _lib.stream_of(out)), "sdpa")
    assert _lib.last_kernel().endswith("split1")
    assert_close(out, oracle(q, k, v, causal), 1.6e-2, 1.6e-2, "unsplit")


# a key / value head for every CU: any cache is served, of one key up to a tile
# and past it, and rows that see no key at all (lower-right, fewer keys than
# queries) are zero
@pytest.mark.parametrize("sq, skv, causal", ((1, 1, 0), (1, 7, 0), (1, 31, 0), (2, 33, 1), (1, 64, 0), (4, 65, 2),
                                             (1, 256, 0), (16, 5, 2), (16, 1, 2), (3, 40, 1)))
@pytest.mark.parametrize("d", (64, 128))
def test_decode_short_caches(sq, skv, causal, d):
    b, h = (16, 16) if torch.cuda.get_device_properties(0).multi_processor_count <= 256 else (32, 32)
    g = torch.Generator().manual_seed(skv + d)
    q, k, v = (torch.randn(b, h, s, d, generator=g).bfloat16() for s in (sq, skv, skv))
    got = sdpa(q.cuda(), k.cuda(), v.cuda(), is_causal=causal > 0,
               causal_variant=CausalVariant(causal) if causal else None)
    assert _lib.last_kernel().startswith("sdpa_decode"), _lib.last_kernel()
    assert_close(got, oracle(q, k, v, causal), 1.6e-2, 1.6e-2, "short cache")
    if causal == 2 and sq > skv:
        assert (got[:, :, :sq - skv] == 0).all()


@pytest.mark.parametrize("b, h", ((1, 2), (8, 32)))
@pytest.mark.parametrize("causal", (0, 2))
def test_empty_cache(b, h, causal, monkeypatch):
    """No keys: zeros, with few heads and with a head for every CU, through the
    native host path, the Python one and the C ABI."""
    q = torch.randn(b, h, 1, 64, device="cuda").bfloat16()
    k = torch.empty(b, h, 0, 64, device="cuda").bfloat16()
    args = dict(is_causal=causal > 0, causal_variant=CausalVariant.LOWER_RIGHT if causal else None)
    assert (sdpa(q, k, k, **args) == 0).all()
    assert _lib.last_kernel().startswith("sdpa_fwd"), _lib.last_kernel()
    with monkeypatch.context() as mp:
        mp.setattr(_lib, "fast", None)
        assert (sdpa(q, k, k, **args) == 0).all()
    out = torch.full_like(q, float("nan"))
    st = lambda t: _lib.i64_array(t.stride())  # noqa: E731
    _lib.check(_lib.load().ntops_sdpa(
        _lib.BF16, b, h, h, 1, 0, 64, q.data_ptr(), st(q), None, st(k), None, st(k), None, 0, None, causal, 0.125,
        out.data_ptr(), st(out), _lib.stream_of(out)), "sdpa")
    assert (out == 0).all()


def test_decode_special_values():
    """NaN and infinite scores, a causal row that sees one key, and a repeated
    call (bit for bit: the slices are combined in a fixed order)."""
    q = torch.randn(1, 4, 1, 64, device="cuda").bfloat16()
    k, v = (torch.randn(1, 2, 900, 64, device="cuda").bfloat16() for _ in range(2))
    a = sdpa(q, k, v, enable_gqa=True)
    assert torch.equal(a, sdpa(q, k, v, enable_gqa=True))
    q[0, 1, 0, 3] = float("nan")
    got = sdpa(q, k, v, enable_gqa=True)
    assert got[0, 1].isnan().all() and torch.equal(got[0, [0, 2, 3]], a[0, [0, 2, 3]])
    # a score of -inf drops its key; one of every key leaves the row as torch's CPU kernel does: zero
    q[0, 1, 0, 3] = 0
    k2 = k.clone()
    k2[:, 0, :, 5] = float("-inf")
    q[0, :, 0, 5] = 1.0
    assert (sdpa(q, k2, v, enable_gqa=True)[0, :2] == 0).all()
    # upper-left: the first row sees the first key alone
    q = torch.randn(1, 1, 16, 64, device="cuda").half()
    k, v = (torch.randn(1, 1, 300, 64, device="cuda").half() for _ in range(2))
    got = sdpa(q, k, v, is_causal=True)
    assert torch.isfinite(got).all()
    assert_close(got[:, :, :1], v[:, :, :1].cpu(), 1e-3, 1e-3, "row 0 sees key 0 alone")


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float32, torch.float64, torch.int8))
@pytest.mark.parametrize("shape", ((2, 3, 1, 64), (3, 5, 7), (1,), (2, 0, 4)))
def test_copy2_matches_two_copies(dtype, shape):
    lib = _lib.load()
    mk = lambda: (torch.randn([n + 2 for n in shape], device="cuda") * 50).to(dtype)  # noqa: E731
    view = lambda t: t[tuple(slice(0, n) for n in shape)]  # noqa: E731
    x0, y0, x1, y1 = (view(mk()) for _ in range(4))
    x1 = x1.contiguous()
    st = lambda t: _lib.i64_array(t.stride())  # noqa: E731

    def copy2(a, b, c, d):
        _lib.check(lib.ntops_copy2(_lib.dtype_code(dtype), len(shape), _lib.i64_array(shape), a.data_ptr(), st(a),
                                   b.data_ptr(), st(b), c.data_ptr(), st(c), d.data_ptr(), st(d), _lib.stream_of(b)),
                   "copy2")

    copy2(x0, y0, x1, y1)
    assert torch.equal(y0, x0) and torch.equal(y1, x1)
    # chained: the second copy reads what the first wrote, and both may have one destination
    copy2(x1, y0, y0, y1)
    assert torch.equal(y0, x1) and torch.equal(y1, x1)
    copy2(x1, y0, x0, y0)
    assert torch.equal(y0, x0)
