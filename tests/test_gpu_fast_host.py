"""The wrappers' native host path against their Python path: the same results
bit for bit over the forms each op accepts, the same errors for those it
refuses, and None (the Python path) for tensors that are not plain."""

import collections
import ctypes
import itertools
from concurrent.futures import ThreadPoolExecutor

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import ntops_amd
from ntops_amd import _lib

T = ntops_amd.torch


def test_native_path_leaves_other_tensors_to_python():
    """CPU tensors, subclasses and non-tensors are not served natively."""
    if _lib.fast is None:
        pytest.skip("the extension is not built")
    _lib.load()
    x = torch.randn(4, 8)

    class Sub(torch.Tensor):
        pass

    for t in (x, x.as_subclass(Sub), 3, None):
        assert _lib.fast.unary(_lib.UNARY_SILU, t) is None
        assert _lib.fast.softmax(t, -1) is None
        assert _lib.fast.rms_norm(t, (8,), None, 1e-6) is None
        assert _lib.fast.layer_norm(t, (8,), None, None, 1e-5) is None
        assert _lib.fast.add_rms_norm(t, t, (8,), None, 1e-6) is None
        assert _lib.fast.mm(t, t) is None
        assert _lib.fast.addmm(t, t, t, 1, 1) is None
        assert _lib.fast.sdpa(t, t, t, None, 0, None, False, None, None, None, None) is None


def forms():
    """(name, call) of every op over layouts, dtypes, shapes and arguments."""
    def r(*s, dtype=torch.bfloat16):
        g = torch.Generator().manual_seed(sum(s) + len(s))
        return torch.randn(*s, generator=g).to(dtype).cuda()

    for dtype in (torch.float32, torch.float16, torch.bfloat16):
        u = lambda *s, dtype=dtype: r(*s, dtype=dtype)  # noqa: E731
        for x in (u(5, 64), u(64, 6).t(), u(3, 4, 40)[:, :, 3:35], u(0, 16), u(7), u(2, 8, 64).unsqueeze(1)):
            yield "silu", lambda x=x: T.silu(x)
            yield "gelu", lambda x=x: T.gelu(x, approximate="tanh")
            for dim in (0, -1, x.dim()):
                yield "softmax", lambda x=x, dim=dim: T.softmax(x, dim)
            c = x.shape[-1]
            for w in (None, u(c), u(c, dtype=torch.float32), u(1, c)[0], u(2 * c)[::2], u(1), u(c + 1)):
                yield "rms_norm", lambda x=x, w=w, c=c: T.rms_norm(x, (c,), w, 1e-6)
                yield "rms_norm int", lambda x=x, w=w, c=c: T.rms_norm(x, c, w)
                yield "layer_norm", lambda x=x, w=w, c=c: T.layer_norm(x, [c], w, w)
                yield "add_rms_norm", lambda x=x, w=w, c=c: T.add_rms_norm(x, x * 2, (c,), w)
            yield "shape", lambda x=x, c=c: T.rms_norm(x, (c + 1,))
        x3 = u(6, 5, 8)
        yield "norm of two dims", lambda x=x3, w=u(5, 8): T.layer_norm(x, (5, 8), w)
        yield "eps", lambda x=x3: T.rms_norm(x, (8,), None, "no")
        for (m, k, n), lay in itertools.product(((1, 64, 48), (9, 128, 40), (70, 24, 33), (5, 20, 16), (300, 256, 264)),
                                                ("NN", "NT", "TN")):
            a = u(m, k) if lay[0] == "N" else u(k, m).t()
            b = u(k, n) if lay[1] == "N" else u(n, k).t()
            # (K-major rows of whole 16-byte runs are what the native path takes)
            kind = "mm odd k" if k % (4 if dtype == torch.float32 else 8) else "mm " + lay
            yield kind, lambda a=a, b=b: T.mm(a, b)
            for cname, c in (("row", u(n)), ("full", u(m, n)), ("column", u(m, 1)), ("row", u(1, n)), ("scalar", u(1)),
                             ("transposed", u(n, m).t()), ("mismatch", u(n + 1))):
                yield "addmm " + cname, lambda a=a, b=b, c=c: T.addmm(c, a, b, beta=0.5, alpha=2)
        yield "mm mismatch", lambda: T.mm(u(4, 16), u(24, 32))
        yield "mm dtypes", lambda: T.mm(u(4, 16), u(16, 32).double())
        for hq, hk, d in ((4, 4, 64), (4, 2, 128), (3, 3, 20)):
            q, k, v = u(2, hq, 5, d), u(2, hk, 300, d), u(2, hk, 300, d)
            yield "sdpa", lambda q=q, k=k, v=v: T.scaled_dot_product_attention(q, k, v, enable_gqa=True)
            yield "sdpa causal", lambda q=q, k=k, v=v: T.scaled_dot_product_attention(
                q.transpose(1, 2).contiguous().transpose(1, 2), k, v, is_causal=True, enable_gqa=True, scale=0.3,
                causal_variant=2)
            for mname, m in (("bool", r(5, 300) > 0), ("own dtype", u(2, 1, 1, 300)),
                             ("f32", r(2, hq, 5, 300, dtype=torch.float32)), ("mismatch", r(4, 300) > 0)):
                yield "sdpa mask " + mname, lambda q=q, k=k, v=v, m=m: T.scaled_dot_product_attention(
                    q, k, v, attn_mask=m, enable_gqa=True)
            yield "sdpa heads", lambda q=q, k=k, v=v: T.scaled_dot_product_attention(q[:, :1], k, v)
            yield "sdpa 3-D", lambda q=q, k=k, v=v: T.scaled_dot_product_attention(q[0], k[0], v[0], enable_gqa=True)

            def cached(q=q, k=k, v=v):
                k, v = k.clone(), v.clone()
                o = T.scaled_dot_product_attention(
                    q, k, v, enable_gqa=True, present_key=k[:, :, :1] * 2, present_value=v[:, :, 1:2].clone(),
                    present_key_slot=k[:, :, 7:8], present_value_slot=v[:, :, 299:])
                return o, k, v
            yield "sdpa cache", cached
        for d, tw in ((64, 64), (64, 32), (24, 24)):
            q, k, s, c = u(2, 9, 4, d), u(2, 9, 2, d), u(9, tw), u(11, tw)
            for inter in (False, True):
                yield "rope " + ("interleaved" if inter else "half"), lambda q=q, k=k, s=s, c=c, i=inter: T.rotary_position_embedding_qk(q, k, s, c, i)
            yield "rope f32 tables" if dtype != torch.float32 else "rope half", lambda q=q, k=k, s=s, c=c: T.rotary_position_embedding_qk(
                q.transpose(0, 1), k.transpose(0, 1), s.float(), c.float(), False)


def outcome(call):
    try:
        r = call()
    except Exception as e:  # noqa: BLE001 -- the outcome is what is compared
        return type(e), str(e)
    return r if isinstance(r, tuple) else (r,)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_native_and_python_paths_agree(monkeypatch):
    assert _lib.fast is not None, "the extension is not built"
    served, native = 0, collections.Counter()

    class Counting:
        """The extension, counting per form and function the calls it serves."""

        def __getattr__(self, fn):
            def call(*args):
                r = getattr(fast, fn)(*args)
                if r is not None:
                    hits.append(fn)
                    native[name] += 1
                    native["fast." + fn] += 1
                return r
            return call

    fast = _lib.fast
    for name, call in forms():
        hits = []
        with monkeypatch.context() as mp:
            mp.setattr(_lib, "fast", Counting())
            got = outcome(call)
        with monkeypatch.context() as mp:
            mp.setattr(_lib, "fast", None)
            exp = outcome(call)
        assert _lib.fast is fast
        if isinstance(exp[0], type):
            assert got == exp, (name, got, exp)
            assert not hits, (name, "refused in Python, served natively")
            continue
        assert not isinstance(got[0], type), (name, got)
        served += 1
        for a, b in zip(got, exp):
            assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride(), name
            assert torch.equal(a, b) or (torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())), name
    assert served > 300
    # every function and every form that is meant to be served natively was
    for fn in ("unary", "softmax", "rms_norm", "layer_norm", "add_rms_norm", "rope_qk", "mm", "addmm", "sdpa"):
        assert native["fast." + fn], fn
    for form in ("silu", "gelu", "norm of two dims", "rms_norm int", "mm NN", "mm NT", "addmm row", "addmm full",
                 "addmm column", "addmm transposed", "sdpa", "sdpa causal", "sdpa mask bool", "sdpa mask own dtype",
                 "sdpa mask f32", "sdpa cache", "rope interleaved", "rope half"):
        assert native[form], form
    # and the others were left to Python
    for form in ("mm TN", "mm odd k", "sdpa 3-D", "rope f32 tables"):
        assert not native[form], form
    # on another stream the work is ordered on that stream
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        big = torch.randn(4096, 4096, device="cuda")
        y = T.silu(big)
        z = T.silu(y)
    s.synchronize()
    assert torch.equal(z, T.silu(T.silu(big)))


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_native_calls_free_the_interpreter():
    """Each op with the library's entry points replaced by PyGILState_Check,
    which returns 0 (NTOPS_OK, so the op returns its output) where the calling
    thread has let the interpreter go and 1 (so it returns None) where not."""
    lib = _lib.load()
    check = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
    x, w = torch.randn(4, 64, device="cuda"), torch.randn(64, 64, device="cuda")
    q = torch.randn(1, 2, 4, 64, device="cuda")
    f = _lib.fast
    assert f.init(dict.fromkeys(_lib.EXPORTED, check), torch._C._cuda_getDevice, _lib._raw_stream)
    try:
        got = {
            "unary": f.unary(1, x), "softmax": f.softmax(x, -1), "rms_norm": f.rms_norm(x, (64,), None, 1e-6),
            "layer_norm": f.layer_norm(x, (64,), None, None, 1e-5),
            "add_rms_norm": f.add_rms_norm(x, x, (64,), None, 1e-6), "rope_qk": f.rope_qk(q, q, w, w, True),
            "mm": f.mm(x, w), "addmm": f.addmm(x, x, w, 1, 1),
            "sdpa": f.sdpa(q, q, q, None, 0, None, False, None, None, None, None),
            "sdpa slots": f.sdpa(q, q, q, None, 0, None, False, q, q, q, q),
        }
    finally:
        _lib._init_fast(lib)
    assert not [name for name, r in got.items() if r is None]


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_native_calls_from_several_threads():
    """Four threads, each on a stream of its own, through calls that allocate
    outputs and workspaces: every result equals the one computed alone."""
    ins = [(torch.randn(40, 4096, device="cuda").bfloat16(), torch.randn(1024, 4096, device="cuda").bfloat16(),
            torch.randn(1, 8, 1, 64, device="cuda").half(), torch.randn(1, 2, 2048, 64, device="cuda").half())
           for _ in range(4)]

    def step(x, w, q, kv):
        return (T.mm(T.silu(T.rms_norm(x, (4096,))), w.t()),
                T.scaled_dot_product_attention(q, kv, kv, enable_gqa=True))

    alone = [step(*i) for i in ins]
    torch.cuda.synchronize()

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            outs = [step(*ins[i]) for _ in range(50)]
        stream.synchronize()
        return all(torch.equal(a, b) for o in outs for a, b in zip(o, alone[i]))

    with ThreadPoolExecutor(4) as pool:
        assert all(pool.map(work, range(4)))


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_native_calls_under_a_dispatch_mode():
    """A mode written in Python sees the native path's allocations, which are
    made without the interpreter, as it sees the Python path's."""
    seen = []

    class Seeing(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    x, w = torch.randn(4, 4096, device="cuda").bfloat16(), torch.randn(64, 4096, device="cuda").bfloat16()
    q, kv = torch.randn(1, 8, 1, 64, device="cuda").half(), torch.randn(1, 2, 2048, 64, device="cuda").half()
    calls = (lambda: T.silu(x), lambda: T.rms_norm(x, (4096,)), lambda: T.mm(x, w.t()),
             lambda: T.scaled_dot_product_attention(q, kv, kv, enable_gqa=True))
    for call in calls:
        exp = call()
        seen.clear()
        with Seeing():
            got = call()
        assert seen and torch.equal(got, exp)
