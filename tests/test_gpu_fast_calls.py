"""The native call paths take ordinary calls, give the wrappers' own results
bit for bit, and leave everything else to the wrappers."""

import ctypes

import pytest
import torch

from tests import gpu_helpers as H

pytestmark = pytest.mark.gpu

from microserve_amd import (_lib, fp8_chunk_prefill_attention, fp8_decode_attention,  # noqa: E402
                            fp8_varlen_prefill_attention, qk_norm_rope_store, store_fp8_kvcache,
                            varlen_attention)


class _Off:
    """Native paths that take nothing: the wrappers' own."""

    def __getattr__(self, name):
        return lambda *a: None


class _Counted:
    """The native paths, noting which took a call and which left it."""

    def __init__(self, fast):
        self.fast, self.took, self.left = fast, [], []

    def __getattr__(self, name):
        def call(*a):
            res = getattr(self.fast, name)(*a)
            (self.left if res is None else self.took).append(name)
            return res
        return call


def _both(monkeypatch, entry, call):
    """`call` on the native path, which must take it, and on the wrappers' own:
    the same bytes (each result copied before the next call)."""
    _lib.load()
    with monkeypatch.context() as m:
        counted = _Counted(_lib.fast)
        m.setattr(_lib, "fast", counted)
        fast = call()
        kept = [None if t is None else t.clone() for t in fast]
        assert counted.took == [entry] and not counted.left
        m.setattr(_lib, "fast", _Off())
        slow = call()
    torch.cuda.synchronize()
    for a, b in zip(kept, slow):
        assert (a is None and b is None) or torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    return fast


def _case(dtype, n=5, hq=8, hk=2, blocks=6):
    gen = torch.Generator().manual_seed(811)
    qkv = torch.randn(n, (hq + 2 * hk) * H.D, generator=gen).to(dtype).to(H.DEV)
    q, k, v = (t.view(n, -1, H.D) for t in qkv.split((hq * H.D, hk * H.D, hk * H.D), -1))
    slots = torch.randperm(blocks * H.BLOCK, generator=gen)[:n].to(H.DEV)
    return q, k, v, slots, H.alloc_cache(blocks, H.BLOCK, hk)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_native_paths_give_the_wrappers_results(dtype, monkeypatch):
    q, k, v, slots, caches = _case(dtype)
    n = q.shape[0]

    def store():
        c = H.alloc_cache(6, H.BLOCK, 2)
        store_fp8_kvcache(k.contiguous(), v, *c, slots)
        return c

    caches = _both(monkeypatch, "store", store)
    qc = q.contiguous()
    lens = torch.tensor([300, 1, 0, 256, 40], dtype=torch.int32, device=H.DEV)
    tables = torch.tensor([[0, 1], [2, -1], [-1, -1], [3, -1], [4, 5]], dtype=torch.int32,
                          device=H.DEV)
    out = torch.empty_like(qc)
    _both(monkeypatch, "decode", lambda: [fp8_decode_attention(qc, *caches, lens, tables, 0.1)])

    def into_out():
        out.fill_(7.0)
        return [fp8_decode_attention(qc, *caches, lens, tables, 0.1, out=out)]

    (got,) = _both(monkeypatch, "decode", into_out)
    assert got is out
    _both(monkeypatch, "prefill", lambda: [
        fp8_chunk_prefill_attention(qc, *caches, tables[:1], 200, 0.1)])
    cu = torch.tensor([0, 2, n], dtype=torch.int32, device=H.DEV)
    ck = torch.tensor([0, 300, 500], dtype=torch.int32, device=H.DEV)
    for bound in (None, 300):
        _both(monkeypatch, "prefill", lambda: [fp8_varlen_prefill_attention(
            qc, *caches, tables[:2], cu, ck, 3, 0.1, max_seqlen_k=bound)])
    for kk in (k, k.contiguous()):
        _both(monkeypatch, "fresh", lambda: [varlen_attention(qc, kk, v, cu, cu, 3)])
    cos, sin = (torch.randn(64, 1, H.D, device=H.DEV).to(dtype) for _ in range(2))
    w = torch.randn(H.D, device=H.DEV).to(dtype)
    pos = torch.arange(n, device=H.DEV)
    for weight in (w, None):
        for return_k in (True, False):
            def prologue():
                c = H.alloc_cache(6, H.BLOCK, 2)
                return [*qk_norm_rope_store(pos, q, k, v, weight, weight, 1e-6, cos, sin, *c,
                                            slots, return_k=return_k), *c]
            _both(monkeypatch, "prologue", prologue)


@pytest.mark.parametrize("by", [1, 2])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_contiguous_inputs_off_16_bytes_give_their_copies_results(dtype, by):
    """A contiguous view may start at any element: the kernels' 16-byte loads
    need its copy, on the native path and on the wrappers'."""
    gen = torch.Generator().manual_seed(821)
    n, hq, hk = 9, 8, 2

    def pair(heads):
        flat = torch.randn(n * heads * H.D + 8, generator=gen).to(dtype).to(H.DEV)
        view = flat[by:by + n * heads * H.D].view(n, heads, H.D)
        assert view.is_contiguous() and view.data_ptr() % 16
        return view, view.clone()

    slots = torch.arange(300, 300 + n, device=H.DEV)
    (k, kc), (v, vc), (q, qc) = pair(hk), pair(hk), pair(hq)
    a, b = H.alloc_cache(4, H.BLOCK, hk), H.alloc_cache(4, H.BLOCK, hk)
    store_fp8_kvcache(k, v, *a, slots)
    store_fp8_kvcache(kc, vc, *b, slots)
    for x, y in zip(a, b):
        assert torch.equal(x.view(torch.uint8), y.view(torch.uint8))
    if dtype == torch.float32:
        return
    lens = torch.full((n,), 309, dtype=torch.int32, device=H.DEV)
    tables = torch.tensor([[0, 1]], dtype=torch.int32, device=H.DEV)
    wide = tables.expand(n, 2).contiguous()
    cu = torch.tensor([0, n], dtype=torch.int32, device=H.DEV)
    ck = torch.tensor([0, 309], dtype=torch.int32, device=H.DEV)
    for call in (lambda q, k, v: fp8_decode_attention(q, *a, lens, wide, 0.1),
                 lambda q, k, v: fp8_chunk_prefill_attention(q, *a, tables, 300, 0.1),
                 lambda q, k, v: fp8_varlen_prefill_attention(q, *a, tables, cu, ck, n, 0.1),
                 lambda q, k, v: varlen_attention(q, k, v, cu, cu, n)):
        assert torch.equal(call(q, k, v), call(qc, kc, vc))


def test_native_paths_leave_the_rest_to_the_wrappers():
    q, k, v, slots, caches = _case(torch.float16)
    _lib.load()
    lens = torch.ones(5, dtype=torch.int32, device=H.DEV)
    tables = torch.zeros(5, 1, dtype=torch.int32, device=H.DEV)

    def taken(q=q.contiguous(), caches=caches, lens=lens, tables=tables, scale=0.1, out=None):
        from microserve_amd.fp8_decode_attention import _scratch
        return _lib.fast.decode(q, *caches, lens, tables, scale, out, _scratch) is not None

    class Sub(torch.Tensor):
        pass

    assert taken()
    assert not taken(q=q)                                       # a strided query
    assert not taken(q=q.contiguous().as_subclass(Sub))
    assert not taken(q=q.contiguous().float())
    assert not taken(lens=lens.long()) and not taken(lens=lens[:4]) and not taken(lens=lens.cpu())
    assert not taken(tables=tables.view(-1)) and not taken(tables=tables.expand(5, 2))
    assert not taken(caches=[caches[0].transpose(0, 1), *caches[1:]])
    assert not taken(scale="0.1") and not taken(out=torch.empty_like(q[:4]))
    from torch.overrides import TorchFunctionMode

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert not taken()
    with pytest.raises(AssertionError):
        fp8_decode_attention(q.contiguous().float(), *caches, lens, tables, 0.1)
    with pytest.raises(AssertionError):
        store_fp8_kvcache(k, v[:4], *caches, slots)
    with pytest.raises(RuntimeError, match="status -2"):
        varlen_attention(q.contiguous(), k, v, lens[:2].cumsum(0, dtype=torch.int32) - 1,
                         lens[:2].cumsum(0, dtype=torch.int32) - 1, 1, softmax_scale=-1.0)


def test_a_failed_launch_raises_and_is_not_tried_again():
    """A positive status is a HIP error that the runtime has already
    forgotten: the native path raises it as the wrapper would, and nothing
    calls the entry point a second time.  (The entry points are stood in for
    by a host function; no kernel runs.)"""
    q, k, v, slots, caches = _case(torch.float16)
    lib = _lib.load()
    real = {n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in _lib.EXPORTED}
    calls = []

    @ctypes.CFUNCTYPE(ctypes.c_int)
    def stub():
        calls.append(1)
        return 719

    address = ctypes.cast(stub, ctypes.c_void_p).value
    entries = ("mskv_store_fp8_kvcache_strided", "mskv_fp8_decode_attention",
               "mskv_fp8_prefill_attention_bounded", "mskv_prefill_attention_strided",
               "mskv_qk_norm_rope_store")
    qc = q.contiguous()
    lens = torch.ones(5, dtype=torch.int32, device=H.DEV)
    tables = torch.zeros(5, 1, dtype=torch.int32, device=H.DEV)
    cu = torch.tensor([0, 5], dtype=torch.int32, device=H.DEV)
    cos, sin = (torch.randn(64, H.D, device=H.DEV).half() for _ in range(2))
    pos = torch.arange(5, device=H.DEV)
    _lib.fast.bind({**real, **{n: address for n in entries}})
    try:
        for what, call in (
                ("store_fp8_kvcache", lambda: store_fp8_kvcache(k, v, *caches, slots)),
                ("fp8_decode_attention",
                 lambda: fp8_decode_attention(qc, *caches, lens, tables, 0.1)),
                ("fp8_chunk_prefill_attention",
                 lambda: fp8_chunk_prefill_attention(qc, *caches, tables[:1], 3, 0.1)),
                ("fp8_varlen_prefill_attention",
                 lambda: fp8_varlen_prefill_attention(qc, *caches, tables[:1], cu, cu, 5, 0.1)),
                ("varlen_attention", lambda: varlen_attention(qc, k, v, cu, cu, 5)),
                ("mskv_qk_norm_rope_store",
                 lambda: qk_norm_rope_store(pos, q, k, v, None, None, 1e-6, cos, sin, *caches,
                                            slots))):
            calls.clear()
            with pytest.raises(RuntimeError, match=rf"{what} failed: status 719 \("):
                call()
            assert len(calls) == 1
    finally:
        _lib.fast.bind(real)
    assert torch.isfinite(fp8_decode_attention(qc, *caches, lens, tables, 0.1).float()).all()
