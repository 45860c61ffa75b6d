"""ctypes binding of the mskv C ABI (``include/mskv.h``).

The library is ``microserve_amd/libmskv.so``, built in-tree by
``python -m microserve_amd.build``.  There is no fallback: if the library is
missing or cannot be loaded every entry point raises, so a GPU run can never
silently take another path.
"""

from __future__ import annotations

import ctypes
import importlib
import os

import torch  # noqa: F401  (the extension below uses its libraries)


_FAST = "microserve_amd._fast_calls"


class _Missing:
    """Stands in for the native call paths while they cannot be imported (the
    package must import to be built).  Every use looks for them again, since
    they may have been built meanwhile, and raises if they are still not
    there: not built, or built but not loadable, with the cause."""

    def __getattr__(self, name):
        global fast
        found = _import_fast()
        if isinstance(found, _Missing):
            cause = vars(found)["cause"]
            if isinstance(cause, ModuleNotFoundError) and cause.name == _FAST:
                raise RuntimeError(f"{_FAST} is not built: run "
                                   "`python -m microserve_amd.build`") from cause
            raise RuntimeError(f"{_FAST} cannot be loaded ({cause}); if it was built against "
                               "another torch, run `python -m microserve_amd.build`") from cause
        fast = found
        if _lib is not None:
            _bind(_lib)
        return getattr(fast, name)


def _import_fast():
    importlib.invalidate_caches()
    try:
        return importlib.import_module(_FAST)
    except ImportError as e:
        missing = _Missing()
        vars(missing)["cause"] = e
        return missing


fast = _import_fast()

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libmskv.so")

FLOAT16 = 0
BFLOAT16 = 1
FLOAT32 = 2  # key/value rows of the store only
INT32 = 0
INT64 = 1

_c_int, _c_i64, _c_f32, _vp = ctypes.c_int, ctypes.c_int64, ctypes.c_float, ctypes.c_void_p
_c_size = ctypes.c_size_t

# name -> (restype, argtypes); mirrors include/mskv.h
_PROTOS = {
    "mskv_version": (_c_int, []),
    "mskv_status_string": (ctypes.c_char_p, [_c_int]),
    "mskv_store_fp8_kvcache": (_c_int, [
        _vp, _vp, _vp, _vp, _vp, _vp, _vp, _c_int,
        _c_i64, _c_int, _c_int, _c_i64, _c_int, _vp]),
    "mskv_store_fp8_kvcache_strided": (_c_int, [
        _vp, _c_i64, _vp, _c_i64, _vp, _vp, _vp, _vp, _vp, _c_int,
        _c_i64, _c_int, _c_int, _c_i64, _c_int, _vp]),
    "mskv_decode_num_splits": (_c_int, [_c_int, _c_int, _c_int, _c_int, _c_int]),
    "mskv_decode_workspace_bytes": (_c_size, [_c_int, _c_int, _c_int, _c_int, _c_int]),
    "mskv_fp8_decode_attention": (_c_int, [
        _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp,
        _c_int, _c_int, _c_int, _c_int, _c_int, _c_i64, _c_int, _c_f32,
        _c_int, _c_int, _vp, _c_size, _vp]),
    "mskv_fp8_decode_attention_noalloc": (_c_int, [
        _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp,
        _c_int, _c_int, _c_int, _c_int, _c_int, _c_i64, _c_int, _c_f32,
        _c_int, _c_int, _vp]),
    "mskv_fp8_prefill_attention": (_c_int, [
        _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _c_int, _vp,
        _c_int, _c_i64, _c_int, _c_int, _c_int, _c_int, _c_int, _c_i64,
        _c_int, _c_f32, _c_int, _vp]),
    "mskv_fp8_prefill_workspace_bytes": (_c_size, [
        _c_int, _c_i64, _c_int, _c_int, _c_int, _c_int, _c_int, _c_int]),
    "mskv_fp8_prefill_attention_ws": (_c_int, [
        _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _c_int, _vp,
        _c_int, _c_i64, _c_int, _c_int, _c_int, _c_int, _c_int, _c_i64,
        _c_int, _c_f32, _c_int, _vp, _c_size, _vp]),
    "mskv_fp8_prefill_bounded_workspace_bytes": (_c_size, [
        _c_int, _c_i64, _c_int, _c_i64, _c_int, _c_int, _c_int, _c_int, _c_int]),
    "mskv_fp8_prefill_attention_bounded": (_c_int, [
        _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _c_int, _vp,
        _c_int, _c_i64, _c_int, _c_i64, _c_int, _c_int, _c_int, _c_int, _c_i64,
        _c_int, _c_f32, _c_int, _vp, _c_size, _vp]),
    "mskv_prefill_attention": (_c_int, [
        _vp, _vp, _vp, _vp, _vp, _vp, _c_int, _c_i64, _c_i64, _c_int,
        _c_int, _c_int, _c_int, _c_f32, _c_int, _vp]),
    "mskv_prefill_attention_strided": (_c_int, [
        _vp, _vp, _c_i64, _vp, _c_i64, _vp, _vp, _vp, _c_int, _c_i64, _c_i64, _c_int,
        _c_int, _c_int, _c_int, _c_f32, _c_int, _vp]),
    "mskv_build_step_inputs": (_c_int, [
        _vp, _vp, _vp, _vp, _vp, _c_int, _c_int, _c_i64, _c_int, _c_int, _c_i64,
        _vp, _vp, _vp, _vp, _vp, _c_int, _vp]),
    "mskv_qk_norm_rope_store": (_c_int, [
        _vp, _vp, _vp, _c_i64, _c_i64, _c_i64, _vp, _vp, _vp, _c_f32, _vp, _vp, _c_i64,
        _vp, _vp, _vp, _vp, _vp, _vp, _vp, _c_int, _c_i64, _c_int, _c_int, _c_int, _c_i64,
        _c_int, _vp]),
}

EXPORTED = tuple(_PROTOS)

_lib = None


def load() -> ctypes.CDLL:
    """Load libmskv.so once; raise with a build hint if it is absent."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise RuntimeError(
            f"mskv HIP library not found at {LIB_PATH}; build it with "
            "`python -m microserve_amd.build` (hipcc, gfx950)")
    lib = ctypes.CDLL(LIB_PATH)
    for name, (res, args) in _PROTOS.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    if not isinstance(fast, _Missing):  # (the library needs only itself)
        _bind(lib)
    _lib = lib
    return lib


def _bind(lib) -> None:
    fast.bind({name: ctypes.cast(getattr(lib, name), _vp).value for name in _PROTOS})


def check(status: int, what: str) -> None:
    """Raise RuntimeError for a non-zero status, as the reference's launcher would."""
    if status != 0:
        msg = load().mskv_status_string(status).decode()
        raise RuntimeError(f"{what} failed: status {status} ({msg})")


def act_dtype(t) -> int:
    import torch
    if t.dtype == torch.float16:
        return FLOAT16
    if t.dtype == torch.bfloat16:
        return BFLOAT16
    raise AssertionError(f"activation dtype must be float16 or bfloat16, got {t.dtype}")


def store_dtype(t) -> int:
    """Element type of the store's key/value rows: fp16, bf16 or fp32 (the
    reference upcasts any float input to fp32, fp8_kv_cache.py:22-23)."""
    import torch
    if t.dtype == torch.float32:
        return FLOAT32
    if t.dtype in (torch.float16, torch.bfloat16):
        return act_dtype(t)
    raise AssertionError(f"key/value dtype must be float16, bfloat16 or float32, got {t.dtype}")


def aligned(t):
    """``t`` contiguous and on 16 bytes, as the kernels' vector loads and
    direct-to-LDS loads read it: itself if it is, else a copy (a contiguous
    view may start at any element)."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def token_rows(t):
    """A ``[tokens, heads, D]`` tensor and the elements between its tokens,
    for a kernel that reads whole tokens at any stride: a view with each
    token's heads together (the v view of a qkv projection) as it is, if its
    rows start on 16 bytes and the stride fits the kernels' 32-bit tile
    offsets; anything else as a contiguous copy."""
    heads, d = t.shape[1], t.shape[2]
    if not t.is_contiguous():
        s0, s1, s2 = t.stride()
        size = t.element_size()
        if (s2 == 1 and s1 == d and heads * d <= s0 <= 1 << 22 and s0 * size % 16 == 0
                and t.data_ptr() % 16 == 0):
            return t, s0
    return aligned(t), heads * d


def on_device(what: str, ref, *tensors) -> None:
    """Every tensor argument must live on ``ref``'s GPU: a kernel handed a
    host pointer faults instead of raising, so mixed placement is rejected
    here (AssertionError, like the reference's argument checks)."""
    assert ref.is_cuda, f"{what} runs on the GPU"
    for t in tensors:
        if t is not None:
            assert t.device == ref.device, (
                f"{what}: every tensor must be on {ref.device}, got one on {t.device}")


def stream_of(t) -> int:
    import torch
    return torch.cuda.current_stream(t.device).cuda_stream
