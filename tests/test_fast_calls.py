"""The native call paths leave every call they cannot take as it stands to
the wrappers: on the CPU, tensors that are not on a GPU."""

import torch

from microserve_amd import _lib


def _args(n=2, hq=4, hk=2):
    kc = torch.zeros(3, 128, hk, 128).to(torch.float8_e4m3fn)
    ks = torch.ones(3, 128, hk)
    q = torch.zeros(n, hq, 128, dtype=torch.float16)
    k = torch.zeros(n, hk, 128, dtype=torch.float16)
    i32 = torch.zeros(n, dtype=torch.int32)
    return q, k, kc, ks, i32


def test_tensors_off_the_gpu_are_left_to_the_wrappers():
    _lib.load()
    q, k, kc, ks, i32 = _args()
    f = _lib.fast
    assert f.store(k, k, kc, kc, ks, ks, i32) is None
    assert f.decode(q, kc, kc, ks, ks, i32, i32.view(-1, 1), 0.1, None, None) is None
    assert f.prefill(q, kc, kc, ks, ks, i32, None, None, 0, 2, 0.1) is None
    assert f.fresh(q, k, k, i32, i32, 2, 0.1) is None
    cos = torch.ones(4, 128, dtype=torch.float16)
    assert f.prologue(i32.long(), q, k, k, None, None, 1e-6, cos, cos, kc, kc, ks, ks, i32,
                      True) is None


def test_wrong_argument_counts_and_types_are_left_to_the_wrappers():
    f = _lib.fast
    for fn in (f.store, f.decode, f.prefill, f.fresh, f.prologue):
        assert fn() is None
        assert fn(*[None] * 7) is None and fn(*["x"] * 15) is None and fn(*[3] * 10) is None
