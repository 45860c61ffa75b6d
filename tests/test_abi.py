"""CPU checks of the C ABI: the library loads, exports every symbol that
include/mskv.h declares, and rejects bad arguments before touching a GPU."""

import ctypes
import os
import re

import pytest

from microserve_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "mskv.h")


def _declared():
    text = open(HEADER).read()
    return sorted(set(re.findall(r"\b(mskv_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_bound_symbols():
    assert _declared() == sorted(_lib.EXPORTED)


def test_library_exports_every_declared_symbol():
    lib = _lib.load()
    for name in _declared():
        assert getattr(lib, name) is not None
    raw = ctypes.CDLL(_lib.LIB_PATH)
    for name in _declared():
        assert hasattr(raw, name), name


def test_status_strings_and_version():
    lib = _lib.load()
    assert lib.mskv_version() >= 100
    assert lib.mskv_status_string(0) == b"ok"
    for code in (-1, -2, -3, 1):
        assert lib.mskv_status_string(code)


def test_split_policy_depends_on_shapes_only():
    lib = _lib.load()
    # Qwen3-8B decode, batch 64 x 4096 tokens: 16 pages per sequence
    s = lib.mskv_decode_num_splits(64, 32, 8, 16, 256)
    assert 1 < s <= 16
    assert lib.mskv_decode_num_splits(64, 32, 8, 16, 256) == s
    # long single sequence is split across many waves, at most 4 pages each
    s = lib.mskv_decode_num_splits(1, 64, 8, 512, 256)
    assert s >= 128
    # a huge batch needs no split
    assert lib.mskv_decode_num_splits(4096, 32, 8, 4, 256) == 1
    assert lib.mskv_decode_workspace_bytes(64, 32, 8, 128, 1) == 0
    assert lib.mskv_decode_workspace_bytes(64, 32, 8, 128, 8) == 64 * 32 * 8 * 129 * 4
    # 256 x 31 splits runs longest-first work items: the partials (padded to
    # 256 bytes), a 16-byte item count, then 16 bytes per (sequence, split)
    part = (256 * 32 * 31 * 129 * 4 + 255) // 256 * 256
    assert lib.mskv_decode_workspace_bytes(256, 32, 8, 128, 31) == part + 16 + 256 * 31 * 16


def test_every_split_starts_within_an_int_of_tokens():
    """A split's first token is split * (pages per split) * block_size in 32
    bits; pages may hold millions of tokens, and a page's splits finer than
    itself must not multiply past that."""
    lib = _lib.load()
    for batch in (1, 2, 16, 300):
        for hq, hk in ((8, 1), (32, 8), (16, 16)):
            for w in (1, 2, 3, 64, 1000):
                for block in (32, 256, 1 << 12, 1 << 20, 1 << 22, 1 << 23, (1 << 24) - 32):
                    if block * hk * 128 > 0x7FFFFFFF or w * block >= 1 << 30:
                        continue  # rejected by the call itself
                    s = lib.mskv_decode_num_splits(batch, hq, hk, w, block)
                    pages = -(-w // s)
                    assert (s - 1) * pages * block <= 0x7FFFFFFF, (batch, hq, hk, w, block, s)
                    # more splits than pages only where they follow the lengths
                    assert s <= w or w * block <= 1 << 22, (batch, hq, hk, w, block, s)


def test_splits_finer_than_a_page_fit_one_workgroup_per_cu():
    lib = _lib.load()
    finer = 0
    for hq, hk in ((32, 8), (64, 8), (16, 8), (8, 1), (4, 2), (24, 1), (32, 32)):
        units = hk * -(-(hq // hk) // 16)
        for batch in (1, 2, 3, 6, 8, 12, 16, 32, 64, 70, 100, 300):
            for w in (1, 2, 3, 4, 6, 16, 32, 64, 128):
                s = lib.mskv_decode_num_splits(batch, hq, hk, w, 256)
                if s > w:
                    finer += 1
                    assert batch * -(-units // 8) * s <= 256 and 2 * s >= 3 * w
                    assert batch * hq * s * 129 * 4 <= 16 << 20
    assert finer > 50


def test_prefill_workspace_stays_small():
    """The partials have a row per query row: a query tensor with more rows
    than max_seqlen_q lets the grid cover must not ask for gigabytes."""
    lib = _lib.load()
    most = 0
    for seqs in (1, 2, 8, 100):
        for max_q in (1, 40, 512, 4096):
            for total in (1, 40, 512, 4096, 1 << 20):
                for hq, hk in ((32, 8), (64, 8), (40, 8), (24, 1), (8, 8)):
                    for w in (4, 128, 4096):
                        n = lib.mskv_fp8_prefill_workspace_bytes(seqs, total, max_q, hq, hk, 128,
                                                                 256, w)
                        assert n <= 35_000_000, (seqs, max_q, total, hq, hk, w, n)
                        most = max(most, n)
    assert most > 30_000_000


def test_prefill_splits_follow_the_bound_of_the_keys():
    lib = _lib.load()

    def ws(keys, new=40, seqs=1, w=64, heads=(32, 8)):
        return lib.mskv_fp8_prefill_bounded_workspace_bytes(seqs, seqs * new, new, keys, *heads,
                                                            128, 256, w)

    # short contexts are not split, however wide their table
    for w in (2, 64, 128):
        assert ws(340, w=w) == 0 and ws(203, new=74, seqs=4, w=w) == 0
        assert ws(812, new=512, w=max(w, 4)) == 0 and ws(256, new=256, w=w) == 0
    # no bound, or one past the table: the table's width, as the unbounded query
    for keys in (0, -1, 64 * 256, 1 << 40):
        assert ws(keys) == lib.mskv_fp8_prefill_workspace_bytes(1, 40, 40, 32, 8, 128, 256, 64) > 0
    # any bound inside the last page says what the table just wide enough says
    for pages in (3, 5, 8, 31):
        want = ws(0, w=pages)
        assert want > 0
        for keys in (256 * pages, 256 * pages - 1, 256 * pages - 255):
            assert ws(keys) == want


def test_argument_validation_without_launch():
    lib = _lib.load()
    EINVAL, EUNSUP, EWS = -1, -2, -3
    # unsupported head_dim
    assert lib.mskv_store_fp8_kvcache(1, 1, 1, 1, 1, 1, 1, 1, 4, 8, 64, 100, 1, None) == EUNSUP
    # bad dtype codes
    assert lib.mskv_store_fp8_kvcache(1, 1, 1, 1, 1, 1, 1, 7, 4, 8, 128, 100, 1, None) == EINVAL
    assert lib.mskv_store_fp8_kvcache(1, 1, 1, 1, 1, 1, 1, 1, 4, 8, 128, 100, 9, None) == EINVAL
    # zero tokens is a no-op
    assert lib.mskv_store_fp8_kvcache(None, None, None, None, None, None, None, 1, 0, 8, 128, 100, 1, None) == 0
    # null pointer with work to do
    assert lib.mskv_store_fp8_kvcache(None, 1, 1, 1, 1, 1, 1, 1, 4, 8, 128, 100, 1, None) == EINVAL
    # decode: heads not divisible, block size not a multiple of 32
    args = [1] * 8
    assert lib.mskv_fp8_decode_attention(*args, 2, 30, 8, 128, 256, 10, 4, 0.1, 1, 1, None, 0, None) == EINVAL
    assert lib.mskv_fp8_decode_attention(*args, 2, 32, 8, 128, 48, 10, 4, 0.1, 1, 1, None, 0, None) == EUNSUP
    # decode: any GQA divisor is accepted (group 24: the last 16-head unit of
    # each kv head is partly idle); with the right split count the call gets
    # past the shape checks to the workspace check
    s24 = lib.mskv_decode_num_splits(2, 48, 2, 4, 256)
    assert s24 > 1
    assert lib.mskv_fp8_decode_attention(*args, 2, 48, 2, 128, 256, 10, 4, 0.1, 1, s24, None, 0, None) == EWS
    # store: fp32 key/value rows are accepted (zero tokens: a no-op)
    assert lib.mskv_store_fp8_kvcache(None, None, None, None, None, None, None, 1, 0, 8, 128, 100, _lib.FLOAT32, None) == 0
    assert lib.mskv_store_fp8_kvcache(1, 1, 1, 1, 1, 1, 1, 1, 4, 8, 128, 100, 3, None) == EINVAL
    # decode: wrong split count, missing workspace
    s = lib.mskv_decode_num_splits(2, 32, 8, 4, 256)
    assert lib.mskv_fp8_decode_attention(*args, 2, 32, 8, 128, 256, 10, 4, 0.1, 1, s + 1, None, 0, None) == EINVAL
    if s > 1:
        assert lib.mskv_fp8_decode_attention(*args, 2, 32, 8, 128, 256, 10, 4, 0.1, 1, s, None, 0, None) == EWS
    # prefill: only one of the two cu_seqlens pointers
    assert lib.mskv_fp8_prefill_attention(1, 1, 1, 1, 1, 1, 1, None, 0, 1, 2, 10, 5, 32, 8, 128, 256, 10, 4, 0.1, 1, None) == EINVAL
    # prefill: block size not a multiple of 128
    assert lib.mskv_fp8_prefill_attention(1, 1, 1, 1, 1, 1, None, None, 0, 1, 1, 10, 10, 32, 8, 128, 64, 10, 4, 0.1, 1, None) == EUNSUP
    # prefill: more query blocks than a grid dimension holds (GQA 16: 8 tokens per block)
    big_q = 8 * 65535 + 1
    assert lib.mskv_fp8_prefill_attention(1, 1, 1, 1, 1, 1, None, None, 0, 1, 1, big_q, big_q, 128, 8, 128, 256, 10, 4, 0.1, 1, None) == EUNSUP
    assert lib.mskv_prefill_attention(1, 1, 1, 1, 1, 1, 1, big_q, big_q, 4 * 65535 * 48 + 1, 32, 8, 128, 0.1, 1, None) == EUNSUP
    # prefills: the row maxima are taken before a positive, finite softmax scale
    for sc in (0.0, -0.1, float("nan"), float("inf"), 3e38):
        assert lib.mskv_fp8_prefill_attention(1, 1, 1, 1, 1, 1, None, None, 0, 1, 1, 10, 10, 32, 8, 128, 256, 10, 4, sc, 1, None) == EUNSUP
        assert lib.mskv_prefill_attention(1, 1, 1, 1, 1, 1, 1, 10, 10, 10, 32, 8, 128, sc, 1, None) == EUNSUP


def test_prefills_reject_pointers_off_16_bytes():
    lib = _lib.load()
    EINVAL, A = -1, 1 << 20  # a 16-byte aligned stand-in address; nothing is launched

    def paged(**off):
        p = {k: A + off.get(k, 0) for k in ("q", "kc", "vc", "out", "ws")}
        return lib.mskv_fp8_prefill_attention_ws(
            p["q"], p["kc"], p["vc"], A, A, A, None, None, 0, p["out"], 1, 10, 10, 32, 8, 128,
            256, 10, 4, 0.1, 1, p["ws"], 1 << 30, None)

    def fresh(**off):
        p = {k: A + off.get(k, 0) for k in ("q", "k", "v", "out")}
        return lib.mskv_prefill_attention(p["q"], p["k"], p["v"], p["out"], A, A, 1, 10, 10, 10,
                                          32, 8, 128, 0.1, 1, None)

    # (without a GPU an aligned call gets as far as a launch that fails)
    for name in ("q", "kc", "vc", "out", "ws"):
        for by in (2, 4, 8):
            assert paged(**{name: by}) == EINVAL
    for name in ("q", "k", "v", "out"):
        for by in (2, 4, 8):
            assert fresh(**{name: by}) == EINVAL


def test_strided_and_workspace_entries_validate_without_launch():
    lib = _lib.load()
    EINVAL, EUNSUP, EWS, A = -1, -2, -3, 1 << 20
    row = 8 * 128

    def store(ks=row, vs=row, act=1):
        return lib.mskv_store_fp8_kvcache_strided(A, ks, A, vs, A, A, A, A, A, 1, 4, 8, 128, 100,
                                                  act, None)

    def fresh(ks=row, vs=row, num_seqs=1):
        return lib.mskv_prefill_attention_strided(A, A, ks, A, vs, A, A, A, num_seqs, 10, 10, 10,
                                                  32, 8, 128, 0.1, 1, None)

    for call in (store, fresh):
        for bad in (row - 8, 0, -row, row + 4, row + 1):  # below a row, off 16 bytes
            assert call(ks=bad) == EINVAL and call(vs=bad) == EINVAL
    assert store(ks=row + 2, act=_lib.FLOAT32) == EINVAL   # fp32: 16 bytes are 4 elements
    assert store(ks=row - 4, act=_lib.FLOAT32) == EINVAL
    # 64 rows of a tile must stay within 32-bit offsets
    assert fresh(ks=1 << 24) == EUNSUP and fresh(vs=(1 << 24) + 8) == EUNSUP
    assert fresh(num_seqs=0) == 0 and fresh(ks=row + 4, num_seqs=0) == EINVAL

    def paged(ws=A, n=0, keys=0):
        return lib.mskv_fp8_prefill_attention_bounded(
            A, A, A, A, A, A, None, None, 3000, A, 1, 64, 64, keys, 32, 8, 128, 256, 100, 12, 0.1,
            1, ws, n, None)

    need = lib.mskv_fp8_prefill_bounded_workspace_bytes(1, 64, 64, 3064, 32, 8, 128, 256, 12)
    assert need > 0
    for n in (0, 1, need - 1):
        assert paged(n=n) == EWS and paged(n=n, keys=3064) == EWS
    assert lib.mskv_fp8_prefill_attention_ws(
        A, A, A, A, A, A, None, None, 3000, A, 1, 64, 64, 32, 8, 128, 256, 100, 12, 0.1, 1, A,
        need - 1, None) == EWS


def test_wrappers_copy_rows_off_16_bytes():
    import torch
    flat = torch.arange(3 * 4 * 128 + 9).to(torch.bfloat16)
    for at in (0, 1, 2, 4, 8):
        view = flat[at:at + 3 * 4 * 128].view(3, 4, 128)
        assert view.is_contiguous()
        rows, stride = _lib.token_rows(view)
        assert stride == 4 * 128 and rows.data_ptr() % 16 == 0
        assert torch.equal(rows, view) and torch.equal(_lib.aligned(view), view)
        assert _lib.aligned(view).data_ptr() % 16 == 0
        if view.data_ptr() % 16 == 0:
            assert rows is view


def test_new_entry_points_validate_without_launch():
    lib = _lib.load()
    EINVAL, EUNSUP = -1, -2
    A = 1 << 20  # a 16-byte aligned stand-in address; nothing is launched
    # fused prologue: args before (q, k, v, strides, positions, weights, eps, cos, sin, maxpos)
    def nr(head_dim=128, qw=A, kw=A, q=A, qs=48 * 128, n=4, eps=1e-6, slot_dtype=1, act=1):
        return lib.mskv_qk_norm_rope_store(
            q, A, A, qs, 48 * 128, 48 * 128, A, qw, kw, eps, A, A, 4096, A, None, A, A, A, A, A,
            slot_dtype, n, 32, 8, head_dim, 1 << 16, act, None)
    assert nr(head_dim=64) == EUNSUP
    assert nr(kw=None) == EINVAL            # one weight without the other
    assert nr(q=A + 8) == EINVAL            # q not 16-byte aligned
    assert nr(qs=32 * 128 - 8) == EINVAL    # token stride shorter than the q heads
    assert nr(eps=-1.0) == EINVAL
    assert nr(slot_dtype=5) == EINVAL
    assert nr(act=3) == EINVAL
    assert nr(n=0) == 0                     # nothing to do
    # step inputs: (token_ids, starts, cu_q, table_off, tables, num_seqs, pad_seqs, total_q,
    #               block_size, table_width, garbage, ids, pos, slot, lens, tables_out, max_q)
    def si(num_seqs=2, pad=2, total_q=3, bs=256, width=4, ids=A, max_q=2):
        return lib.mskv_build_step_inputs(A, A, A, A, A, num_seqs, pad, total_q, bs, width, 0,
                                          ids, A, A, A, A, max_q, None)
    assert si(pad=1) == EINVAL              # fewer padded rows than sequences
    assert si(bs=0) == EINVAL
    assert si(width=-1) == EINVAL
    assert si(ids=None) == EINVAL           # rows to write but no output
    assert si(num_seqs=70000, pad=70000) == EUNSUP  # grid y limit
    assert si(num_seqs=0, pad=0, total_q=0) == 0


def test_python_wrappers_reject_like_the_reference():
    torch = pytest.importorskip("torch")
    from microserve_amd import fp8_decode_attention, store_fp8_kvcache
    kc = torch.zeros(2, 256, 8, 128, dtype=torch.float8_e4m3fn)
    ks = torch.ones(2, 256, 8)
    k = torch.zeros(3, 8, 128, dtype=torch.bfloat16)
    with pytest.raises(AssertionError):       # wrong scale dtype
        store_fp8_kvcache(k, k, kc, kc, ks.double(), ks.double(), torch.zeros(3, dtype=torch.int64))
    with pytest.raises(AssertionError):       # wrong head_dim layout
        store_fp8_kvcache(k[..., :64], k[..., :64], kc, kc, ks, ks, torch.zeros(3, dtype=torch.int64))
    q = torch.zeros(2, 16, 128, dtype=torch.float32)
    with pytest.raises(AssertionError):       # fp32 query
        fp8_decode_attention(q, kc, kc, ks, ks, torch.ones(2, dtype=torch.int32),
                             torch.zeros(2, 1, dtype=torch.int32), 0.1)
    with pytest.raises(AssertionError):       # int64 lengths
        fp8_decode_attention(q.bfloat16(), kc, kc, ks, ks, torch.ones(2, dtype=torch.int64),
                             torch.zeros(2, 1, dtype=torch.int32), 0.1)


def test_wrappers_reject_tensors_off_the_gpu():
    """A host tensor among GPU arguments is rejected before any launch (a
    kernel given a host pointer would fault).  Checked with CPU tensors only:
    the first check (the reference tensor on the GPU) already fails here."""
    import torch
    from microserve_amd import _lib as L
    with pytest.raises(AssertionError, match="runs on the GPU"):
        L.on_device("x", torch.zeros(1))
