"""The native host path (csrc/host/fa_native.cpp): it takes exactly the calls that the Python
path would run, with the same results, and leaves every other call to it."""
import pytest
import torch

import flag_attn
from flagattention_amd import _lib, gqa, mla


def test_calls_without_gpu_tensors_are_left_to_python():
    """CPU tensors, subclasses, non-tensors and wrong argument counts get None, nothing runs."""
    fast = _lib.native()
    i32 = torch.ones(2, dtype=torch.int32)
    q = torch.zeros((2, 16, 4, 64), dtype=torch.float16)

    class Sub(torch.Tensor):
        pass

    assert fast.mla_metadata(i32, 16, 1, None, None, None) is None
    assert fast.mla_metadata("x", 16, 1, None, None, None) is None
    assert fast.mla_metadata(i32.as_subclass(Sub), 16, 1, None, None, None) is None
    assert fast.contiguous(q, q, q, False, None, False) is None
    assert fast.contiguous(q, q, q, 0, None, False) is None
    assert fast.contiguous(q) is None
    assert fast.paged(q, q, q, i32, i32, 1.0, 1, 0) is None
    assert fast.topk_indices(torch.zeros((1, 1, 4)), i32, 2, False) is None
    assert fast.cache_write(q, q, q, i32, False) is None
    assert fast.mla_decode(*[None] * 11) is None
    assert fast.ABI_VERSION == _lib.ABI_VERSION


@pytest.mark.parametrize("d", gqa.HEAD_DIMS)
def test_split_rule_is_the_python_one(d):
    """Every line of the split rule lies at the same place in both: the extents on each side of
    it (key counts around the split lengths and their limits, row counts around a work-group's,
    pairs up to a full chip)."""
    fast = _lib.native()
    lens = sorted({1, 5000, 8191, 8192, 8193, 70001} |
                  {k * 128 + e for k in range(1, 17) for e in (0, 1)})
    for cus in (64, 256, 304):
        for pairs in (1, 2, 7, 8, 31, 32, 64, 100, 255, 256, 300):
            for rows in (1, 8, 15, 16, 17, 40, 127, 128, 129, 400, 1500, 4096):
                for n in lens:
                    assert fast.split_counts(pairs, rows, d, n, cus) == (
                        gqa.choose_splits(pairs, 1, rows, n, cus, head_dim=d),
                        gqa.contiguous_splits(1, pairs, rows, n, cus, d)), (pairs, rows, n, cus)


def test_short_splits_fit_the_chip_at_once():
    """At head dims 256 and 512 a CU holds one work-group of the 16-row kernel: splits of under
    256 keys must not leave some of them for a second turn."""
    for d in (256, 512):
        for pairs in range(1, 256):
            for n in (257, 300, 520, 800, 1200, 3000):
                s = gqa.choose_splits(1, pairs, 16, n, 256, head_dim=d)
                assert s <= -(-n // gqa.MIN_SPLIT_TOKENS) or s * pairs <= 256, (d, pairs, n, s)


def _both(monkeypatch, call):
    """The call's results with and without the native path."""
    a = call()
    with monkeypatch.context() as m:
        m.setattr(_lib, "native", lambda: None)
        b = call()
    torch.cuda.synchronize()
    return a, b


def _same(a, b):
    a, b = (x if isinstance(x, tuple) else (x,) for x in (a, b))
    assert len(a) == len(b)
    for x, y in zip(a, b):
        if x is None:
            assert y is None
            continue
        assert x.dtype == y.dtype and x.shape == y.shape and x.stride() == y.stride()
        assert x.requires_grad == y.requires_grad and torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hk,M,N,D,causal,scale,layout", [
    (1, 4, 2, 1, 700, 64, False, None, "bhtd"),    # split, 16-row kernel
    (2, 8, 1, 3, 300, 128, True, 0.2, "bthd"),     # 24 rows, unsplit
    (2, 8, 1, 3, 3000, 128, True, -1, "bthd"),     # 24 rows, split
    (4, 8, 8, 128, 900, 128, True, None, "bthd"),  # too many partial values for short splits
    (1, 8, 2, 5, 385, 128, True, None, "bhtd"),    # few keys, short splits
    (1, 8, 2, 5, 384, 128, True, None, "bhtd"),    # one key fewer: unsplit
    (2, 4, 1, 9, 257, 256, False, None, "bthd"),   # head dim 256 from 257
    (1, 8, 8, 400, 512, 128, True, None, "bthd"),  # too many partial values: unsplit
    (1, 4, 1, 1, 4000, 64, False, None, "bhtd"),   # too many short splits at head dim 64
    (1, 4, 1, 1, 8193, 128, False, None, "bhtd"),  # and at 128
    (1, 2, 2, 200, 2000, 256, True, None, "bhtd"),
    (1, 2, 2, 5, 40, 32, False, None, "bthd"),
    (1, 1, 1, 2, 900, 512, True, None, "bhtd"),
    (1, 2, 1, 4, 64, 64, True, None, "odd"),       # rows not 16-byte aligned: left to Python
])
def test_contiguous_matches_python_path(monkeypatch, B, Hq, Hk, M, N, D, causal, scale, layout):
    def mk(h, t):
        if layout == "odd":
            return torch.randn((B, h, t, D + 1), device="cuda").half()[..., 1:]
        x = torch.randn((B, t, h, D) if layout == "bthd" else (B, h, t, D), device="cuda").half()
        return x.transpose(1, 2) if layout == "bthd" else x

    q, k, v = mk(Hq, M).requires_grad_(), mk(Hk, N), mk(Hk, N)
    assert (_lib.native().contiguous(q, k, v, causal, scale, True) is None) == (layout == "odd")
    _same(*_both(monkeypatch, lambda: flag_attn.flash_attention(
        q, k, v, causal, scale, return_log_normalizer=True)[:2]))
    _same(*_both(monkeypatch, lambda: flag_attn.flash_attention_split_kv(q, k, v, causal, scale)))


@pytest.mark.gpu
@pytest.mark.parametrize("num_splits", [0, 1, 3, 40])
@pytest.mark.parametrize("seqs,Hq,Hk,D,block,max_len", [
    (3, 8, 2, 64, 16, 1000), (70, 16, 4, 128, 32, 300), (1, 2, 2, 512, 24, 5000)])
def test_paged_matches_python_path(monkeypatch, num_splits, seqs, Hq, Hk, D, block, max_len):
    cache = torch.randn((64, Hk, block, D), device="cuda").bfloat16()
    q = torch.randn((Hq, seqs, D), device="cuda").bfloat16().transpose(0, 1)
    lens = torch.randint(1, max_len + 1, (seqs,), dtype=torch.int32, device="cuda")
    bt = torch.randint(0, 64, (seqs, -(-max_len // block)), dtype=torch.int32, device="cuda")
    args = (q, cache, cache.flip(0), lens, bt, D ** -0.5, max_len, num_splits)
    assert _lib.native().paged(*args) is not None
    _same(*_both(monkeypatch, lambda: flag_attn.paged_attention(*args)))


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["dense", "sparse", "fp8"])
@pytest.mark.parametrize("B,h,s_q,parts", [(1, 16, 1, None), (5, 128, 2, None), (3, 40, 3, 7)])
def test_mla_matches_python_path(monkeypatch, mode, B, h, s_q, parts):
    lens = torch.randint(1, 900, (B,), dtype=torch.int32, device="cuda")
    bt = torch.randperm(B * 16, device="cuda").to(torch.int32).view(B, 16)
    q = torch.randn((B, s_q, h, 576), device="cuda").bfloat16()
    topk = None if mode == "dense" else 200
    idx = (None if topk is None else
           torch.randint(-1, 900, (B, s_q, topk), dtype=torch.int32, device="cuda"))
    if mode == "fp8":
        kc = torch.zeros((B * 16, 64, 1, 656), dtype=torch.uint8, device="cuda")
        flag_attn.concat_and_cache_mla(
            torch.randn((B * 1024, 512), device="cuda").bfloat16(),
            torch.randn((B * 1024, 64), device="cuda").bfloat16(), kc,
            torch.arange(B * 1024, device="cuda"), True)
    else:
        kc = torch.randn((B * 16, 64, 1, 576), device="cuda").bfloat16()
    meta = lambda: flag_attn.get_mla_metadata(  # noqa: E731
        lens, s_q * h, 1, num_heads_q=h, topk=topk, num_sm_parts=parts)
    assert _lib.native().mla_metadata(lens, s_q * h, 1, h, topk, parts) is not None
    assert _lib.native().mla_metadata(lens.long(), s_q * h, 1, h, topk, parts) is None
    (md, ns), python = _both(monkeypatch, meta)
    _same((md, ns), python)
    assert md._fa_mla_sig == python[0]._fa_mla_sig and ns._fa_mla_sig == python[1]._fa_mla_sig
    args = (q, kc, bt, lens, 512, md, ns, None, mode == "dense", mode == "fp8", idx)
    assert _lib.native().mla_decode(*args) is not None
    assert _lib.native().mla_decode(q.float(), *args[1:]) is None
    _same(*_both(monkeypatch, lambda: flag_attn.flash_mla_with_kvcache(*args)))
    with pytest.raises(mla.MLAArgumentError):  # metadata of another batch
        other, other_ns = flag_attn.get_mla_metadata(lens.repeat(2), s_q * h, 1, num_heads_q=h,
                                                     topk=topk)
        assert _lib.native().mla_decode(*args[:5], other, *args[6:]) is None
        flag_attn.flash_mla_with_kvcache(q, kc, bt, lens, 512, other, ns, None, False,
                                         mode == "fp8", idx)


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("slots", [torch.int32, torch.int64])
def test_write_and_topk_match_python_path(monkeypatch, fp8, slots):
    kv = torch.randn((77, 512), device="cuda").bfloat16()
    pe = torch.randn((77, 64), device="cuda").bfloat16()
    at = torch.randperm(128, device="cuda")[:154][::2][:64].to(slots)
    kv, pe = kv[: at.numel()], pe[: at.numel()]
    row, dt = (656, torch.uint8) if fp8 else (576, torch.bfloat16)

    def write():
        cache = torch.zeros((2, 64, 1, row), dtype=dt, device="cuda")
        flag_attn.concat_and_cache_mla(kv, pe, cache, at, fp8)
        return cache

    fresh = torch.zeros((2, 64, 1, row), dtype=dt, device="cuda")
    assert _lib.native().cache_write(kv, pe, fresh, at, fp8) is True
    assert _lib.native().cache_write(kv, pe, fresh, at.float(), fp8) is None
    _same(*_both(monkeypatch, write))
    for n, k in ((700, 64), (40000, 2048)):
        scores = torch.randn((2, 2, n), device="cuda")
        lens = torch.tensor([n, n // 2], dtype=torch.int32, device="cuda")
        assert _lib.native().topk_indices(scores, lens, k, True) is not None
        assert _lib.native().topk_indices(scores.half(), lens, k, True) is None
        _same(*_both(monkeypatch, lambda: flag_attn.topk_indices(scores, lens, k, True)))


@pytest.mark.gpu
def test_timing_hook_still_fires():
    """The benchmark hook's events bracket the next decode launch (the Python path)."""
    q = torch.randn((1, 2, 1, 64), device="cuda").half()
    ev = (torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
    gqa.timing_events = ev
    flag_attn.flash_attention(q, q, q)
    torch.cuda.synchronize()
    assert gqa.timing_events is None and ev[0].elapsed_time(ev[1]) > 0
