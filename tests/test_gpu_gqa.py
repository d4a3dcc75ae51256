"""GPU parity of the grouped-query decode path (flag_attn.paged_attention,
flag_attn.flash_attention_split_kv, flag_attn.flash_attention) against the CPU oracle.

The sweeps are the reference's own: ``tests/flag_attn/test_paged_attention.py:79-157``
(fp16, uniform(+-D^-0.5) inputs, block tables drawn with replacement, ``allclose(atol=2e-3,
rtol=1e-5)`` against ``testing.paged_attention``) and
``tests/flag_attn/test_flash_attention.py:82-127`` (``test_attention_splitkv``: scale 10,
BHTD / BTHD strides, fp16 / bf16, causal or not, the rule
``max|hyp - ref| <= 2 max|torch_lowp - ref| + 1e-5``).  The paged sweeps apply that rule
too (against ``gqa_oracle.paged_attention_lowp``) beside the reference's ``allclose``.  Inputs are seeded here (the
reference's paged tests are not).  Caches are generated on the GPU; the oracle gets CPU
copies of the pages the block tables name.
"""
import pytest
import torch

import flag_attn
from oracle import gqa_oracle as go
from tests._helpers import DEV, assert_lowp_rule, need_gpu, say

pytestmark = pytest.mark.gpu
NUM_BLOCKS = 1000
CACHE_BYTES = 256 << 20  # per cache; fewer pages than NUM_BLOCKS when they are large


def base_paged_attention(num_seqs, num_query_heads, query_group_size, head_size, block_size,
                         max_seq_len, num_splits=0, dtype=torch.float16, seed=0):
    need_gpu()
    say(f"paged seqs={num_seqs} H={num_query_heads} g={query_group_size} D={head_size} "
        f"bs={block_size} len={max_seq_len} splits={num_splits} {dtype}")
    gen = torch.Generator().manual_seed(seed)
    dgen = torch.Generator(device=DEV).manual_seed(seed)
    num_kv_heads = num_query_heads // query_group_size
    context_lens = torch.randint(1, max_seq_len, (num_seqs,), generator=gen, dtype=torch.int32)
    context_lens[0] = max_seq_len
    max_context_len = int(context_lens.max())
    max_blocks = (max_context_len + block_size - 1) // block_size
    page_bytes = num_kv_heads * block_size * head_size * 2
    nblocks = max(64, min(NUM_BLOCKS, CACHE_BYTES // page_bytes))
    scale = head_size ** -0.5
    q = torch.empty((num_seqs, num_query_heads, head_size), device=DEV, dtype=dtype)
    q.uniform_(-scale, scale, generator=dgen)
    k_cache = torch.empty((nblocks, num_kv_heads, block_size, head_size), device=DEV, dtype=dtype)
    k_cache.uniform_(-scale, scale, generator=dgen)
    v_cache = torch.empty_like(k_cache).uniform_(-scale, scale, generator=dgen)
    block_tables = torch.randint(0, nblocks, (num_seqs, max_blocks), generator=gen,
                                 dtype=torch.int32)
    out = flag_attn.paged_attention(q, k_cache, v_cache, context_lens.to(DEV),
                                    block_tables.to(DEV), scale, max_context_len, num_splits)
    torch.cuda.synchronize()
    # oracle on the pages the tables name (remapped onto a compact pool)
    need = torch.unique(block_tables.flatten()).long()
    remap = torch.full((nblocks,), -1, dtype=torch.long)
    remap[need] = torch.arange(need.numel())
    kc = k_cache[need.to(DEV)].cpu()
    vc = v_cache[need.to(DEV)].cpu()
    bt = remap[block_tables.long()].to(torch.int32)
    ref = go.paged_attention_ref(q.cpu(), kc, vc, bt, context_lens, scale)
    err = float((out.cpu().float() - ref.float()).abs().max())
    say(f"  max |out - ref| = {err:.3e}")
    assert torch.allclose(out.cpu(), ref, atol=2e-3, rtol=1e-5)
    # the reference's allclose alone passes a kernel that drops a page at these output
    # sizes; the three-way rule against the fp32 result and the low-precision leg does not
    ref32 = go.paged_attention_ref(q.cpu(), kc, vc, bt, context_lens, scale, out_fp32=True)
    low = go.paged_attention_lowp(q.cpu(), kc, vc, bt, context_lens, scale)
    assert_lowp_rule(out.cpu(), ref32, low)


@pytest.mark.parametrize("num_seqs", [1, 32])
@pytest.mark.parametrize("num_query_heads", [64])
@pytest.mark.parametrize("query_group_size", [1, 8])
@pytest.mark.parametrize("head_size", [64, 128])
@pytest.mark.parametrize("block_size", [16, 128, 256])
@pytest.mark.parametrize("max_seq_len", [512, 4096])
def test_paged_attention_default(num_seqs, num_query_heads, query_group_size, head_size,
                                 block_size, max_seq_len):
    base_paged_attention(num_seqs, num_query_heads, query_group_size, head_size, block_size,
                         max_seq_len, seed=num_seqs * 7 + head_size + block_size + max_seq_len)


@pytest.mark.parametrize("num_seqs", [1, 16])
@pytest.mark.parametrize("num_query_heads", [64])
@pytest.mark.parametrize("query_group_size", [1, 8])
@pytest.mark.parametrize("head_size", [32, 64])
@pytest.mark.parametrize("block_size", [16])
@pytest.mark.parametrize("max_seq_len", [2048])
@pytest.mark.parametrize("num_splits", [1, 2, 3, 4, 5, 6, 7, 8])
def test_paged_attention_by_num_splits(num_seqs, num_query_heads, query_group_size, head_size,
                                       block_size, max_seq_len, num_splits):
    base_paged_attention(num_seqs, num_query_heads, query_group_size, head_size, block_size,
                         max_seq_len, num_splits, seed=num_splits * 13 + num_seqs + head_size)


@pytest.mark.parametrize("num_seqs, num_query_heads, query_group_size, head_size, block_size, "
                         "max_seq_len, num_splits", [
                             (1, 12, 1, 64, 16, 2, 0),
                             (16, 64, 8, 32, 16, 2048, 2),
                             (16, 64, 1, 64, 16, 2048, 6),
                         ])
def test_paged_attention_by_case(num_seqs, num_query_heads, query_group_size, head_size,
                                 block_size, max_seq_len, num_splits):
    base_paged_attention(num_seqs, num_query_heads, query_group_size, head_size, block_size,
                         max_seq_len, num_splits, seed=5)


@pytest.mark.parametrize("head_size,group,dtype", [
    (16, 4, torch.float16), (256, 2, torch.float16), (128, 8, torch.bfloat16),
    (256, 1, torch.bfloat16), (32, 16, torch.bfloat16),
])
@pytest.mark.parametrize("num_splits", [0, 3])
def test_paged_attention_more_shapes(head_size, group, dtype, num_splits):
    """Head dims 16 and 256, bf16, and query groups beyond the reference's sweep (16 rows
    per work-group at group 16)."""
    base_paged_attention(8, 32, group, head_size, 16, 1500, num_splits, dtype=dtype,
                         seed=head_size + group)


@pytest.mark.parametrize("d", [64, 512])
def test_paged_attention_bad_page_is_masked(d):
    """A block-table entry outside the cache reads as a masked key instead of faulting."""
    need_gpu()
    gen = torch.Generator().manual_seed(3)
    h, bs = 8, 16
    kc = torch.randn((10, h, bs, d), generator=gen).half()
    vc = torch.randn((10, h, bs, d), generator=gen).half()
    q = torch.randn((1, h, d), generator=gen).half()
    bt = torch.tensor([[0, 1000, 2]], dtype=torch.int32)
    lens = torch.tensor([48], dtype=torch.int32)
    out = flag_attn.paged_attention(q.to(DEV), kc.to(DEV), vc.to(DEV), lens.to(DEV), bt.to(DEV),
                                    d ** -0.5, 48, 1)
    keep = torch.tensor([[0, 2]], dtype=torch.int32)  # the same keys without the bad page
    ref_lens = torch.tensor([32], dtype=torch.int32)
    ref = go.paged_attention_ref(q, kc, vc, keep, ref_lens, d ** -0.5)
    assert torch.allclose(out.cpu(), ref, atol=2e-3, rtol=1e-5)


SPLITKV_SHAPES = [
    (2, 4, 4, 1, 612, 128), (2, 4, 4, 1, 1034, 64), (2, 4, 4, 1, 2048, 32),
    (2, 4, 4, 1, 4096, 16), (2, 4, 4, 1, 4001, 32), (2, 4, 4, 1, 4096, 64),
    (2, 4, 4, 2, 4000, 128), (1, 2, 2, 4, 8202, 16), (1, 2, 2, 1, 8192, 32),
    (2, 4, 2, 1, 612, 128), (2, 4, 1, 1, 1034, 64), (2, 4, 2, 1, 2048, 32),
    (2, 4, 1, 1, 4096, 16), (2, 4, 2, 1, 4001, 32), (2, 4, 1, 1, 4096, 64),
    (2, 4, 2, 2, 4000, 128), (1, 2, 1, 4, 8202, 16), (1, 2, 1, 1, 8192, 32),
]


def _splitkv_inputs(B, Hq, Hk, M, N, D, dtype, stride_order, scale, seed):
    gen = torch.Generator().manual_seed(seed)
    if stride_order == "BHTD":
        q = torch.empty((B, Hq, M, D)).normal_(0.0, scale, generator=gen)
        k = torch.empty((B, Hk, N, D)).normal_(0.0, scale, generator=gen)
        v = torch.empty((B, Hk, N, D)).normal_(0.0, scale, generator=gen)
        return q.to(dtype), k.to(dtype), v.to(dtype)
    q = torch.empty((B, M, Hq, D)).normal_(0.0, scale, generator=gen).transpose(1, 2)
    k = torch.empty((B, N, Hk, D)).normal_(0.0, scale, generator=gen).transpose(1, 2)
    v = torch.empty((B, N, Hk, D)).normal_(0.0, scale, generator=gen).transpose(1, 2)
    return q.to(dtype), k.to(dtype), v.to(dtype)


def _max_diff(a, b):
    return float((a.float() - b.float()).abs().max())


@pytest.mark.parametrize("scale", [10.0])
@pytest.mark.parametrize("B, Hq, Hk, M, N, D", SPLITKV_SHAPES)
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("stride_order", ["BHTD", "BTHD"])
def test_attention_splitkv(B, Hq, Hk, M, N, D, causal, stride_order, dtype, scale):
    need_gpu()
    q, k, v = _splitkv_inputs(B, Hq, Hk, M, N, D, dtype, stride_order, scale, 10086 + N + M)
    o_ref, _ = go.flash_attention_ref(q, k, v, causal, upcast=True)
    o_torch, _ = go.flash_attention_ref(q, k, v, causal, upcast=False)
    # the reference test calls flash_attention, which takes its split-KV path at these shapes
    o_hyp = flag_attn.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), causal).cpu()
    torch_max_diff = _max_diff(o_torch, o_ref)
    hyp_max_diff = _max_diff(o_hyp, o_ref)
    assert o_hyp.dtype == dtype and o_hyp.shape == q.shape
    assert hyp_max_diff <= 2 * torch_max_diff + 1e-5, (hyp_max_diff, torch_max_diff)


@pytest.mark.parametrize("B, Hq, Hk, M, N, D", SPLITKV_SHAPES[::3])
@pytest.mark.parametrize("causal", [True, False])
def test_flash_attention_split_kv_and_lse(B, Hq, Hk, M, N, D, causal):
    """flash_attention_split_kv gives the same o; flash_attention's log normaliser matches
    the oracle's logsumexp."""
    need_gpu()
    q, k, v = _splitkv_inputs(B, Hq, Hk, M, N, D, torch.bfloat16, "BHTD", 1.0, N)
    o_ref, lse_ref = go.flash_attention_ref(q, k, v, causal, upcast=True)
    o_torch, _ = go.flash_attention_ref(q, k, v, causal, upcast=False)
    o1 = flag_attn.flash_attention_split_kv(q.to(DEV), k.to(DEV), v.to(DEV), causal).cpu()
    o2, lse, tot, seed, off = flag_attn.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), causal,
                                                        return_log_normalizer=True)
    assert tot is None and seed is None and off is None
    assert torch.equal(o1, o2.cpu())
    assert _max_diff(o1, o_ref) <= 2 * _max_diff(o_torch, o_ref) + 1e-5
    assert lse.shape == (B, Hq, M) and lse.dtype == torch.float32
    assert torch.allclose(lse.cpu(), lse_ref, atol=1e-3, rtol=1e-4)


@pytest.mark.parametrize("block_size,group,num_splits", [
    (8, 1, 0), (8, 1, 3), (24, 1, 3), (24, 4, 0), (48, 8, 5), (48, 2, 1),
])
def test_paged_attention_odd_block_sizes(block_size, group, num_splits):
    """Pages below 16 tokens (the reference allows them at query group 1, paged.py:46) and
    page sizes that are not powers of two (the kernel divides instead of shifting, and looks
    pages up per lane), with split starts (next_pow2 partitions) that do not fall on page
    boundaries."""
    base_paged_attention(8, 16, group, 64, block_size, 1500, num_splits,
                         seed=block_size * 10 + group + num_splits)


@pytest.mark.parametrize("seqs,h_kv,group,D,block_size,max_len", [
    (1, 1, 8, 128, 16, 257),    # 3 splits of 96, the last of 65 keys
    (3, 2, 4, 64, 16, 385),
    (1, 4, 4, 512, 16, 1000),
    (2, 2, 1, 256, 32, 1025),
    (1, 1, 4, 128, 16, 8192),   # 64 splits, the most
])
def test_paged_attention_short_splits(seqs, h_kv, group, D, block_size, max_len):
    """Splits of 128 keys (one tile per wave), which few work-groups take on their own."""
    from flagattention_amd import gqa
    need_gpu()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert gqa.choose_splits(seqs, h_kv, group, max_len, cus, head_dim=D) == -(-max_len // 128)
    base_paged_attention(seqs, h_kv * group, group, D, block_size, max_len, 0, seed=max_len)


def _oracle_chunked(q, k, v, causal, upcast, chunk=4):
    """flash_attention_ref over batch slices (the GQA repeat of a whole batch would not fit
    in host memory at these shapes)."""
    outs, lses = [], []
    for b0 in range(0, q.shape[0], chunk):
        o, lse = go.flash_attention_ref(q[b0:b0 + chunk], k[b0:b0 + chunk], v[b0:b0 + chunk],
                                        causal, upcast=upcast)
        outs.append(o)
        lses.append(lse)
    return torch.cat(outs), torch.cat(lses)


@pytest.mark.parametrize("B, Hq, Hk, M, N, D, causal", [
    (64, 32, 8, 1, 2048, 128, False),
    (32, 64, 64, 2, 1500, 64, True),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("stride_order", ["BHTD", "BTHD"])
def test_unsplit_contiguous_decode(B, Hq, Hk, M, N, D, causal, dtype, stride_order):
    """Shapes with enough (sequence, KV head, row block) work-groups to fill the GPU take no
    split: the decode kernel writes out and lse itself (no combine).  These are the shapes
    for which the reference's flash_attention takes its _fwd_kernel branch and returns L
    (flash.py:78-101, split_kv.py:249-251)."""
    from flagattention_amd import gqa
    need_gpu()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert gqa.choose_splits(B, Hk, (Hq // Hk) * M, N, cus) == 1
    q, k, v = _splitkv_inputs(B, Hq, Hk, M, N, D, dtype, stride_order, 1.0, N + M)
    o_ref, lse_ref = _oracle_chunked(q, k, v, causal, True)
    o_low, _ = _oracle_chunked(q, k, v, causal, False)
    o1, lse, _, _, _ = flag_attn.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), causal,
                                                 return_log_normalizer=True)
    o2 = flag_attn.flash_attention_split_kv(q.to(DEV), k.to(DEV), v.to(DEV), causal)
    torch.cuda.synchronize()
    assert o1.dtype == dtype and o1.shape == q.shape
    assert torch.equal(o1.cpu(), o2.cpu())
    assert_lowp_rule(o1.cpu(), o_ref, o_low)
    assert lse.shape == (B, Hq, M) and lse.dtype == torch.float32
    assert float((lse.cpu() - lse_ref).abs().max()) <= 1e-3


@pytest.mark.parametrize("M, N, causal", [
    (16, 300, False), (64, 700, True), (200, 1000, True), (40, 24, True), (33, 33, True),
    (17, 5, False),
])
def test_flash_attention_many_queries(M, N, causal):
    """flash_attention with more query positions than a decode step (the reference's
    forward takes any M, flash.py:269-300): rows of 16 (head, position) pairs per
    work-group.  Causal with M > N leaves the first M - N positions no key: out 0,
    lse -inf (the LARGER_M convention of split_kv.py:161-164, flash.py's _fwd_kernel)."""
    need_gpu()
    q, k, v = _splitkv_inputs(2, 4, 2, M, N, 64, torch.float16, "BHTD", 1.0, M * 1000 + N)
    o_ref, lse_ref = go.flash_attention_ref(q, k, v, causal, upcast=True)
    o_low, _ = go.flash_attention_ref(q, k, v, causal, upcast=False)
    o, lse, _, _, _ = flag_attn.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), causal,
                                                return_log_normalizer=True)
    torch.cuda.synchronize()
    o, lse = o.cpu(), lse.cpu()
    assert bool(torch.isfinite(o).all())
    assert_lowp_rule(o, o_ref, o_low)
    assert torch.equal(torch.isneginf(lse), torch.isneginf(lse_ref))
    fin = ~torch.isneginf(lse_ref)
    assert float((lse[fin] - lse_ref[fin]).abs().max()) <= 1e-3
    if causal and M > N:
        assert float(o[:, :, : M - N].abs().max()) == 0.0


@pytest.mark.parametrize("num_seqs", [1, 8])
@pytest.mark.parametrize("query_group_size", [1, 8])
@pytest.mark.parametrize("block_size", [16, 128])
@pytest.mark.parametrize("max_seq_len", [512, 2048])
def test_paged_attention_head_size_512(num_seqs, query_group_size, block_size, max_seq_len):
    """head_size 512, which the reference's paged_attention accepts (paged.py:45): the
    reference sweep's inputs at that head size (the dims-split kernel)."""
    base_paged_attention(num_seqs, 64, query_group_size, 512, block_size, max_seq_len,
                         seed=num_seqs + query_group_size + block_size + max_seq_len)


@pytest.mark.parametrize("num_splits,dtype,block_size", [
    (1, torch.float16, 16), (3, torch.float16, 16), (8, torch.bfloat16, 16),
    (0, torch.bfloat16, 24), (5, torch.float16, 8),
])
def test_paged_attention_head_size_512_splits(num_splits, dtype, block_size):
    base_paged_attention(4, 16, 1 if block_size < 16 else 4, 512, block_size, 1500, num_splits,
                         dtype=dtype, seed=num_splits + block_size)


@pytest.mark.parametrize("M, N, causal", [(1, 3000, False), (3, 700, True)])
def test_flash_attention_head_size_512(M, N, causal):
    """The contiguous decode at head dim 512 (beyond the reference's flash_attention, which
    stops at 128): split and unsplit shapes through the dims-split kernel."""
    need_gpu()
    for B, Hq, Hk in ((2, 4, 2), (64, 16, 4)):
        q, k, v = _splitkv_inputs(B, Hq, Hk, M, N, 512, torch.bfloat16, "BTHD", 1.0, N + B)
        o_ref, lse_ref = _oracle_chunked(q, k, v, causal, True)
        o_low, _ = _oracle_chunked(q, k, v, causal, False)
        o, lse, _, _, _ = flag_attn.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), causal,
                                                    return_log_normalizer=True)
        torch.cuda.synchronize()
        assert_lowp_rule(o.cpu(), o_ref, o_low)
        assert float((lse.cpu() - lse_ref).abs().max()) <= 1e-3


@pytest.mark.parametrize("N", [1, 31, 32, 33, 64, 65, 96, 97, 128])
def test_flash_attention_head_size_512_few_tiles(N):
    """One to four 32-token tiles per work-group at head dim 512: the dims-split loop
    requests K two tiles ahead and V one, so these are its pipeline's start and end cases
    (no next tile, a next tile without the one after it)."""
    need_gpu()
    q, k, v = _splitkv_inputs(3, 8, 2, 1, N, 512, torch.float16, "BHTD", 1.0, 700 + N)
    o_ref, lse_ref = _oracle_chunked(q, k, v, False, True)
    o_low, _ = _oracle_chunked(q, k, v, False, False)
    o, lse, _, _, _ = flag_attn.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), False,
                                                return_log_normalizer=True)
    torch.cuda.synchronize()
    assert_lowp_rule(o.cpu(), o_ref, o_low)
    assert float((lse.cpu() - lse_ref).abs().max()) <= 1e-3


@pytest.mark.parametrize("head_size", [64, 512])
def test_paged_attention_split_longer_than_lds_table(head_size):
    """A split of more than 2,048 pages (8-token pages, one split over 20,000 tokens): the
    split's block-table slice does not fit in LDS and the pages are looked up in global
    memory (the other loop of both kernels)."""
    base_paged_attention(2, 4, 1, head_size, 8, 20000, 1, seed=head_size)


@pytest.mark.parametrize("head_size", [16, 64, 128, 256, 512])
@pytest.mark.parametrize("num_splits", [16, 32, 128])
def test_paged_attention_many_splits(head_size, num_splits):
    """The combine on both sides of its team size (one wave per row up to 16 splits, four
    above) with splits past the end of the short sequences (empty partials)."""
    base_paged_attention(3, 4, 2, head_size, 16, 4096, num_splits, seed=head_size + num_splits)


def _laid_out(x, form):
    """The values of [B, H, T, D] tensor x in another memory layout."""
    b, h, t, d = x.shape
    if form == "bhtd":
        return x.to(DEV).contiguous()
    if form == "bthd":
        return x.to(DEV).transpose(1, 2).contiguous().transpose(1, 2)
    if form == "padded":  # rows of a wider buffer
        wide = torch.zeros((b, h, t + 3, d + 8), dtype=x.dtype, device=DEV)
        wide[:, :, :t, :d] = x.to(DEV)
        return wide[:, :, :t, :d]
    wide = torch.zeros((b, h, t, d + 1), dtype=x.dtype, device=DEV)  # "odd": rows not 16-aligned
    wide[..., 1:] = x.to(DEV)
    return wide[..., 1:]


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("B, Hq, Hk, M, N, causal, form", [
    (1, 2, 2, 17, 1, False, "bhtd"),      # the fewest rows, one key
    (2, 6, 2, 43, 65, True, "bthd"),      # 129 rows: a second work-group with one row
    (1, 8, 1, 16, 64, True, "padded"),    # 128 rows, one whole tile
    (1, 3, 1, 11, 63, True, "bhtd"),      # 33 rows: a second wave with one row
    (2, 4, 4, 127, 127, True, "odd"),     # realigned by a copy, short of a tile
    (8, 16, 8, 300, 193, True, "bthd"),   # M > N, every work-group resident at once
    (1, 4, 2, 40, 2100, True, "padded"),  # splits, the last one ragged
    (1, 8, 2, 5, 385, True, "bhtd"),      # short splits of few keys, the last of one key
    (2, 8, 1, 4, 257, False, "bthd"),     # at head dim 256 already here, unsplit otherwise
    (3, 3, 1, 200, 1600, False, "bhtd"),  # a batch that is not a multiple of the XCDs
])
def test_flash_attention_many_rows(D, B, Hq, Hk, M, N, causal, form):
    """More than 16 query rows per KV head (128 per work-group, 32 per wave, 32- or 64-key
    tiles): edges of rows, tiles and splits, each layout, both dtypes, both signs of the
    scale.  Same rule and lse bar as the other contiguous decodes."""
    need_gpu()
    for dtype, scale in ((torch.float16, D ** -0.5), (torch.bfloat16, -D ** -0.5)):
        q, k, v = _splitkv_inputs(B, Hq, Hk, M, N, D, dtype, "BHTD", 1.0, D + M + N)
        o_ref, lse_ref = go.flash_attention_ref(q, k, v, causal, sm_scale=scale, upcast=True)
        o_low, _ = go.flash_attention_ref(q, k, v, causal, sm_scale=scale, upcast=False)
        o, lse, _, _, _ = flag_attn.flash_attention(
            *(_laid_out(x, form) for x in (q, k, v)), causal, scale, return_log_normalizer=True)
        torch.cuda.synchronize()
        o, lse = o.cpu(), lse.cpu()
        assert bool(torch.isfinite(o).all())
        assert_lowp_rule(o, o_ref, o_low)
        assert torch.equal(torch.isneginf(lse), torch.isneginf(lse_ref))
        fin = ~torch.isneginf(lse_ref)
        assert float((lse[fin] - lse_ref[fin]).abs().max()) <= 1e-3


def test_flash_attention_many_rows_late_maximum():
    """Scores that keep growing along the keys (each tile's maximum far above the one before):
    the accumulators are rescaled at every tile, and no probability overflows fp16."""
    need_gpu()
    q, k, v = _splitkv_inputs(1, 2, 1, 40, 700, 64, torch.float16, "BHTD", 1.0, 5)
    q[..., 0], k[..., 0] = 8.0, torch.arange(700, dtype=torch.float16) / 16
    o_ref, lse_ref = go.flash_attention_ref(q, k, v, False, upcast=True)
    o_low, _ = go.flash_attention_ref(q, k, v, False, upcast=False)
    o, lse, _, _, _ = flag_attn.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), False,
                                                return_log_normalizer=True)
    torch.cuda.synchronize()
    assert_lowp_rule(o.cpu(), o_ref, o_low)
    assert float((lse.cpu() - lse_ref).abs().max()) <= 1e-3


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("M, N", [(40, 100), (17, 2100)])  # ragged tiles; short and long splits
def test_flash_attention_many_rows_scale_zero(D, M, N):
    """sm_scale 0 weighs every visible key alike, also where a tile has masked keys (0 times
    a masked score must not become NaN): out is the mean of the visible V rows, lse the log of
    their number."""
    need_gpu()
    for dtype, causal, scale in ((torch.float16, True, 0.0), (torch.bfloat16, False, -0.0)):
        q, k, v = _splitkv_inputs(1, 2, 1, M, N, D, dtype, "BHTD", 1.0, D + N)
        o_ref, lse_ref = go.flash_attention_ref(q, k, v, causal, sm_scale=scale, upcast=True)
        o_low, _ = go.flash_attention_ref(q, k, v, causal, sm_scale=scale, upcast=False)
        o, lse, _, _, _ = flag_attn.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), causal, scale,
                                                    return_log_normalizer=True)
        torch.cuda.synchronize()
        assert_lowp_rule(o.cpu(), o_ref, o_low)
        assert float((lse.cpu() - lse_ref).abs().max()) <= 1e-5  # log of a number up to 2,100


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("dtype, amp", [
    (torch.float16, 30.0),       # largest scores of about 2^12 in log2 units
    (torch.float16, 300.0),      # of 2^19
    (torch.float16, 10000.0),    # of 2^29: their rounding alone is past fp16's range
    (torch.bfloat16, 300000.0),  # of 2^39, and past bf16's
])
def test_flash_attention_many_rows_large_scores(D, dtype, amp):
    """Scores far apart: the largest takes all the weight.  Its exponent has to be 0 whatever
    the size of the scores, so that out is its V row to the bit and lse the score itself."""
    need_gpu()
    for causal, sign, N in ((True, 1, 700), (False, 1, 2100), (False, -1, 300)):
        q, k, v = _splitkv_inputs(1, 2, 1, 40, N, D, torch.float32, "BHTD", 1.0, D + N)
        q, k, v = (amp * q).to(dtype), (amp * k).to(dtype), v.to(dtype)
        scale = sign * D ** -0.5
        s = torch.matmul(q.double(), k.double().transpose(2, 3).contiguous()) * scale
        if causal:
            s = s.masked_fill(~torch.ones(40, N, dtype=torch.bool).tril(N - 40), float("-inf"))
        top, at = s.topk(2, dim=-1)
        # rows whose two best scores an fp32 sum over D products, with its scale, tells apart
        # by the 40 that leave e^-40 to all others
        size = (q.double().norm(dim=-1) * k.double().norm(dim=-1).max() * abs(scale))
        clear = top[..., 0] - top[..., 1] > 40 + (D + 2) * 2.0 ** -23 * size
        assert float(clear.float().mean()) > 0.5  # most rows count
        o, lse, _, _, _ = flag_attn.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), causal, scale,
                                                    return_log_normalizer=True)
        torch.cuda.synchronize()
        want = v[0, 0][at[..., 0]]
        assert torch.equal(o.cpu()[clear], want[clear])
        err = (lse.cpu().double() - top[..., 0]).abs()
        assert bool((err <= (D + 2) * 2.0 ** -23 * size)[clear].all())


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("N", [100, 500, 1536, 2100])  # both sides of the halves rule
def test_flash_attention_many_rows_error(D, N):
    """64 query rows at once are as close to the 64-bit result as 16 rows at a time (the 16-row
    kernel; 256 pairs, so neither splits).  Both round P and the output to 16 bits, errors that
    are independent from key to key: over a million output values their 2-norm varies by under
    0.1%, a reference that leaves more of the large P inexact adds 1% to 6%."""
    need_gpu()
    for dtype in (torch.bfloat16, torch.float16):
        gen = torch.Generator(device=DEV).manual_seed(D + N)
        q, k, v = (torch.randn((4, 64, t, D), device=DEV, generator=gen).to(dtype)
                   for t in (64, N, N))
        many = flag_attn.flash_attention(q, k, v)
        few = torch.cat([flag_attn.flash_attention(c, k, v) for c in q.split(16, dim=2)], dim=2)
        err = {"many": 0.0, "few": 0.0}
        for b in range(4):
            s = torch.matmul(q[b].double(), k[b].double().transpose(1, 2).contiguous()) * D ** -0.5
            exact = torch.matmul(torch.softmax(s, dim=-1), v[b].double())
            for name, o in (("many", many), ("few", few)):
                err[name] += float((o[b].double() - exact).square().sum())
        say(f"D={D} N={N} {dtype}: many / few {(err['many'] / err['few']) ** 0.5:.4f}")
        assert err["many"] <= 1.005 ** 2 * err["few"]


@pytest.mark.parametrize("B, M, N", [(0, 40, 100), (0, 40, 500), (0, 1, 100), (0, 1, 3000),
                                     (0, 40, 3000), (2, 0, 100), (2, 0, 3000)])
def test_empty_batch_or_query_is_the_librarys_argument_error(B, M, N):
    """No sequence or no query position: the library's argument check answers, whatever the
    number of keys (no split rule divides by the empty extent before it)."""
    need_gpu()
    q, k = (torch.zeros((B, h, t, 64), dtype=torch.float16, device=DEV) for h, t in ((4, M), (2, N)))
    for call in (flag_attn.flash_attention, flag_attn.flash_attention_split_kv):
        with pytest.raises(RuntimeError, match="must be >= 1"):
            call(q, k, k)
    if M == 1:
        lens = torch.zeros((0,), dtype=torch.int32, device=DEV)
        cache = torch.zeros((4, 2, 16, 64), dtype=torch.float16, device=DEV)
        with pytest.raises(RuntimeError, match="must be >= 1"):
            flag_attn.paged_attention(q[:, :, 0], cache, cache, lens, lens.new_zeros((0, 8)), 1.0, N)


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("N", [300, 2100])  # references per half and per tile
def test_flash_attention_many_rows_huge_values(D, N):
    """One V row of the largest finite bf16 value, of any weight: the sums of a row never grow
    past the weights' own, whatever the maxima of the tiles after it."""
    need_gpu()
    q, k, v = _splitkv_inputs(1, 4, 2, 40, N, D, torch.bfloat16, "BHTD", 1.0, D + N)
    v[:, 0, 50], v[:, 1, 7] = torch.finfo(torch.bfloat16).min, torch.finfo(torch.bfloat16).max
    o = flag_attn.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV)).cpu()
    kd, vd = (x.double().repeat_interleave(2, dim=1) for x in (k, v))
    p = torch.softmax(torch.matmul(q.double(), kd.transpose(2, 3).contiguous()) * D ** -0.5, dim=-1)
    ref = torch.matmul(p, vd)
    # P and out round to 8 bits (2^-9 each), the scores' own error is far below
    assert bool(((o.double() - ref).abs() <= 2.0 ** -7 * ref.abs()).all())


@pytest.mark.parametrize("D, P, N, same", [
    (64, 8, 64, False), (64, 8, 65, True), (64, 8, 256, True),  # one tile; the edges
    (64, 64, 200, True), (64, 72, 200, False),   # 256 and 288 work-groups of 16 rows
    (128, 4, 192, False), (128, 4, 193, True), (256, 4, 256, True),
    (128, 5, 200, False), (256, 5, 200, False),  # 20 of them
])
def test_flash_attention_few_keys(D, P, N, same):
    """Up to 256 keys: many rows run as blocks of 16 rows, with the bits of calls of 16 rows,
    where that is the faster kernel; outside, the many-row kernel."""
    need_gpu()
    gen = torch.Generator(device=DEV).manual_seed(P + N)
    q, k, v = (torch.randn((1, P, t, D), device=DEV, generator=gen).half() for t in (64, N, N))
    o = flag_attn.flash_attention(q, k, v)
    parts = torch.cat([flag_attn.flash_attention(c, k, v) for c in q.split(16, dim=2)], dim=2)
    assert torch.equal(o, parts) == same
    ref, _ = go.flash_attention_ref(q.cpu(), k.cpu(), v.cpu(), False, upcast=True)
    low, _ = go.flash_attention_ref(q.cpu(), k.cpu(), v.cpu(), False, upcast=False)
    assert_lowp_rule(o.cpu(), ref, low)
