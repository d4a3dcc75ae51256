"""GPU parity of the MLA decode with up to 32 query rows per KV stream (its own kernel:
csrc/fa_decode_few.hip) against the CPU oracle: the edges of its 16-row tiles, segments of
every tile count around its four-buffer ring, masks, strides, and scores far above the
softmax reference."""
import pytest
import torch

from oracle import mla_oracle as orc
from tests._helpers import (assert_close, dense_refs, need_gpu, run_dense, run_sparse, say,
                            sparse_refs)
from tests.test_gpu_decode import _plant_key

pytestmark = pytest.mark.gpu
SCALE = 192 ** -0.5
# 32-token tiles: 1 .. 9 of them, whole and one token into the next, and an empty sequence
LENS = [1, 32, 33, 64, 65, 97, 129, 0, 161, 193, 224, 288, 31]


@pytest.mark.parametrize("h_q,s_q,causal", [
    (1, 1, False), (15, 1, False), (16, 1, False), (17, 1, False), (31, 1, False),
    (32, 1, False), (8, 2, True), (5, 3, True), (8, 4, True), (16, 2, False), (33, 1, False),
])
@pytest.mark.parametrize("parts", [None, 1, 5])
def test_dense_rows_and_tile_counts(h_q, s_q, causal, parts):
    need_gpu()
    say(f"dense few h={h_q} s={s_q} causal={causal} parts={parts}")
    q, kc, bt, ld = orc.make_dense_inputs(len(LENS), h_q, s_q, LENS, seed=h_q * 8 + s_q,
                                          scale=1.0, extra_blocks=2)
    out, lse, _, _ = run_dense(q, kc, bt, ld, SCALE, causal, parts)
    assert_close(out, lse, *dense_refs(q, kc, bt, ld, SCALE, causal))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("h_q,s_q", [(1, 1), (16, 2), (17, 1), (32, 1), (33, 1)])
@pytest.mark.parametrize("topk,parts", [(1, None), (32, 1), (64, 1), (96, None), (100, 3),
                                        (160, 1), (192, 1), (500, None)])
def test_sparse_rows_and_tile_counts(fp8, h_q, s_q, topk, parts):
    need_gpu()
    say(f"sparse few fp8={fp8} h={h_q} s={s_q} topk={topk} parts={parts}")
    lens = [700, 1500]
    q, kc, bt, ld = orc.make_dense_inputs(2, h_q, s_q, lens, seed=h_q + topk, scale=1.0,
                                          extra_blocks=1)
    if fp8:
        kc = orc.make_fp8_cache(kc.shape[0], seed=topk + 7, lat_scale=1.0)
    idx = orc.make_sparse_indices(2, s_q, topk, lens, seed=topk + 3)
    out, lse = run_sparse(q, kc, bt, ld, idx, SCALE, fp8, parts)
    assert_close(out, lse, *sparse_refs(q, kc, bt, ld, idx, SCALE, fp8))


@pytest.mark.parametrize("h_q", [16, 32])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_dense_wide_score_spread(h_q, sign):
    """A key scoring > 2^64 above the first tile's row max rebases the row in place."""
    need_gpu()
    lens = [700, 300]
    q, kc, bt, ld = orc.make_dense_inputs(2, h_q, 1, lens, seed=77, scale=0.1)
    q.fill_(sign)
    _plant_key(kc, bt, 0, 500, 1.5)  # 90 log2 units above the first tile
    _plant_key(kc, bt, 1, 10, 1.5)   # in the first tile
    out, lse, _, _ = run_dense(q, kc, bt, ld, sign * SCALE, False, 1)
    ref_out, ref_lse, low = dense_refs(q, kc, bt, ld, sign * SCALE, False)
    assert float(ref_lse[0].min()) > 60.0
    assert_close(out, lse, ref_out, ref_lse, low)


def test_dense_strided_q_and_cache():
    """q rows and cache rows of wider buffers, pages out of order, a bad page id."""
    need_gpu()
    q, kc, bt, ld = orc.make_dense_inputs(2, 16, 2, [200, 130], seed=9, scale=1.0, extra_blocks=1)
    qw = torch.zeros((2, 2, 20, 592), dtype=q.dtype)
    qw[:, :, :16, :576] = q
    kw = torch.zeros((kc.shape[0], 64, 1, 584), dtype=kc.dtype)
    kw[..., :576] = kc
    ref = dense_refs(q, kc, bt, ld, SCALE, True)
    import flag_attn
    lens, table = ld.to("cuda"), bt.to("cuda")
    md, ns = flag_attn.get_mla_metadata(lens, 32, 1)
    out, lse = flag_attn.flash_mla_with_kvcache(qw.to("cuda")[:, :, :16, :576],
                                                kw.to("cuda")[..., :576], table, lens, 512, md,
                                                ns, SCALE, True)
    torch.cuda.synchronize()
    assert_close(out.cpu(), lse.cpu(), *ref)


@pytest.mark.parametrize("B,h_q,lens,parts", [
    (1, 16, [9000], None),               # one sequence over every part: 8 waves per row
    (3, 40, [2500, 0, 700], None),       # 85 parts per sequence at most, an empty sequence
    (12, 5, [900] * 11 + [1], 240),      # 20 per sequence: 4 waves; one of a single split
    (2, 130, [3000, 64], 18),            # 9 per sequence, more rows than a work-group
    (2, 16, [3000, 64], 16),             # 8 per sequence: one wave per row
])
def test_dense_combine_many_splits(B, h_q, lens, parts):
    """Split counts on both sides of the combine's choices of waves per row."""
    need_gpu()
    q, kc, bt, ld = orc.make_dense_inputs(B, h_q, 1, lens, seed=B + h_q, scale=1.0,
                                          extra_blocks=1)
    out, lse, _, _ = run_dense(q, kc, bt, ld, SCALE, False, parts)
    assert_close(out, lse, *dense_refs(q, kc, bt, ld, SCALE, False))


@pytest.mark.parametrize("h_q", [16, 32, 48])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("topk,parts", [(2047, 1), (2048, 1), (2048, 3), (2049, 1), (513, 1)])
def test_sparse_translation_limit(h_q, fp8, topk, parts):
    """Index lists on both sides of the in-kernel translation's limit and of its 512-slot
    rounds, with page ids outside the cache and ids past the length among them."""
    need_gpu()
    lens = [2600, 700]
    q, kc, bt, ld = orc.make_dense_inputs(2, h_q, 1, lens, seed=topk, scale=1.0, extra_blocks=1)
    if fp8:
        kc = orc.make_fp8_cache(kc.shape[0], seed=topk + 7, lat_scale=1.0)
    idx = torch.randint(-3, 2700, (2, 1, topk),
                        generator=torch.Generator().manual_seed(topk)).to(torch.int32)
    bt = bt.clone()
    bt[0, 3], bt[1, 0] = kc.shape[0], -1
    out, lse = run_sparse(q, kc, bt, ld, idx, SCALE, fp8, parts)
    assert_close(out, lse, *sparse_refs(q, kc, bt, ld, idx, SCALE, fp8))
