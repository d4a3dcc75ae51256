"""The metadata kernel's 32-bit and 64-bit partitions and its closed form for sparse decode,
against the spec, bit for bit."""
import ctypes
import random

import pytest
import torch

import flag_attn
import flagattention_amd as fa
from flagattention_amd import _lib
from oracle import mla_oracle as orc
from tests._helpers import need_gpu, say

pytestmark = pytest.mark.gpu


def _check(lens, parts, topk, overhead=None):
    ld = torch.tensor(lens, dtype=torch.int32, device="cuda")
    if overhead is None:
        overhead = fa.mla.overhead_blocks(bool(topk))
        md, ns = flag_attn.get_mla_metadata(ld, 16, 1, num_heads_q=16, topk=topk or None,
                                            num_sm_parts=parts)
    else:  # costs that only callers of the C ABI ask for
        md = torch.empty((parts, 8), dtype=torch.int32, device="cuda")
        ns = torch.empty((len(lens) + 1,), dtype=torch.int32, device="cuda")
        _lib.check(_lib.load().fa_mla_get_metadata(
            ld.data_ptr(), len(lens), topk, parts, overhead, md.data_ptr(), ns.data_ptr(),
            torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    want_md, want_ns = orc.metadata_spec(lens, parts, overhead, topk)
    assert md.cpu().tolist() == want_md and ns.cpu().tolist() == want_ns


@pytest.mark.parametrize("top", [64 * 2**17 - 64, 64 * 2**17 - 63, 2**31 - 1])
@pytest.mark.parametrize("B,parts", [(1, 256), (7, 1024), (63, 100)])
def test_lengths_around_the_32_bit_limit(top, B, parts):
    """One sequence of 2^17 - 1 blocks (32-bit), of 2^17 and of the longest length (64-bit)."""
    need_gpu()
    lens = [(i * 7919) % 5000 for i in range(B)]
    lens[B // 2] = top
    _check(lens, parts, 0)


@pytest.mark.parametrize("overhead", [0, 1, 65536, 65537])
@pytest.mark.parametrize("topk", [0, 300])
def test_other_overheads(overhead, topk):
    need_gpu()
    _check([100, 0, 4000, 64, 129], 37, topk, overhead)


def test_random_shapes():
    """Dense and sparse, 1..1024 parts, more and fewer parts than blocks, both thread counts."""
    need_gpu()
    rng = random.Random(5)
    for i in range(150):
        B = rng.choice((1, 2, 3, rng.randint(1, 70), rng.randint(1, 1100), 4096 if i < 2 else 5))
        parts = rng.choice((1, 7, 8, 255, 256, 257, 1024, rng.randint(1, 1024)))
        topk = rng.choice((0, 0, 1, 64, 65, 2048, rng.randint(1, 9000)))
        top = rng.choice((10, 700, 70000))
        lens = [rng.choice((0, 1, rng.randint(0, top))) for _ in range(B)]
        say(f"{i}: B={B} parts={parts} topk={topk} top={top}")
        _check(lens, parts, topk)
