"""Performance cases of the framework: the calls that a decoding or prefilling program makes
through ``flag_attn``, over the sizes that it makes them at.

A case is a dict of plain values; ``op`` names the operation:

* ``mla``     one MLA decode step over a bf16 paged latent cache: scheduler metadata + decode
              (a serving loop computes both every step, since the lengths change every step);
* ``sparse``  the same step over the top-k token lists of each query token, bf16 or fp8 rows;
* ``topk``    the index producer in front of a sparse step;
* ``write``   new tokens written into the paged latent cache (prefill or decode sized);
* ``paged``   grouped-query decode of one token per sequence over a paged K/V cache;
* ``splitkv`` flash decoding over contiguous K/V (long context, few sequences);
* ``flash``   ``flash_attention`` with several query positions: speculative verification,
              chunked prefill and whole-prompt prefill.

Sequence lengths are a fixed ragged spread of the case's range (so that a case's work does
not depend on the seed); the seed decides which sequence has which length, and every value,
page and index.
"""
import math
from statistics import NormalDist

import torch

import flag_attn

PAGE = 64
D_QK, D_V = 576, 512
MLA_SCALE = 192 ** -0.5
DEV = "cuda"
MAX_CACHE_BYTES = 2.2e9  # drawn GQA / flash cases: K and V together
FP8_MAX = 448.0


def listed():
    return [
        # two short sequences, 16 query heads: a lightly loaded server, all launch latency
        dict(name="mla_h16_b2_len384", op="mla", batch=2, heads=16, s_q=1, len_lo=256,
             len_hi=384, skew=False, causal=False),
        # one rank of an 8-way tensor-parallel model of 128 heads
        dict(name="mla_h16_b64_len8k", op="mla", batch=64, heads=16, s_q=1, len_lo=4096,
             len_hi=8192, skew=False, causal=False),
        # all 128 heads on one GPU (data-parallel attention), a full batch: the headline case
        dict(name="mla_h128_b64_len8k", op="mla", batch=64, heads=128, s_q=1, len_lo=4096,
             len_hi=8192, skew=False, causal=False),
        # multi-token prediction: two query tokens, a few sequences far longer than the rest
        dict(name="mla_h128_b32_sq2_skew", op="mla", batch=32, heads=128, s_q=2, len_lo=128,
             len_hi=65536, skew=True, causal=True),
        # sparse decode, 2,048 of 32,768 tokens, bf16 rows
        dict(name="sparse_bf16_b64_top2048", op="sparse", batch=64, heads=128, s_q=1, fp8=False,
             length=32768, topk=2048),
        # sparse decode over the quantised cache, 65,536 tokens per sequence
        dict(name="sparse_fp8_b128_top2048", op="sparse", batch=128, heads=128, s_q=1, fp8=True,
             length=65536, topk=2048),
        # the indices of the step above: long score rows, ragged lengths
        dict(name="topk_b128_len64k", op="topk", batch=128, s_q=1, length=65536, len_lo=32768,
             topk=2048),
        # a prefill's tokens quantised into the cache
        dict(name="write_fp8_t131072", op="write", tokens=131072, fp8=True, slots64=True),
        # a few short chats with grouped-query attention, 16-token pages
        dict(name="paged_b8_g8_d128_ctx1k", op="paged", batch=8, h_q=32, h_kv=4, d=128, block=16,
             len_lo=97, len_hi=1000, fp16=True),
        # a full batch of long sequences
        dict(name="paged_b64_g8_d128_ctx8k", op="paged", batch=64, h_q=64, h_kv=8, d=128,
             block=16, len_lo=8192, len_hi=8192, fp16=True),
        # long-context flash decoding, multi-head, an odd context
        dict(name="splitkv_b2_h16_ctx131k", op="splitkv", batch=2, h_q=16, h_kv=16, d=128,
             n=131001, fp16=True),
        # chunked prefill: 2,048 new tokens behind a 1,901-token prefix
        dict(name="flash_b2_h32_m2048_n3949", op="flash", batch=2, h_q=32, h_kv=8, d=128, m=2048,
             n=3949, causal=True, fp16=False, lse=True, bthd=True),
    ]


def _log_int(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(("mla", "mla", "mla", "sparse", "sparse", "topk", "write", "paged", "paged",
                     "splitkv", "flash", "flash"))
    if op == "mla":
        batch = _log_int(rng, 1, 128)
        heads = rng.choice((16, 16, 32, 64, 128))
        s_q = rng.choice((1, 1, 1, 2, 4))
        # at most the token-heads of the largest listed case
        most = max(64, min(65536, 400000 // batch, 64 * 8192 * 128 // (batch * heads * s_q)))
        hi = _log_int(rng, 64, most)
        return dict(op=op, batch=batch, heads=heads, s_q=s_q, len_lo=max(1, int(hi * rng.random())),
                    len_hi=hi, skew=False, causal=s_q > 1)
    if op == "sparse":
        batch = _log_int(rng, 1, 128)
        heads = rng.choice((16, 32, 64, 128))
        s_q = 1 if heads * batch > 8192 else rng.choice((1, 1, 2))
        topk = rng.choice((256, 512, 1024, 2048))
        fp8 = rng.random() < 0.5
        length = _log_int(rng, topk, min(65536, 64 * 65536 // batch))
        return dict(op=op, batch=batch, heads=heads, s_q=s_q, fp8=fp8, length=length, topk=topk)
    if op == "topk":
        length = _log_int(rng, 512, 65536)
        return dict(op=op, batch=_log_int(rng, 1, 128), s_q=rng.choice((1, 1, 2)) if
                    length < 32768 else 1, length=length,
                    len_lo=max(1, int(length * rng.uniform(0.3, 1.0))),
                    topk=rng.choice((256, 512, 1024, 2048)))
    if op == "write":
        return dict(op=op, tokens=_log_int(rng, 1, 131072), fp8=rng.random() < 0.5,
                    slots64=rng.random() < 0.5)
    d = rng.choice((64, 128, 128, 256))
    h_kv = rng.choice((1, 2, 4, 8, 16))
    group = rng.choice((1, 4, 8)) if h_kv < 16 else rng.choice((1, 4))
    h_q = h_kv * group
    fp16 = rng.random() < 0.5
    if op == "paged":
        batch = _log_int(rng, 1, 64)
        hi = _log_int(rng, 64, min(16384, int(MAX_CACHE_BYTES / (4 * d * h_kv * batch))))
        return dict(op=op, batch=batch, h_q=h_q, h_kv=h_kv, d=d,
                    block=rng.choice((16, 16, 32, 64, 128)),
                    len_lo=max(1, int(hi * rng.random())), len_hi=hi, fp16=fp16)
    if op == "splitkv":
        batch = _log_int(rng, 1, 8)
        n = _log_int(rng, 256, min(131072, int(MAX_CACHE_BYTES / (4 * d * h_kv * batch))))
        return dict(op=op, batch=batch, h_q=h_q, h_kv=h_kv, d=d, n=n, fp16=fp16)
    batch = _log_int(rng, 1, 16)
    m = _log_int(rng, 2, 4096)
    # at most the products of the largest listed case
    most = max(16, int(32 * 2048 * 5950 * 128 / (batch * h_q * d * m)))
    most = min(most, 16384, int(MAX_CACHE_BYTES / (4 * d * h_kv * batch)))
    m = min(m, most)
    return dict(op=op, batch=batch, h_q=h_q, h_kv=h_kv, d=d, m=m,
                n=m if rng.random() < 0.4 else _log_int(rng, m, most),
                causal=rng.random() < 0.75, fp16=fp16, lse=rng.random() < 0.5,
                bthd=rng.random() < 0.5)


def _lens(case):
    """The case's lengths, shortest first: evenly spaced over its range, or log-normal
    (median 4,096, sigma 1, clipped to the range) at even steps of the distribution."""
    b, lo, hi = case["batch"], case["len_lo"], case["len_hi"]
    if case.get("skew"):
        at = [NormalDist().inv_cdf((i + 0.5) / b) for i in range(b)]
        return [max(lo, min(hi, int(round(4096 * math.exp(z))))) for z in at]
    return [lo + int(round((hi - lo) * i / max(1, b - 1))) for i in range(b)] if b > 1 else [hi]


class _Source:
    """Random values on the GPU and choices on the host, from one seed."""

    def __init__(self, seed):
        self.gpu = torch.Generator(device=DEV).manual_seed(seed)
        self.cpu = torch.Generator().manual_seed(seed)

    def normal(self, shape, dtype):
        return torch.randn(shape, generator=self.gpu, device=DEV, dtype=dtype)

    def lens(self, case):
        ls = torch.tensor(_lens(case), dtype=torch.int32)
        return ls[torch.randperm(len(ls), generator=self.cpu)]

    def table(self, lens, block):
        """(block table, pages): every sequence's pages, scattered over the pool."""
        nblk = [-(-int(x) // block) for x in lens]
        perm = torch.randperm(sum(nblk), generator=self.cpu).to(torch.int32)
        bt = torch.zeros((len(nblk), max(nblk)), dtype=torch.int32)
        at = 0
        for i, n in enumerate(nblk):
            bt[i, :n] = perm[at:at + n]
            at += n
        return bt.to(DEV), at


def _fp8_rows(src, pages):
    """Quantised cache rows: e4m3 codes of unit normal latents with the 128-dim tiles' scales
    amax / 448, then the bf16 rope dims."""
    kc = torch.empty((pages, PAGE, 1, 656), dtype=torch.uint8, device=DEV)
    for c0 in range(0, pages, 4096):
        n = min(pages, c0 + 4096) - c0
        lat = src.normal((n, PAGE, 1, 4, 128), torch.bfloat16).float()
        sc = lat.abs().amax(-1, keepdim=True) / FP8_MAX
        row = kc[c0:c0 + n]
        row[..., :512] = (lat / sc).to(torch.float8_e4m3fn).view(torch.uint8).view(n, PAGE, 1, 512)
        row[..., 512:528] = sc.view(n, PAGE, 1, 4).contiguous().view(torch.uint8)
        row[..., 528:] = src.normal((n, PAGE, 1, 64), torch.bfloat16).view(torch.uint8)
    return kc


def prepare(case, seed):
    src = _Source(seed)
    op = case["op"]
    if op in ("mla", "sparse"):
        b, s_q, h = case["batch"], case["s_q"], case["heads"]
        lens = src.lens(case) if op == "mla" else torch.full((b,), case["length"], dtype=torch.int32)
        bt, pages = src.table(lens, PAGE)
        st = dict(op=op, lens=lens.to(DEV), bt=bt, s_q=s_q, h=h, causal=case.get("causal", False),
                  fp8=case.get("fp8", False), indices=None, topk=None,
                  q=src.normal((b, s_q, h, D_QK), torch.bfloat16))
        if st["fp8"]:
            st["kc"] = _fp8_rows(src, pages)
        else:
            st["kc"] = src.normal((pages, PAGE, 1, D_QK), torch.bfloat16)
        if op == "sparse":
            # distinct tokens in no order, about 2% of the slots empty
            n, k = case["length"], case["topk"]
            r = torch.rand((b * s_q, n), generator=src.gpu, device=DEV)
            idx = torch.topk(r, k, dim=1).indices.to(torch.int32)
            drop = torch.rand((b * s_q, k), generator=src.gpu, device=DEV) < 0.02
            st["indices"] = torch.where(drop, torch.full_like(idx, -1), idx).view(b, s_q, k)
            st["topk"] = k
        return st
    if op == "topk":
        b = case["batch"]
        lens = src.lens(dict(batch=b, len_lo=case["len_lo"], len_hi=case["length"]))
        return dict(op=op, scores=src.normal((b, case["s_q"], case["length"]), torch.float32),
                    lens=lens.to(DEV), topk=case["topk"], causal=case["s_q"] > 1)
    if op == "write":
        t = case["tokens"]
        pages = -(-t // PAGE)
        slots = torch.randperm(pages * PAGE, generator=src.cpu)[:t]
        return dict(op=op, kv_c=src.normal((t, D_V), torch.bfloat16),
                    k_pe=src.normal((t, D_QK - D_V), torch.bfloat16), fp8=case["fp8"],
                    slots=slots.to(torch.int64 if case["slots64"] else torch.int32).to(DEV),
                    cache=torch.zeros((pages, PAGE, 1, 656 if case["fp8"] else D_QK), device=DEV,
                                      dtype=torch.uint8 if case["fp8"] else torch.bfloat16))
    dt = torch.float16 if case["fp16"] else torch.bfloat16
    b, h_q, h_kv, d = case["batch"], case["h_q"], case["h_kv"], case["d"]
    if op == "paged":
        lens = src.lens(case)
        bt, pages = src.table(lens, case["block"])
        shape = (pages, h_kv, case["block"], d)
        return dict(op=op, q=src.normal((b, h_q, d), dt), k=src.normal(shape, dt),
                    v=src.normal(shape, dt), lens=lens.to(DEV), bt=bt, scale=d ** -0.5,
                    most=int(lens.max()))
    m = case.get("m", 1)
    if case.get("bthd"):  # the projections' own layout, seen as [B, H, T, D]
        q = src.normal((b, m, h_q, d), dt).transpose(1, 2)
        k = src.normal((b, case["n"], h_kv, d), dt).transpose(1, 2)
        v = src.normal((b, case["n"], h_kv, d), dt).transpose(1, 2)
    else:
        q = src.normal((b, h_q, m, d), dt)
        k = src.normal((b, h_kv, case["n"], d), dt)
        v = src.normal((b, h_kv, case["n"], d), dt)
    return dict(op=op, q=q, k=k, v=v, causal=case.get("causal", False), lse=case.get("lse", False))


def run(st):
    op = st["op"]
    if op in ("mla", "sparse"):
        md, ns = flag_attn.get_mla_metadata(st["lens"], st["s_q"] * st["h"], 1,
                                            num_heads_q=st["h"], topk=st["topk"])
        out, lse = flag_attn.flash_mla_with_kvcache(
            st["q"], st["kc"], st["bt"], st["lens"], D_V, md, ns, MLA_SCALE, st["causal"],
            is_fp8_kvcache=st["fp8"], indices=st["indices"])
        return {"out": out, "lse": lse}
    if op == "topk":
        return {"indices": flag_attn.topk_indices(st["scores"], st["lens"], st["topk"],
                                                  st["causal"])}
    if op == "write":
        flag_attn.concat_and_cache_mla(st["kv_c"], st["k_pe"], st["cache"], st["slots"], st["fp8"])
        return {"cache": st["cache"]}
    if op == "paged":
        return {"out": flag_attn.paged_attention(st["q"], st["k"], st["v"], st["lens"], st["bt"],
                                                 st["scale"], st["most"])}
    if op == "splitkv":
        return {"out": flag_attn.flash_attention_split_kv(st["q"], st["k"], st["v"])}
    if st["lse"]:
        out, lse, *_ = flag_attn.flash_attention(st["q"], st["k"], st["v"], st["causal"],
                                                 return_log_normalizer=True)
        return {"out": out, "lse": lse}
    return {"out": flag_attn.flash_attention(st["q"], st["k"], st["v"], st["causal"])}


def work(case):
    op = case["op"]
    if op in ("mla", "sparse"):
        b, s_q, h = case["batch"], case["s_q"], case["heads"]
        io = b * s_q * h * (2 * D_QK + 2 * D_V + 4)
        if op == "mla":
            tokens = sum(_lens(case))
            pairs = tokens * s_q
            if case["causal"]:
                pairs -= b * s_q * (s_q - 1) // 2
            data = tokens * 2 * D_QK + 4 * (tokens // PAGE + 2 * b)
        else:
            pairs = b * s_q * case["topk"] * 0.98
            data = pairs * (656 if case["fp8"] else 2 * D_QK) + 4 * b * s_q * case["topk"]
        return {"bytes": io + data, "flops": pairs * h * 2 * (D_QK + D_V)}
    if op == "topk":
        seen = sum(_lens(dict(batch=case["batch"], len_lo=case["len_lo"], len_hi=case["length"])))
        return {"bytes": 4 * case["s_q"] * (seen + case["batch"] * case["topk"]), "flops": 0}
    if op == "write":
        return {"bytes": case["tokens"] * (2 * D_QK + (656 if case["fp8"] else 2 * D_QK)
                                           + (8 if case["slots64"] else 4)), "flops": 0}
    b, h_q, h_kv, d = case["batch"], case["h_q"], case["h_kv"], case["d"]
    m = case.get("m", 1)
    tokens = sum(_lens(case)) if op == "paged" else b * case["n"]
    pairs = tokens * m - (b * m * (m - 1) // 2 if case.get("causal") else 0)
    data = 4 * d * h_kv * tokens + 4 * d * b * h_q * m
    if op == "paged":
        data += 4 * (tokens // case["block"] + b)
    if case.get("lse"):
        data += 4 * b * h_q * m
    return {"bytes": data, "flops": 4 * d * h_q * pairs}


def tolerance(case):
    # indices and cache bytes are the same in any correct implementation
    if case["op"] in ("topk", "write"):
        return "exact"
    # bf16 operands, probabilities and outputs (and bf16 split partials of the MLA decode)
    if case["op"] in ("mla", "sparse") or not case["fp16"]:
        return {"rel": 1e-2, "max": 0.1}
    # fp16 operands, probabilities and outputs
    return {"rel": 2e-3, "max": 0.02}


def _attend(q, k, v, scale, hide=None):
    """64-bit attention of q [rows, D] over k [n, D], v [n, E]: (out, log-normaliser)."""
    s = (q @ k.t()) * scale
    if hide is not None:
        s = s.masked_fill(hide, -math.inf)
    lse = torch.logsumexp(s, dim=1)
    out = torch.exp(s - torch.where(lse.isinf(), torch.zeros_like(lse), lse)[:, None]) @ v
    return out, lse


def _latent_rows(st, b, tokens):
    """Cache rows of one sequence's tokens in 64 bits."""
    rows = st["bt"][b].long()[tokens // PAGE] * PAGE + tokens % PAGE
    if not st["fp8"]:
        return st["kc"].view(-1, D_QK)[rows].double()
    raw = st["kc"].view(-1, 656)[rows]
    lat = raw[:, :512].contiguous().view(torch.float8_e4m3fn).double().view(-1, 4, 128)
    sc = raw[:, 512:528].contiguous().view(torch.float32).double().view(-1, 4, 1)
    rope = raw[:, 528:].contiguous().view(torch.bfloat16).double()
    return torch.cat([(lat * sc).view(-1, 512), rope], dim=1)


def exact(case, seed):
    op = case["op"]
    if op == "topk" or (op == "write" and case["fp8"]):
        return None  # whole numbers
    st = prepare(case, seed)
    if op == "write":
        rows = torch.zeros_like(st["cache"]).view(-1, D_QK).double()
        rows[st["slots"].long()] = torch.cat([st["kv_c"], st["k_pe"]], dim=1).double()
        return {"cache": rows.view_as(st["cache"])}
    if op in ("mla", "sparse"):
        q = st["q"].double()
        b, s_q, h, _ = q.shape
        out = torch.empty((b, s_q, h, D_V), dtype=torch.float64, device=DEV)
        lse = torch.empty((b, h, s_q), dtype=torch.float64, device=DEV)
        for i in range(b):
            n = int(st["lens"][i])
            kv = _latent_rows(st, i, torch.arange(n, device=DEV)) if op == "mla" else None
            for s in range(s_q):
                if op == "mla":
                    seen = kv[:max(0, n - (s_q - 1 - s))] if st["causal"] else kv
                else:
                    idx = st["indices"][i, s].long()
                    seen = _latent_rows(st, i, idx[idx >= 0])
                out[i, s], lse[i, :, s] = _attend(q[i, s], seen, seen[:, :D_V], MLA_SCALE)
        return {"out": out, "lse": lse}
    q = st["q"].double()
    if op == "paged":
        out = torch.empty_like(q)
        block = st["k"].shape[2]
        group = q.shape[1] // st["k"].shape[1]
        for i in range(q.shape[0]):
            n = int(st["lens"][i])
            pages = st["bt"][i].long()[:-(-n // block)]
            for hk in range(st["k"].shape[1]):
                k, v = (st[x][pages, hk].reshape(-1, q.shape[2])[:n].double() for x in "kv")
                at = slice(hk * group, (hk + 1) * group)
                out[i, at], _ = _attend(q[i, at], k, v, st["scale"])
        return {"out": out}
    b, h_q, m, d = q.shape
    n, group = st["k"].shape[2], h_q // st["k"].shape[1]
    out = torch.empty((b, h_q, m, d), dtype=torch.float64, device=DEV)
    lse = torch.empty((b, h_q, m), dtype=torch.float64, device=DEV)
    hide = None
    if st["causal"]:  # the last query position sees every key
        hide = torch.ones((m, n), dtype=torch.bool, device=DEV).triu(n - m + 1)
    for i in range(b):
        for h in range(h_q):
            k, v = st["k"][i, h // group].double(), st["v"][i, h // group].double()
            out[i, h], lse[i, h] = _attend(q[i, h], k, v, d ** -0.5, hide)
    return {"out": out, "lse": lse} if st["lse"] else {"out": out}
