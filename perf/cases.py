"""The framework's work, as cases that can be timed and compared.

Each case is a dict of plain values; `op` names the path:

  dense        one decode step over a bf16 or fp8 KV cache
  kivi         one decode step over a 2/4-bit KIVI cache with a bf16 residual window
  kivi_pack    quantizing and packing a prefilled cache into that format
  pq           one decode step over product-quantized keys and values
  pq_paged     the same over a paged cache of sequences of different lengths, with
               outlier key channels and dense (bf16 or fp8) values
  pq_encode    encoding a prefilled cache into product-quantizer codes
  quest        one page-sparse decode step from kept page metadata
  sparse       the two-pass sparse decode step (score every key, per-head top-k, gather)
  token_topk   the group-shared token top-k decode step
  select       one query chunk of a sparse prefill (streaming top-k, then attention)

Caches hold N(0, 1) keys and values, as every workload of this repository
(bytes_amd/workloads.py); KIVI keys have a few channels eight times as large.
"""
import math

import torch

from bytes_amd import attention_kernels as AK
from bytes_amd import kivi as KV
from bytes_amd import pq as PQ
from bytes_amd import quest as QU
from bytes_amd import sparse as SP
from bytes_amd import sparse_attention as SA

BF16, F16, F32, F64, F8 = torch.bfloat16, torch.float16, torch.float32, torch.float64, torch.float8_e4m3fn
M_SUB = 8          # dims per product-quantizer subspace


def listed():
    return [
        # the smallest call: one sequence of a small model (14/2 heads of 64), latency and launches count
        {"name": "dense_b1_8k", "op": "dense", "dtype": "bf16", "B": 1, "Hq": 14, "Hk": 2, "D": 64, "L": 8192},
        # a small serving batch over an fp8 cache
        {"name": "dense_fp8_b4_16k", "op": "dense", "dtype": "fp8", "B": 4, "Hq": 28, "Hk": 4, "D": 128, "L": 16384},
        # the headline decode step: 2-bit KIVI, a small serving batch
        {"name": "kivi2_b4_16k", "op": "kivi", "bits": 2, "B": 4, "Hq": 28, "Hk": 4, "D": 128, "L": 16384, "R": 128},
        # 4-bit KIVI at the batch the reference's latency study quotes
        {"name": "kivi4_b32_16k", "op": "kivi", "bits": 4, "B": 32, "Hq": 64, "Hk": 8, "D": 128, "L": 16384, "R": 128},
        # building the headline step's cache after prefill
        {"name": "kivi_pack2_b4_16k", "op": "kivi_pack", "bits": 2, "dtype": "f16", "B": 4, "Hk": 4, "D": 128,
         "L": 16256},
        # one long sequence over product-quantized keys and values
        {"name": "pq_b1_32k", "op": "pq", "B": 1, "Hq": 28, "Hk": 4, "D": 128, "L": 32768, "K": 256},
        # serving: eight sequences of different lengths in a paged cache
        {"name": "pq_paged_b8_8k", "op": "pq_paged", "B": 8, "Hq": 28, "Hk": 4, "D": 128, "L": 8192, "K": 256, "C": 4,
         "block": 16, "dtype": "bf16"},
        # encoding a 32K-token prompt's keys (or values) of one layer
        {"name": "pq_encode_32k", "op": "pq_encode", "B": 1, "Hk": 4, "D": 128, "L": 32768, "K": 256},
        # page-sparse decode of one long sequence, 2048 of 32768 tokens
        {"name": "quest_b1_32k", "op": "quest", "B": 1, "Hq": 28, "Hk": 4, "D": 128, "L": 32768, "kb": 2048,
         "page": 16},
        # the two-pass decode at the reference's quoted batch, 4-bit score keys, 5% of the keys
        {"name": "sparse_int4_b32_16k", "op": "sparse", "bits": 4, "B": 32, "Hq": 64, "Hk": 8, "D": 128, "L": 16384,
         "frac": 0.05},
        # the largest: long-context token top-k over a 4 GiB cache
        {"name": "token_topk_b8_128k", "op": "token_topk", "bits": 16, "B": 8, "Hq": 24, "Hk": 8, "D": 128,
         "L": 131072, "kb": 1024},
        # the last query chunk of an 8K-token sparse prefill of the small model, 10% of the keys
        {"name": "select_q256_8k", "op": "select", "B": 1, "Hq": 14, "Hk": 2, "D": 64, "L": 8192, "Qc": 256,
         "kb": 819, "k_chunk": 2048},
    ]


# (query heads, KV heads, head dim) of the configurations, tests and harness of this repository
_HEADS = [(14, 2, 64), (28, 4, 128), (24, 8, 128), (64, 8, 128), (8, 1, 64), (32, 8, 128)]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["dense", "dense", "kivi", "kivi", "kivi_pack", "pq", "pq_paged", "pq_encode", "quest", "sparse",
                     "token_topk", "select"])
    Hq, Hk, D = rng.choice(_HEADS)
    B = _log_int(rng, 1, 32)
    c = {"op": op, "B": B, "Hq": Hq, "Hk": Hk, "D": D}
    if op == "dense":
        c["dtype"] = rng.choice(["bf16", "fp8"])
        c["L"] = _log_int(rng, 1000, min(131072, max(1001, 2 ** 29 // (B * Hk * D))))
    elif op == "kivi":
        c["bits"] = rng.choice([2, 4])
        c["R"] = rng.choice([32, 128, rng.randint(0, 128)])
        top = min(65536, max(1057, 2 ** 29 // (B * Hk * D)))
        c["L"] = _log_int(rng, 1024, top) // 32 * 32 + c["R"]
    elif op == "kivi_pack":
        del c["Hq"]
        c["bits"] = rng.choice([2, 4])
        c["dtype"] = rng.choice(["f16", "bf16"])
        c["L"] = _log_int(rng, 1024, min(32768, max(1057, 2 ** 28 // (B * Hk * D)))) // 32 * 32
    elif op == "pq":
        c["K"] = 256
        c["B"] = B = _log_int(rng, 1, 8)
        c["L"] = _log_int(rng, 1000, 65536 // B)
    elif op == "pq_paged":
        c["B"] = B = _log_int(rng, 1, 16)
        c["L"] = _log_int(rng, 1000, 65536 // B)
        c.update(K=256, C=rng.choice([1, 2, 4]), block=rng.choice([16, 32]), dtype=rng.choice(["bf16", "fp8"]))
    elif op == "pq_encode":
        del c["Hq"]
        c["K"] = rng.choice([256, 256, 64])
        c["B"] = B = _log_int(rng, 1, 4)
        c["L"] = _log_int(rng, 1000, 32768 // B)
    elif op == "quest":
        c["B"] = B = _log_int(rng, 1, 8)
        c["L"] = _log_int(rng, 2000, 65536)
        c["page"] = 16
        c["kb"] = max(16, int(c["L"] * rng.uniform(0.03, 0.15)))
    elif op == "sparse":
        c["bits"] = rng.choice([16, 8, 4, 2])
        c["L"] = _log_int(rng, 2000, min(65536, 2 ** 29 // (B * Hk * D)))
        c["frac"] = rng.choice([0.01, 0.02, 0.05, 0.1])
    elif op == "token_topk":
        c["bits"] = rng.choice([16, 8, 4, 2])
        c["B"] = B = _log_int(rng, 1, 8)
        c["L"] = _log_int(rng, 8192, 131072)
        c["kb"] = _log_int(rng, 128, min(4096, c["L"] // 8))
    else:
        c["B"] = 1
        c["Hq"], c["Hk"], c["D"] = Hq, Hk, D = rng.choice([(14, 2, 64), (28, 4, 128), (8, 1, 64)])
        c["L"] = _log_int(rng, 1500, 16384)
        c["Qc"] = rng.choice([64, 128, 256, rng.randint(16, 256)])
        c["kb"] = max(1, round(rng.choice([0.05, 0.1]) * c["L"]))
        c["k_chunk"] = rng.choice([2048, 4096])
    return c


# ---------------------------------------------------------------------------
# inputs: plain torch on the GPU, from the seed alone
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, dtype=BF16):
    return torch.randn(*shape, generator=g, device="cuda", dtype=dtype)


def _qkv(case, g):
    B, Hq, Hk, D, L = (case[n] for n in ("B", "Hq", "Hk", "D", "L"))
    return _randn(g, B, Hq, 1, D), _randn(g, B, Hk, L, D), _randn(g, B, Hk, L, D)


def _pack_last_dim(x, bits):
    """The KIVI format along the last dim: (int32 words, fp16 scale, fp16 min) per 32 elements."""
    lead, T = x.shape[:-1], x.shape[-1]
    code = torch.empty(*lead, T * bits // 32, dtype=torch.int32, device=x.device)
    scale = torch.empty(*lead, T // 32, dtype=F16, device=x.device)
    mn = torch.empty_like(scale)
    fpi = 32 // bits
    shift = torch.arange(fpi, device=x.device, dtype=torch.int64) * bits
    for b in range(x.shape[0]):                   # one batch row at a time: the fp32 copies stay small
        xg = x[b].float().reshape(*x.shape[1:-1], T // 32, 32)
        lo, hi = xg.amin(-1, keepdim=True), xg.amax(-1, keepdim=True)
        s = (hi - lo).clamp_min(1e-8) / (2 ** bits - 1)
        c = ((xg - lo) / s).round_().clamp_(0, 2 ** bits - 1).to(torch.int64).reshape(*x.shape[1:-1], T // fpi, fpi)
        w = (c << shift).sum(-1)
        code[b] = torch.where(w >= 2 ** 31, w - 2 ** 32, w).to(torch.int32)
        scale[b], mn[b] = s.squeeze(-1).to(F16), lo.squeeze(-1).to(F16)
    return code, scale, mn


def _unpack_last_dim(code, scale, mn, bits):
    """float64 values of _pack_last_dim's format."""
    fpi = 32 // bits
    shift = torch.arange(fpi, device=code.device, dtype=torch.int32) * bits
    c = (code.unsqueeze(-1) >> shift) & (2 ** bits - 1)
    c = c.reshape(*scale.shape, 32).to(F64)
    return (c * scale.to(F64).unsqueeze(-1) + mn.to(F64).unsqueeze(-1)).reshape(*scale.shape[:-1], -1)


def _pack_score_keys(k, bits):
    """The packed score-key format along head_dim: (uint8 codes, bf16 scale, bf16 min) per 32 dims."""
    B, Hk, S, D = k.shape
    per = 8 // bits
    out = torch.empty(B, Hk, S, D // per, dtype=torch.uint8, device=k.device)
    scale = torch.empty(B, Hk, S, D // 32, dtype=BF16, device=k.device)
    mn = torch.empty_like(scale)
    shift = torch.arange(per, device=k.device, dtype=torch.int32) * bits
    for b in range(B):
        xg = k[b].float().reshape(Hk, S, D // 32, 32)
        lo, hi = xg.amin(-1, keepdim=True), xg.amax(-1, keepdim=True)
        s = (hi - lo).clamp_min(1e-8) / (2 ** bits - 1)
        c = ((xg - lo) / s).round_().clamp_(0, 2 ** bits - 1).to(torch.int32).reshape(Hk, S, D // per, per)
        out[b] = (c << shift).sum(-1).to(torch.uint8)
        scale[b], mn[b] = s.squeeze(-1).to(BF16), lo.squeeze(-1).to(BF16)
    return out, scale, mn


def _score_keys64(p, scale, mn, bits):
    """float64 keys of one (b, KV head) of _pack_score_keys' format: [S, D]."""
    per = 8 // bits
    shift = torch.arange(per, device=p.device, dtype=torch.uint8) * bits
    c = ((p.unsqueeze(-1) >> shift) & (2 ** bits - 1)).reshape(p.shape[0], scale.shape[-1], 32).to(F64)
    return (c * scale.to(F64).unsqueeze(-1) + mn.to(F64).unsqueeze(-1)).reshape(p.shape[0], -1)


def _codebook(g, Hk, M, K):
    """Per-head codebooks whose codewords are training points: [Hk, M, K, 8] fp16."""
    return _randn(g, Hk, M, K, M_SUB).to(F16)


def _nearest(x, cb):
    """Codes [B, Hk, L, M] of x [B, Hk, L, D] against per-head codebooks."""
    B, Hk, L, D = x.shape
    M = D // M_SUB
    idx = torch.empty(B, Hk, L, M, dtype=torch.uint8, device=x.device)
    for h in range(Hk):
        for j in range(M):
            c = cb[h, j].float()
            xs = x[:, h, :, j * M_SUB:(j + 1) * M_SUB].float().reshape(-1, M_SUB)
            idx[:, h, :, j] = (0.5 * (c * c).sum(-1) - xs @ c.t()).argmin(-1).to(torch.uint8).reshape(B, L)
    return idx


def _lut(q, cb, scale):
    """[B, Hq, M, K] fp32: scale * q . codeword, per subspace."""
    B, Hq, _, D = q.shape
    Hk, M, K, _ = cb.shape
    qs = q.float().reshape(B, Hk, Hq // Hk, M, M_SUB)
    lut = (qs.unsqueeze(-2) * cb.float().reshape(1, Hk, 1, M, K, M_SUB)).sum(-1)
    return (lut * scale).reshape(B, Hq, M, K).contiguous()


def _lens(case):
    """Sequence lengths of a paged batch: from L down to about L/3, no two alike."""
    B, L = case["B"], case["L"]
    return [max(1, L - (2 * L // 3) * b // B - 7 * b) for b in range(B)]


def _inputs(case, seed):
    g = _gen(seed)
    op, D = case["op"], case["D"]
    x = {"case": case, "scale": 1.0 / math.sqrt(D)}
    if op in ("dense", "quest", "sparse", "token_topk"):
        x["q"], x["k"], x["v"] = _qkv(case, g)
    if op == "dense" and case["dtype"] == "fp8":
        x["k"], x["v"] = x["k"].to(F8), x["v"].to(F8)
    elif op in ("sparse", "token_topk"):
        if case["bits"] == 8:
            x["ks"] = x["k"].to(F8)
        elif case["bits"] < 8:
            x["ks"], x["ksc"], x["kmn"] = _pack_score_keys(x["k"], case["bits"])
    elif op == "kivi":
        q, k, v = _qkv(case, g)
        k[..., torch.randperm(D, generator=g, device="cuda")[:4]] *= 8
        Sq, bits = case["L"] - case["R"], case["bits"]
        x["q"], x["kr"], x["vr"] = q, k[:, :, Sq:].contiguous(), v[:, :, Sq:].contiguous()
        x["k"] = _pack_last_dim(k[:, :, :Sq].transpose(2, 3).contiguous().to(F16), bits)
        x["v"] = _pack_last_dim(v[:, :, :Sq].to(F16), bits)
    elif op == "kivi_pack":
        B, Hk, L = case["B"], case["Hk"], case["L"]
        dt = F16 if case["dtype"] == "f16" else BF16
        k, v = _randn(g, B, Hk, L, D), _randn(g, B, Hk, L, D)
        k[..., torch.randperm(D, generator=g, device="cuda")[:4]] *= 8
        x["kt"], x["v"] = k.transpose(2, 3).contiguous().to(dt), v.to(dt)
    elif op == "pq":
        q, k, v = _qkv(case, g)
        x["q"] = q
        x["kcb"], x["vcb"] = (_codebook(g, case["Hk"], D // M_SUB, case["K"]) for _ in range(2))
        x["ki"], x["vi"] = _nearest(k, x["kcb"]), _nearest(v, x["vcb"])
    elif op == "pq_paged":
        B, Hq, Hk, L, bs, C = (case[n] for n in ("B", "Hq", "Hk", "L", "block", "C"))
        nb = [(n + bs - 1) // bs for n in _lens(case)]
        total, most = sum(nb), max(nb)
        order = torch.randperm(total, generator=g, device="cuda").to(torch.int32)
        x["table"] = torch.full((B, most), -1, dtype=torch.int32, device="cuda")
        at = 0
        for b in range(B):
            x["table"][b, :nb[b]] = order[at:at + nb[b]]
            at += nb[b]
        x["lens"] = torch.tensor(_lens(case), dtype=torch.int32, device="cuda")
        cb = _codebook(g, Hk, D // M_SUB, case["K"])
        k = _randn(g, total, Hk, bs, D)
        x["ki"] = _nearest(k, cb)
        x["lut"] = _lut(_randn(g, B, Hq, 1, D), cb, x["scale"])
        x["ko"] = 4 * _randn(g, total, Hk, bs, C)
        x["qo"] = x["scale"] * _randn(g, B, Hq, C)
        v = _randn(g, total, Hk, bs, D)
        x["v"] = v.to(F8) if case["dtype"] == "fp8" else v
    elif op == "pq_encode":
        x["x"] = _randn(g, case["Hk"], case["B"], case["L"], D)
        x["cb"] = _codebook(g, case["Hk"], D // M_SUB, case["K"])
    elif op == "select":
        B, Hq, Hk, L, Qc = (case[n] for n in ("B", "Hq", "Hk", "L", "Qc"))
        x["q"] = _randn(g, B, Hq, Qc, D)
        x["k"], x["v"] = _randn(g, B, Hk, L, D), _randn(g, B, Hk, L, D)
        x["pos"] = torch.arange(L - Qc, L)
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    if case["op"] == "quest":
        x["meta"] = QU.quest_page_minmax(x["k"], case["page"])      # kept beside the cache
    return x


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(x):
    c = x["case"]
    op, sc = c["op"], x["scale"]
    if op == "dense":
        f = AK.decode_attn_fp8 if c["dtype"] == "fp8" else AK.decode_attn_bf16
        return f(x["q"], x["k"], x["v"], sc)
    if op == "kivi":
        return KV.kivi_decode_attn(x["q"], *x["k"], x["kr"], *x["v"], x["vr"], c["bits"], 32)
    if op == "kivi_pack":
        return [KV.quantize_and_pack_along_last_dim(x[n], 32, c["bits"]) for n in ("kt", "v")]
    if op == "pq":
        return PQ.decode_attn_pq_kv_fused(x["q"], x["kcb"], x["ki"], x["vi"], x["vcb"], sc)
    if op == "pq_paged":
        return PQ.paged_attn_pq_lut_asym(x["lut"], x["ki"], x["ko"], x["qo"], x["v"], x["table"], x["lens"],
                                         block_size=c["block"])
    if op == "pq_encode":
        return PQ.pq_encode(x["x"], x["cb"])
    if op == "quest":
        return QU.quest_decode(x["q"], x["k"], x["v"], c["kb"], sc, page=c["page"], meta=x["meta"])
    if op == "sparse":
        ks = x["k"] if c["bits"] == 16 else x["ks"]
        return SP.sparse_decode_scalar(x["q"], ks, x.get("ksc"), x.get("kmn"), x["k"], x["v"], c["frac"], sc,
                                       score_bits=c["bits"])
    if op == "token_topk":
        if c["bits"] == 16:
            return SP.token_topk_decode(x["q"], x["k"], x["v"], c["kb"], sc)
        return SP.token_topk_decode(x["q"], x["k"], x["v"], c["kb"], sc, k_score=x["ks"], score_scale=x.get("ksc"),
                                    score_zero=x.get("kmn"), score_bits=c["bits"] if c["bits"] < 8 else None)
    idx = SA.select_topk("exact", x["q"], x["k"], x["pos"], c["L"], c["kb"], c["k_chunk"], sc)
    return idx, SA.attend_topk(x["q"], x["k"], x["v"], idx, x["pos"], sc)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    op, B, Hk, D, L = (case[n] for n in ("op", "B", "Hk", "D", "L"))
    Hq = case.get("Hq", Hk)
    qo = 2 * B * Hq * D * 2                       # q in, out
    row = D * 2
    if op == "dense":
        es = 1 if case["dtype"] == "fp8" else 2
        return {"bytes": 2 * B * Hk * L * D * es + qo, "flops": 4 * B * Hq * L * D}
    if op == "kivi":
        R, Sq = case["R"], L - case["R"]
        per = 2 * (D * case["bits"] // 8 + D // 32 * 4)
        return {"bytes": B * Hk * (Sq * per + R * 2 * row) + qo, "flops": 4 * B * Hq * L * D}
    if op == "kivi_pack":
        n = 2 * B * Hk * L * D
        return {"bytes": n * 2 + n * case["bits"] // 8 + n // 32 * 4, "flops": 6 * n}
    M = D // M_SUB
    if op == "pq":
        return {"bytes": B * Hk * L * 2 * M + 2 * Hk * M * case["K"] * 16 + qo, "flops": 4 * B * Hq * L * D}
    if op == "pq_paged":
        n = sum(_lens(case))
        es = 1 if case["dtype"] == "fp8" else 2
        return {"bytes": n * Hk * (M + 2 * case["C"] + D * es) + B * Hq * M * case["K"] * 4 + n // case["block"] * 4
                + qo // 2, "flops": n * Hq * (2 * D + M + 2 * case["C"])}
    if op == "pq_encode":
        n = B * Hk * L
        return {"bytes": n * (row + M) + Hk * M * case["K"] * 16, "flops": n * M * case["K"] * 3 * M_SUB}
    if op == "quest":
        pages = (L + case["page"] - 1) // case["page"]
        kb = min(L, (case["kb"] + case["page"] - 1) // case["page"] * case["page"])
        # the rows are read once per KV head where its query heads pick the same pages, and once per query head
        # where they pick different ones: the expected union of independent picks
        G, f = Hq // Hk, kb / L
        rows = L * (1 - (1 - f) ** G)
        return {"bytes": int(B * Hk * (pages * 2 * row + rows * 2 * row) + qo),
                "flops": B * Hq * (4 * kb * D + 3 * pages * D)}
    if op in ("sparse", "token_topk"):
        keys = {16: 2 * D, 8: D, 4: D // 2 + D // 32 * 4, 2: D // 4 + D // 32 * 4}[case["bits"]]
        G = Hq // Hk
        if op == "sparse":
            kb = max(1, round(case["frac"] * L))
            rows = L * (1 - (1 - kb / L) ** G)
            extra = 0
        else:
            kb = rows = case["kb"]
            extra = B * Hk * kb * 4
        return {"bytes": int(B * Hk * (L * keys + rows * 2 * row) + qo + extra),
                "flops": B * Hq * (2 * L * D + 4 * kb * D)}
    Qc, kb = case["Qc"], case["kb"]
    return {"bytes": B * Hk * L * 2 * row + B * Hq * Qc * (2 * row + kb * 8),
            "flops": B * Hq * Qc * (2 * L * D + 4 * kb * D)}


def tolerance(case):
    op = case["op"]
    if op in ("kivi_pack", "pq_encode"):
        return "exact"                            # codes, scales and minima are whole values or single roundings
    if op == "pq":
        return {"rel": 1e-3, "max": 1e-2}         # fp16 output and probabilities: 2.1e-4 off 64 bits
    if op == "token_topk":
        # indices ascend: one key exchanged at a row's threshold (equal to the last fp32 digit) shifts the others
        return {"rel": 1e-2, "max": 5e-2, "differ": 0.01}
    if op == "select":
        # indices by score: neighbours whose fp32 scores agree to the last digits may change places
        return {"rel": 1e-2, "max": 5e-2, "differ": 2e-3}
    return {"rel": 1e-2, "max": 5e-2}             # bf16 outputs and probabilities: 2.1e-3 to 2.4e-3 off 64 bits


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _attend64(q, k, v, scale):
    """q [.., n, D], k, v [.., T, D] float64."""
    return torch.softmax((q @ k.transpose(-1, -2)) * scale, -1) @ v


def _top64(s, kb):
    return s.topk(kb, dim=-1).indices


def exact(case, seed):
    x = _inputs(case, seed)
    op, sc = case["op"], x["scale"]
    B, Hk, D, L = case["B"], case["Hk"], case["D"], case["L"]
    if op == "pq_encode":
        return None
    if op == "kivi_pack":
        got = []
        for n in ("kt", "v"):
            t = x[n]
            lo = torch.empty(*t.shape[:-1], t.shape[-1] // 32, dtype=F64, device=t.device)
            s = torch.empty_like(lo)
            for b in range(B):
                tg = t[b].to(F64).reshape(*t.shape[1:-1], -1, 32)
                lo[b] = tg.amin(-1)
                s[b] = (tg.amax(-1) - lo[b]).clamp_min(1e-8) / (2 ** case["bits"] - 1)
            got.append([None, s, lo])
        return got
    Hq = case["Hq"]
    G = Hq // Hk
    if op == "select":
        q = x["q"].to(F64)
        out = torch.empty_like(q)
        for b in range(B):
            for h in range(Hq):
                k, v = x["k"][b, h // G].to(F64), x["v"][b, h // G].to(F64)
                s = (q[b, h] @ k.t()) * sc
                pos = x["pos"].to(s.device).unsqueeze(-1)
                s.masked_fill_(torch.arange(L, device=s.device) > pos, -math.inf)
                top = s.topk(case["kb"], dim=-1)
                p = torch.softmax(top.values, -1)
                out[b, h] = torch.zeros_like(s).scatter_(1, top.indices, p) @ v
        return [None, out]
    out = torch.empty(B, Hq, 1, D, dtype=F64, device="cuda")
    if op == "pq_paged":
        M, bs = D // M_SUB, case["block"]
        for b, n in enumerate(_lens(case)):
            blocks = x["table"][b, :(n + bs - 1) // bs].long()
            rows = lambda t, hk: t[blocks, hk].to(F64).reshape(-1, t.shape[-1])[:n]    # noqa: E731
            for hk in range(Hk):
                codes = x["ki"][blocks, hk].reshape(-1, M)[:n].long()
                ko, v = rows(x["ko"], hk), rows(x["v"], hk)
                for h in range(hk * G, hk * G + G):
                    lut = x["lut"][b, h].to(F64)
                    s = lut.gather(1, codes.t()).sum(0) + ko @ x["qo"][b, h].to(F64)
                    out[b, h, 0] = torch.softmax(s, -1) @ v
        return out
    for b in range(B):
        for hk in range(Hk):
            q = x["q"][b, hk * G:hk * G + G, 0].to(F64)
            if op == "kivi":
                bits = case["bits"]
                kq = _unpack_last_dim(*(t[b, hk] for t in x["k"]), bits).t()
                vq = _unpack_last_dim(*(t[b, hk] for t in x["v"]), bits)
                k, v = torch.cat([kq, x["kr"][b, hk].to(F64)]), torch.cat([vq, x["vr"][b, hk].to(F64)])
            elif op == "pq":
                j = torch.arange(D // M_SUB, device="cuda")
                k, v = (x[cb][hk].to(F64)[j, x[i][b, hk].long()].reshape(L, D) for cb, i in (("kcb", "ki"),
                                                                                         ("vcb", "vi")))
            else:
                k, v = x["k"][b, hk].to(F64), x["v"][b, hk].to(F64)
            if op in ("dense", "kivi", "pq"):
                o = _attend64(q, k, v, sc)
            elif op == "quest":
                page = case["page"]
                n = (L + page - 1) // page
                kp = torch.cat([k, k[-1:].expand(n * page - L, D)]).reshape(n, page, D)
                lo, hi = kp.amin(1), kp.amax(1)
                bound = q.clamp_min(0) @ hi.t() + q.clamp_max(0) @ lo.t()
                pick = _top64(bound, min(n, max(1, -(-case["kb"] // page))))
                keep = torch.zeros(G, n, dtype=torch.bool, device="cuda").scatter_(1, pick, True)
                keep = keep.repeat_interleave(page, 1)[:, :L]
                o = torch.softmax(((q @ k.t()) * sc).masked_fill(~keep, -math.inf), -1) @ v
            else:
                ks = k
                if case["bits"] == 8:
                    ks = x["ks"][b, hk].to(F64)
                elif case["bits"] < 8:
                    ks = _score_keys64(x["ks"][b, hk], x["ksc"][b, hk], x["kmn"][b, hk], case["bits"])
                s = q @ ks.t()
                if op == "sparse":
                    pick = _top64(s, max(1, round(case["frac"] * L)))
                    keep = torch.zeros(G, L, dtype=torch.bool, device="cuda").scatter_(1, pick, True)
                    o = torch.softmax(((q @ k.t()) * sc).masked_fill(~keep, -math.inf), -1) @ v
                else:
                    pick = _top64(s.sum(0), case["kb"])
                    o = _attend64(q, k[pick], v[pick], sc)
            out[b, hk * G:hk * G + G, 0] = o
    return [out, None] if op == "token_topk" else out
