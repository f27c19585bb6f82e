"""Token scoring, deterministic top-k and gather attention vs the CPU oracle.

Scores and attention outputs: north_star tolerance (fp32 scores compared to
1e-3 absolute); top-k indices: bit-exact against the oracle run on the same
fp32 scores.
"""
import math

import pytest
import torch

from bytes_amd import sparse as SP
from bytes_amd import workloads as W
from oracle import reference as R

MAX_ABS, MEAN_ABS = 2e-2, 2e-3
SCORE_TOL = 1e-3
pytestmark = pytest.mark.gpu


def _check(out, ref, tag):
    d = (out.float().cpu() - ref.float()).abs()
    print(f"{tag}: max-abs {d.max():.3e} mean-abs {d.mean():.3e}", flush=True)
    assert d.max() <= MAX_ABS and d.mean() <= MEAN_ABS, tag


@pytest.mark.parametrize("B,Hq,Hk,S,D", [(2, 8, 2, 1000, 128), (1, 24, 8, 4099, 128), (2, 4, 4, 300, 64),
                                          (1, 40, 2, 777, 128)])
def test_score_per_head(dev, B, Hq, Hk, S, D):
    x = W.dense(B, Hq, Hk, D, S, seed=S)
    s = SP.sparse_score_scalar(x["q"].to(dev), x["k"].to(dev), 0.088)
    ref = R.sparse_score_scalar(x["q"], x["k"], 0.088)
    assert s.shape == (B, Hq, S) and s.dtype == torch.float32
    assert (s.cpu() - ref).abs().max() <= SCORE_TOL


@pytest.mark.parametrize("B,Hq,Hk,S", [(2, 24, 8, 5000), (1, 4, 1, 129), (1, 32, 2, 1024)])
def test_group_scores(dev, B, Hq, Hk, S):
    x = W.dense(B, Hq, Hk, 128, S, seed=S + 1)
    s = SP.group_scores(x["q"].to(dev), x["k"].to(dev), 0.088)
    ref = R.group_scores(x["q"], x["k"], 0.088)
    assert s.shape == (B, Hk, S)
    assert (s.cpu() - ref).abs().max() <= SCORE_TOL


def test_group_scores_long_ragged(dev):
    """A cache long enough that each wave of the score pass runs several
    iterations and stores whole batches of group sums, with a ragged last
    range (S = 200003), plain and with the fused selection histogram of the
    top-k pipeline: scores against the oracle, the pipeline's selection
    bit-exact against the oracle's top-k on the same scores."""
    B, Hq, Hk, S = 2, 24, 8, 200003
    x = W.dense(B, Hq, Hk, 128, S, seed=5)
    q, k, v = (x[n].to(dev) for n in ("q", "k", "v"))
    s = SP.group_scores(q, k, 0.088)
    ref = R.group_scores(x["q"], x["k"], 0.088)
    assert (s.cpu() - ref).abs().max() <= SCORE_TOL
    _, idx = SP.token_topk_decode(q, k, v, 1024, 0.088)
    assert torch.equal(idx.cpu().long(), R.topk_indices(s.cpu(), 1024, sorted_by_score=False))


@pytest.mark.parametrize("fp8,D", [(True, 128), (False, 64)])
def test_score_per_head_full_lds_buffer(dev, fp8, D):
    """Per-head scores (16 query heads on one KV head) on a row long enough
    that, on 256 CUs, each score workgroup's token range is the largest its
    LDS score buffer holds for 16 head rows (768 tokens for fp8 keys and for
    D = 64), with a ragged end: slices at the start, across workgroup
    boundaries and at the end against the oracle (fp8 keys widened to bf16,
    which is exact)."""
    B, Hq, Hk = 1, 16, 1
    S = 2048 * 768 + 555
    g = torch.Generator(device=dev).manual_seed(17)
    q = torch.randn(B, Hq, 1, D, device=dev, generator=g, dtype=torch.bfloat16)
    k = torch.randn(B, Hk, S, D, device=dev, generator=g, dtype=torch.bfloat16)
    if fp8:
        k = k.to(torch.float8_e4m3fn)
    s = SP.sparse_score_scalar(q, k, 0.088, score_bits=8 if fp8 else 16)
    assert s.shape == (B, Hq, S)
    qc = q.cpu()
    for a, b in ((0, 2000), (768 - 300, 768 + 300), (7 * 768 - 200, 7 * 768 + 200), (S - 3000, S)):
        ks = k[:, :, a:b].cpu()
        ref = R.sparse_score_scalar(qc, ks.to(torch.bfloat16) if fp8 else ks, 0.088)
        d = (s[:, :, a:b].cpu() - ref).abs().max().item()
        print(f"tokens {a}..{b}: max-abs {d:.3e}", flush=True)
        assert d <= SCORE_TOL, (a, b)
    del k, s
    torch.cuda.empty_cache()


@pytest.mark.parametrize("fp8", [False, True])
def test_group_scores_full_lds_buffer(dev, fp8):
    """Rows long enough that, on 256 CUs, each score workgroup's token range
    is the largest its LDS score buffer holds (6144 tokens with bf16 keys,
    8192 with fp8), with a ragged end: group sums at the start, across
    workgroup boundaries and at the end of every row against the oracle on
    those key slices (fp8 keys widened to bf16, which is exact)."""
    B, Hq, Hk, D = 1, 24, 8, 128
    cap = 8192 if fp8 else 6144
    S = 2048 * cap // Hk + 1001
    g = torch.Generator(device=dev).manual_seed(11)
    q = torch.randn(B, Hq, 1, D, device=dev, generator=g, dtype=torch.bfloat16)
    k = torch.randn(B, Hk, S, D, device=dev, generator=g, dtype=torch.bfloat16)
    if fp8:
        k = k.to(torch.float8_e4m3fn)
    s = SP.group_scores(q, k, 0.088)
    assert s.shape == (B, Hk, S)
    qc = q.cpu()
    for a, b in ((0, 3000), (cap - 700, cap + 700), (5 * cap - 300, 5 * cap + 300), (S - 4000, S)):
        ks = k[:, :, a:b].cpu()
        ref = R.group_scores(qc, ks.to(torch.bfloat16) if fp8 else ks, 0.088)
        d = (s[:, :, a:b].cpu() - ref).abs().max().item()
        print(f"tokens {a}..{b}: max-abs {d:.3e}", flush=True)
        assert d <= SCORE_TOL, (a, b)
    del k, s
    torch.cuda.empty_cache()


def _tie_heavy(rows, n, seed):
    g = torch.Generator().manual_seed(seed)
    s = torch.randint(-8, 8, (rows, n), generator=g).float() * 0.25      # many exact ties
    s[0, ::7] = 0.0
    s[0, 1::7] = -0.0
    if rows > 1:
        s[1, 5] = float("nan")
        s[1, 9] = float("-nan")
        s[1, 11] = float("inf")
        s[1, 12] = float("-inf")
    return s


@pytest.mark.parametrize("sorted_out", [True, False])
@pytest.mark.parametrize("rows,n,k", [(3, 1000, 1), (3, 1000, 17), (4, 4096, 256), (2, 1001, 1001),
                                      (5, 333, 100), (28, 2048, 128), (2, 20000, 8192), (3, 70000, 3000),
                                      (1100, 17000, 100)])
def test_topk_bit_exact_with_ties(dev, rows, n, k, sorted_out):
    s = _tie_heavy(rows, n, seed=n + k)
    got = SP.topk_indices(s.to(dev), k, sorted=sorted_out).cpu()
    ref = R.topk_indices(s, k, sorted_by_score=sorted_out)
    assert got.dtype == torch.int32
    assert torch.equal(got.long(), ref)


@pytest.mark.parametrize("rows,n,k", [(3, 40000, 10000), (2, 65536, 16384), (2, 9000, 9000), (130, 20000, 12000),
                                      (2, 131072, 32768), (3, 20000, 8193)])
def test_topk_large_k(dev, rows, n, k):
    """k above 8192: the same set by ascending index (sorted=False), and in the
    total order (sorted=True: blocks of 8192 sorted in LDS, merged by rank),
    both bit-exact against the oracle on tie-heavy rows."""
    s = _tie_heavy(rows, n, seed=n + k)
    got = SP.topk_indices(s.to(dev), k, sorted=False).cpu()
    assert torch.equal(got.long(), R.topk_indices(s, k, sorted_by_score=False))
    got_s = SP.topk_indices(s.to(dev), k, sorted=True).cpu()
    assert torch.equal(got_s.long(), R.topk_indices(s, k, sorted_by_score=True))


@pytest.mark.parametrize("k", [8193, 13107, 32768, 65536, 131071])
def test_topk_large_k_c5_rows(dev, k):
    """k above 8192 on the C5 row shape (64 x 131072): threshold-digit
    candidates, per-row selection and per-slice ordered writes, with a tied
    block at the threshold, a row of rounded (heavily tied) scores and a row
    whose keys share one top digit (the whole-row exact fallback)."""
    g = torch.Generator().manual_seed(k)
    s = torch.randn(64, 131072, generator=g)
    s[3, 1000:1100] = 5.0
    s[5, :] = s[5, :].round()
    s[7, :] = 1.0 + torch.rand(131072, generator=g) * 0.2    # one top digit for every key
    got = SP.topk_indices(s.to(dev), k, sorted=False).cpu().long()
    assert torch.equal(got, R.topk_indices(s, k, sorted_by_score=False))


def test_topk_large_k_row_batches(dev):
    """More rows than one launch group (1024) with k above 8192."""
    s = _tie_heavy(1100, 20000, seed=1)
    got = SP.topk_indices(s.to(dev), 9000, sorted=False).cpu().long()
    assert torch.equal(got, R.topk_indices(s, 9000, sorted_by_score=False))


@pytest.mark.parametrize("sorted_out", [True, False])
@pytest.mark.parametrize("rows,n,k", [(600, 2048, 128), (600, 1000, 1), (300, 4096, 256), (700, 2051, 17),
                                      (260, 64, 64), (1000, 4095, 200)])
def test_topk_many_short_rows(dev, rows, n, k, sorted_out):
    """More rows than CUs with n <= 4096 and k <= 256 (ties, +-0, NaN, +-inf and all-equal rows included)."""
    s = _tie_heavy(rows, n, seed=n + k + rows)
    s[2] = 0.5                                             # an all-equal row
    s[3, : n // 2] = float("inf")                          # more infinities than k
    got = SP.topk_indices(s.to(dev), k, sorted=sorted_out).cpu()
    assert torch.equal(got.long(), R.topk_indices(s, k, sorted_by_score=sorted_out))


@pytest.mark.parametrize("rows,n,k", [(1, 1, 1), (1, 3, 2), (5, 64, 64), (28, 2048, 1024), (3, 4096, 4096),
                                      (4, 4096, 1024), (2, 3000, 2000), (280, 1500, 512), (7, 4095, 1)])
def test_topk_small_rows(dev, rows, n, k):
    """Rows of at most 4096 elements: one 256-thread workgroup per row (sorted output up to k = 1024; larger sorted k takes the
    whole-row sort)."""
    s = _tie_heavy(rows, n, seed=3 * n + k)
    if rows > 3:
        s[2] = -1.5                                          # an all-equal row
        s[3, : n // 2] = float("-inf")
        s[3, n // 2:] = float("inf")
    for so in (True, False):
        got = SP.topk_indices(s.to(dev), k, sorted=so).cpu()
        assert torch.equal(got.long(), R.topk_indices(s, k, sorted_by_score=so)), so
    big = torch.zeros(rows * n + 1)
    big[1:] = s.reshape(-1)
    view = big.to(dev)[1:].reshape(rows, n)                  # rows not 16-byte aligned
    assert torch.equal(SP.topk_indices(view, k, sorted=False).cpu().long(),
                       R.topk_indices(s, k, sorted_by_score=False))


@pytest.mark.parametrize("rows,n,k,shift", [(16, 3000, 150, 0.0), (16, 3000, 750, 0.0), (28, 2048, 128, 0.0),
                                            (4, 1000, 999, 0.0), (28, 2048, 128, 40.0), (8, 4096, 1, 0.0)])
def test_topk_small_rows_continuous(dev, rows, n, k, shift):
    """Rows of distinct continuous scores (and the same shifted far from zero,
    as page bounds sit): the digit pass that reaches a crossing bin of a few
    keys ranks those keys directly; the result must equal the oracle's."""
    g = torch.Generator().manual_seed(rows * n + k)
    s = torch.randn(rows, n, generator=g) + shift
    for so in (True, False):
        got = SP.topk_indices(s.to(dev), k, sorted=so).cpu()
        assert torch.equal(got.long(), R.topk_indices(s, k, sorted_by_score=so)), so


@pytest.mark.parametrize("rows,n,k", [(300, 2048, 128), (28, 2048, 128), (280, 4096, 600), (5, 1000, 17)])
def test_topk_narrow_range_rows(dev, rows, n, k):
    """Scores in a narrow range (every key shares its top bits; the digit
    passes start below them), with exact ties and an all-equal row, for more
    and fewer rows than CUs."""
    g = torch.Generator().manual_seed(rows + n + k)
    s = 3.0 + torch.rand(rows, n, generator=g) * 0.5
    s[0, 10:40] = 3.25                                       # a block of exact ties
    s[1] = 3.125                                             # an all-equal row
    if n > 100:
        s[2, :5] = 3.0 + 2.0 ** -20                          # keys one ulp-scale apart
    for so in (True, False):
        got = SP.topk_indices(s.to(dev), k, sorted=so).cpu()
        assert torch.equal(got.long(), R.topk_indices(s, k, sorted_by_score=so)), so


@pytest.mark.parametrize("rows,n,k", [(257, 4097, 40), (300, 8191, 8191), (3, 8193, 1), (5, 16384, 819),
                                      (256, 16385, 1000), (256, 32768, 3000), (513, 16500, 1024),
                                      (512, 40001, 200), (256, 65536, 9000)])
def test_topk_rows_selected_by_counting(dev, rows, n, k):
    """Rows of 4097 to 65536 elements held in one workgroup's registers (sorted
    up to k = 1024): continuous scores, the same shifted and narrowed, ties
    and lattices, half the row -inf or +inf, NaN of both signs, one value in
    the whole row, one value far above the others, and rows that start off
    16-byte boundaries."""
    g = torch.Generator().manual_seed(n + k)
    s = torch.randn(rows, n, generator=g)
    m = min(rows, 256)
    s[: m // 4 * 4].reshape(4, -1, n)[1] *= 1e-3
    s[: m // 4 * 4].reshape(4, -1, n)[1] += 40.0
    s[: m // 4 * 4].reshape(4, -1, n)[2] = s[: m // 4 * 4].reshape(4, -1, n)[2].mul(8).round() / 8
    for i, f in enumerate([lambda r: r.fill_(-2.5), lambda r: r[: n // 2].fill_(float("-inf")),
                           lambda r: r[n // 3:].fill_(float("inf")), lambda r: r[::7].fill_(float("nan"))]):
        if i + 1 < rows:
            f(s[i + 1])
    if rows > 8:
        s[5, 3] = -float("nan")
        s[6, n - 1] = 3e38
        s[7] = torch.where(torch.arange(n) % 3 == 0, 0.0, -0.0)
        s[8] = torch.arange(n).float()
    want = {so: R.topk_indices(s, k, sorted_by_score=so) for so in ((True, False) if k <= 1024 else (False,))}
    for so, w in want.items():
        assert torch.equal(SP.topk_indices(s.to(dev), k, sorted=so).cpu().long(), w), so
    big = torch.zeros(rows * n + 1, device=dev)
    big[1:] = s.reshape(-1).to(dev)
    assert torch.equal(SP.topk_indices(big[1:].reshape(rows, n), k, sorted=False).cpu().long(), want[False])


def test_topk_many_short_rows_unaligned(dev):
    s = _tie_heavy(400, 1500, seed=11)
    big = torch.zeros(400 * 1500 + 1)
    big[1:] = s.reshape(-1)
    view = big.to(dev)[1:].reshape(400, 1500)              # rows not 16-byte aligned
    for srt in (True, False):
        assert torch.equal(SP.topk_indices(view, 100, sorted=srt).cpu().long(),
                           R.topk_indices(s, 100, sorted_by_score=srt))


def test_topk_unaligned_rows(dev):
    s = _tie_heavy(6, 2051, seed=3)
    big = torch.zeros(6 * 2051 + 1)
    big[1:] = s.reshape(-1)
    view = big.to(dev)[1:].reshape(6, 2051)                # rows not 16-byte aligned
    assert torch.equal(SP.topk_indices(view, 300).cpu().long(), R.topk_indices(s, 300))


@pytest.mark.parametrize("case", ["narrow", "all_equal"])
def test_topk_crowded_digit_rows(dev, case):
    """Every key of a row shares its top 11 bits: the candidate list overflows and
    the whole-row exact selection runs."""
    g = torch.Generator().manual_seed(5)
    if case == "narrow":
        s = 1.0 + torch.rand(3, 20000, generator=g) * 0.2
        s[1, 7777] = 1.1                                      # plus exact ties
        s[1, 7778] = 1.1
    else:
        s = torch.full((3, 20000), 0.5)
    for k in (1, 100, 8192):
        for so in (True, False):
            got = SP.topk_indices(s.to(dev), k, sorted=so).cpu().long()
            assert torch.equal(got, R.topk_indices(s, k, sorted_by_score=so)), (case, k, so)


@pytest.mark.parametrize("k", [256, 1024, 4096])
def test_topk_c5_rows(dev, k):
    """64 rows x 131072 fp32 (BASELINE C5 selection shape)."""
    g = torch.Generator().manual_seed(k)
    s = torch.randn(64, 131072, generator=g)
    s[3, 1000:1100] = 5.0                                   # a tied block straddling the boundary
    s[5, :] = s[5, :].round()                               # heavy ties at the threshold
    for so in (True, False):
        got = SP.topk_indices(s.to(dev), k, sorted=so).cpu().long()
        assert torch.equal(got, R.topk_indices(s, k, sorted_by_score=so)), so


def _gather_case(dev, B, Hq, Hk, S, D, kb, per_head, seed, chunk=0):
    x = W.dense(B, Hq, Hk, D, S, seed=seed)
    g = torch.Generator().manual_seed(seed)
    H = Hq if per_head else Hk
    idx = torch.randint(0, S, (B, H, kb), generator=g)
    idx[..., ::13] = -1                                     # masked entries
    idx[..., 1::29] = S                                     # sentinel (unfilled slot)
    if kb > 4:
        idx[..., 2] = idx[..., 4]                           # a repeated row counts twice
    out = SP.sparse_gather_attn(x["q"].to(dev), x["k"].to(dev), x["v"].to(dev), idx.to(dev), 0.09, chunk=chunk)
    ref = R.sparse_gather_attn(x["q"], x["k"], x["v"], idx, 0.09)
    assert out.shape == (B, Hq, 1, D) and out.dtype == torch.bfloat16
    _check(out, ref, f"gather B{B} Hq{Hq} Hk{Hk} S{S} D{D} kb{kb} per_head{per_head} chunk{chunk}")


@pytest.mark.parametrize("B,Hq,Hk,S,D,kb", [(2, 8, 2, 2000, 128, 100), (1, 24, 8, 5000, 128, 1000),
                                             (1, 7, 1, 300, 64, 31), (2, 28, 4, 4096, 128, 2048)])
@pytest.mark.parametrize("per_head", [1, 0])
def test_gather_matches_oracle(dev, B, Hq, Hk, S, D, kb, per_head):
    _gather_case(dev, B, Hq, Hk, S, D, kb, per_head, seed=kb + per_head)


@pytest.mark.parametrize("chunk", [128, 1024])
def test_gather_split_counts(dev, chunk):
    _gather_case(dev, 1, 8, 2, 40000, 128, 37000, 0, seed=7, chunk=chunk)     # 290 / 37 splits


def test_gather_single_valid_row(dev):
    x = W.dense(1, 4, 1, 128, 64, seed=1)
    idx = torch.full((1, 1, 40), -1)
    idx[0, 0, 17] = 5
    out = SP.sparse_gather_attn(x["q"].to(dev), x["k"].to(dev), x["v"].to(dev), idx.to(dev), 0.1)
    # one row survives the mask: the output is that value row for every head
    assert torch.allclose(out.cpu().float()[0, :, 0], x["v"][0, 0, 5].float().expand(4, -1), atol=1e-2)


@pytest.mark.parametrize("frac", [0.05, 0.25])
def test_sparse_decode_scalar_pipeline(dev, frac):
    x = W.dense(2, 8, 2, 128, 3000, seed=11)
    q, k, v = (x[n].to(dev) for n in ("q", "k", "v"))
    sc = 1 / math.sqrt(128)
    out = SP.sparse_decode_scalar(q, k, None, None, k, v, frac, sc, score_bits=16)
    ref = R.sparse_decode_scalar(x["q"], x["k"], x["k"], x["v"], frac, sc)
    _check(out, ref, f"sparse_decode_scalar frac {frac}")
    # selection is bit-exact given the same fp32 scores
    s = SP.sparse_score_scalar(q, k, sc)
    kb = SP.budget(frac, 3000)
    assert torch.equal(SP.topk_indices(s, kb).cpu().long(), R.topk_indices(s.cpu(), kb))


@pytest.mark.parametrize("kb", [256, 1024, 4096, 32768])
def test_token_topk_c5_full(dev, kb):
    """BASELINE C5 at full size: B8 Hq24 Hkv8 D128 L131072."""
    x = W.c5_topk(seed=0, device=dev)
    q, k, v = x["q"], x["k"], x["v"]
    sc = x["scale"]
    out, idx = SP.token_topk_decode(q, k, v, kb, sc)
    # scores of batch 0 against the oracle
    s = SP.group_scores(q, k, sc)
    ref_s0 = R.group_scores(q[:1].cpu(), k[:1].cpu(), sc)
    assert (s[:1].cpu() - ref_s0).abs().max() <= SCORE_TOL
    # selection bit-exact on the same scores (the pipeline returns the set by ascending index)
    ref_idx = R.topk_indices(s.cpu(), kb, sorted_by_score=False)
    assert torch.equal(idx.cpu().long(), ref_idx)
    # attention over the selected rows: dense oracle on the gathered rows
    B, Hk = k.shape[:2]
    gi = idx.long().unsqueeze(-1).expand(B, Hk, kb, k.shape[-1])
    ks, vs = torch.gather(k, 2, gi).cpu(), torch.gather(v, 2, gi).cpu()
    _check(out, R.decode_attn(q.cpu(), ks, vs, scale=sc), f"C5 kb{kb}")


@pytest.mark.parametrize("B,Hk,G,S,D", [(1, 2, 64, 257, 64), (2, 1, 65, 1000, 128), (1, 1, 1792, 2047, 64),
                                        (1, 3, 100, 3, 128)])
def test_score_many_heads_per_kv_head(dev, B, Hk, G, S, D):
    """64 or more heads per KV head (folded query chunks) take the block kernel:
    the same bits as the streaming kernel gives 16 heads at a time, for token
    counts and head counts that fill no block, into rows of a wider buffer too."""
    from bytes_amd.sparse import _score
    g = torch.Generator().manual_seed(S + G)
    q = torch.randn(B, Hk * G, 1, D, generator=g).to(torch.bfloat16).to(dev)
    k = torch.randn(B, Hk, S, D, generator=g).to(torch.bfloat16).to(dev)
    got = SP.sparse_score_scalar(q, k, 0.3)
    qg = q.reshape(B, Hk, G, 1, D)
    want = torch.empty(B, Hk, G, S, device=dev)
    for h0 in range(0, G, 16):
        n = min(16, G - h0)
        part = qg[:, :, h0:h0 + n].reshape(B, Hk * n, 1, D)
        want[:, :, h0:h0 + n] = SP.sparse_score_scalar(part, k, 0.3).reshape(B, Hk, n, S)
    assert torch.equal(got, want.reshape(B, Hk * G, S))
    wide = torch.full((B, Hk * G, (S + 7) // 4 * 4), 7.0, device=dev)
    _score(q, k, 0.3, group_sum=False, out=wide[:, :, 4:4 + S] if wide.shape[2] >= S + 4 else wide[:, :, :S])
    lo = 4 if wide.shape[2] >= S + 4 else 0
    assert torch.equal(wide[:, :, lo:lo + S], got)
    assert (wide[:, :, :lo] == 7).all() and (wide[:, :, lo + S:] == 7).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,Hk,G,S", [(2, 2, 70, 13200),       # 1040 blocks of 16 heads x 256 tokens: two a workgroup
                                      (1, 1, 520, 8200),       # 1089, a head block of 8
                                      (1, 2, 64, 8192),        # 256: at most one workgroup per CU
                                      (1, 1, 64, 65536)])      # 1024: one block a workgroup
def test_score_many_heads_rule(dev, B, Hk, G, S, D):
    """Both sides of the lines between the block and the streaming kernel: the
    same bits as 16 heads at a time."""
    g = torch.Generator(device=dev).manual_seed(S + G)
    q = torch.randn(B, Hk * G, 1, D, generator=g, device=dev).to(torch.bfloat16)
    k = torch.randn(B, Hk, S, D, generator=g, device=dev).to(torch.bfloat16)
    got = SP.sparse_score_scalar(q, k, 0.3).reshape(B, Hk, G, S)
    qg = q.reshape(B, Hk, G, 1, D)
    for h0 in range(0, G, 16):
        n = min(16, G - h0)
        part = SP.sparse_score_scalar(qg[:, :, h0:h0 + n].reshape(B, Hk * n, 1, D), k, 0.3)
        assert torch.equal(got[:, :, h0:h0 + n], part.reshape(B, Hk, n, S)), h0


@pytest.mark.parametrize("rows,n", [(300, 4097), (300, 8192), (4, 8193), (32, 9000), (33, 9000), (40, 12287),
                                    (40, 12288), (3, 16384), (300, 16384), (260, 32768), (256, 65536)])
def test_topk_rows_past_the_first_counts(dev, rows, n):
    """Rows whose k-th score the interpolated counts do not find: few distinct
    values, neighbouring ones, values far from a line in key space and ordered
    rows, on both sides of the row and length rules, against a stable sort."""
    g = torch.Generator(device=dev).manual_seed(n + rows)
    x = torch.randn(rows, n, generator=g, device=dev)
    at = torch.arange(n, device=dev)
    ulp = torch.randint(0, 3, (rows, n), generator=g, device=dev)
    kinds = {"integers": (2 * x).round(),
             "bf16": x.to(torch.bfloat16).float(),
             "neighbours": (1.0 + ulp * 2.0 ** -23),
             "two values": torch.where(x > 1, 3e30, -1e-30),
             "wide": torch.exp(40 * x).clamp(1e-37, 1e37) * torch.sign(x),
             "ascending": x.sort(1).values,
             "masked": x.masked_fill(at >= n // 20, -math.inf),
             "far from the sample": torch.where(at < n // 2, x, x * 1e-6 + 50)}
    for kind, s in kinds.items():
        want = torch.sort(s, dim=1, descending=True, stable=True).indices
        for k in (1, 65, n // 10, n - 1):
            got = SP.topk_indices(s, k, sorted=False).long()
            assert torch.equal(got, want[:, :k].sort(1).values), (kind, k)
