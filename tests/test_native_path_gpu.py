"""The operators' native call path against their Python wrappers: the same bits
for every layout and dtype either takes, and the same refusals."""
import pytest
import torch

from bytes_amd import _lib
from bytes_amd import attention_kernels as AK
from bytes_amd import kivi as KV
from bytes_amd import pq as PQ
from bytes_amd import quest as QU
from bytes_amd import sparse as SP
from bytes_amd import sparse_attention as SA
from bytes_amd import workloads as W

pytestmark = pytest.mark.gpu
F8 = torch.float8_e4m3fn


class _Count:
    """Stands for the native module: counts the calls it took."""

    def __init__(self, inner):
        self.inner, self.taken, self.refused = inner, 0, 0

    def __getattr__(self, name):
        f = getattr(self.inner, name)

        def g(*a):
            r = f(*a)
            if r is None:
                self.refused += 1
            else:
                self.taken += 1
            return r
        return g


def _both(monkeypatch, fn, *args, taken=True, **kw):
    """fn through the Python wrapper alone, then through the native path."""
    native = _lib.native()
    monkeypatch.setattr(_lib, "_native", _lib._NoNative())
    want = fn(*args, **kw)
    count = _Count(native)
    monkeypatch.setattr(_lib, "_native", count)
    got = fn(*args, **kw)
    monkeypatch.setattr(_lib, "_native", native)
    assert (count.taken > 0) == taken, (fn.__name__, count.taken, count.refused)
    for a, b in zip(got if isinstance(got, tuple) else (got,), want if isinstance(want, tuple) else (want,)):
        assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
        assert torch.equal(a.view(torch.uint8) if a.dtype == F8 else a, b.view(torch.uint8) if b.dtype == F8 else b)
    return got


def _qkv(dev, B, Hq, Hk, S, D, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device=dev, dtype=torch.bfloat16)      # noqa: E731
    return r(B, Hq, 1, D), r(B, Hk, S, D), r(B, Hk, S, D)


@pytest.mark.parametrize("B,Hq,Hk,S,D", [(1, 14, 2, 777, 64), (3, 7, 7, 130, 128), (2, 40, 2, 65, 128)])
def test_dense_layouts(dev, monkeypatch, B, Hq, Hk, S, D):
    q, k, v = _qkv(dev, B, Hq, Hk, S, D)
    _both(monkeypatch, AK.decode_attn_bf16, q, k, v)
    _both(monkeypatch, AK.decode_attn_bf16, q, k, v, 0.1, chunk=64)
    _both(monkeypatch, AK.decode_attn_fp8, q, k.to(F8), v.to(F8), 0.1)
    bshd = k.transpose(1, 2).contiguous().transpose(1, 2)                       # [B, S, Hk, D] storage
    _both(monkeypatch, AK.decode_attn_bf16, q, bshd, v, 1)
    q8 = torch.randn(B, Hq, 8, D, device=dev).to(torch.bfloat16)
    _both(monkeypatch, AK.decode_attn_bf16, q8[:, :, 3:4], k, v)                # a strided query row
    _both(monkeypatch, AK.decode_attn_bf16, q, k[:, :, 1:], v[:, :, 1:])
    # layouts that need a copy stay in Python
    wide = torch.randn(B, Hk, S, D + 1, device=dev).to(torch.bfloat16)[..., 1:]
    _both(monkeypatch, AK.decode_attn_bf16, q, wide, v, taken=False)
    _both(monkeypatch, AK.decode_attn_bf16, q, k.transpose(2, 3).contiguous().transpose(2, 3), v, taken=False)
    qg = q.clone().requires_grad_()
    out = _both(monkeypatch, AK.decode_attn_bf16, qg, k, v)
    assert not out.requires_grad
    for bad in ((q, k.half(), v), (q, k, v[:, :, 1:]), (q[..., :32], k[..., :32], v[..., :32]), (q.cpu(), k, v),
                (q, k.cpu(), v), (q, k[:, :, :0], v[:, :, :0]), ("q", k, v)):
        with pytest.raises(ValueError):
            AK.decode_attn_bf16(*bad)


def test_tensor_subclass_and_vmap_are_not_taken(dev, monkeypatch):
    class Sub(torch.Tensor):
        pass
    q, k, v = _qkv(dev, 1, 4, 2, 100, 64)
    assert _lib.native().dense(q.as_subclass(Sub), k, v, 1.0, 0, False) is None
    seen = []
    torch.vmap(lambda x: (seen.append(_lib.native().dense(x, k, v, 1.0, 0, False)), x)[1])(q.unsqueeze(0))
    assert seen == [None]


@pytest.mark.parametrize("bits,D,L,R", [(2, 128, 1024 + 128, 128), (4, 128, 992 + 7, 7), (2, 64, 320, 0)])
def test_kivi(dev, monkeypatch, bits, D, L, R):
    raw = W.kivi_raw(2, 8, 2, D, L, R, seed=1, device=dev)
    x = W.kivi_pack_inputs(raw, lambda t, g, b: _both(monkeypatch, KV.quantize_and_pack_along_last_dim, t, g, b), bits)
    a = [x[n] for n in ("Q", "Kq", "K_scale", "K_mn", "K_residual", "Vq", "V_scale", "V_mn", "V_residual")]
    _both(monkeypatch, KV.kivi_decode_attn, *a, bits)
    _both(monkeypatch, KV.kivi_decode_attn, *a, bits, 32, scale=0.2, chunk=256)
    f32 = [t.float() if t.dtype == torch.float16 else t for t in a]
    _both(monkeypatch, KV.kivi_decode_attn, *f32, bits, taken=False)
    with pytest.raises(ValueError):
        KV.kivi_decode_attn(*a, bits, 64)
    t = torch.randn(3, 5, 192, device=dev)
    for dt in (torch.float32, torch.bfloat16):
        _both(monkeypatch, KV.quantize_and_pack_along_last_dim, t.to(dt), 96, bits)
    _both(monkeypatch, KV.quantize_and_pack_along_last_dim, t.transpose(0, 1), 32, bits, taken=False)


def test_pq(dev, monkeypatch):
    B, Hq, Hk, S, D, M, K = 2, 8, 2, 300, 128, 16, 64
    g = torch.Generator(device=dev).manual_seed(2)
    q, _, v = _qkv(dev, B, Hq, Hk, S, D)
    for lead in ((Hk,), ()):
        kcb, vcb = (torch.randn(*lead, M, K, 8, generator=g, device=dev).half() for _ in range(2))
        ki, vi = (torch.randint(0, K, (B, Hk, S, M), generator=g, device=dev).to(torch.uint8) for _ in range(2))
        _both(monkeypatch, PQ.decode_attn_pq_kv_fused, q, kcb, ki, vi, vcb, 0.1)
        _both(monkeypatch, PQ.decode_attn_pq_kv_fused, q, kcb.float(), ki, vi, vcb.float(), 0.1, taken=False)
        _both(monkeypatch, PQ.decode_attn_pq_kv_fused, q, kcb, ki.long(), vi, vcb, 0.1, taken=False)
    lut = torch.randn(B, Hq, M, K, generator=g, device=dev)
    for C, dt in ((1, torch.bfloat16), (3, torch.float32), (16, torch.float16)):
        ko = torch.randn(B, Hk, S, C, generator=g, device=dev).to(dt)
        qo = torch.randn(B, Hq, C, generator=g, device=dev).to(torch.bfloat16)
        for vv in (v, v.to(F8)):
            _both(monkeypatch, PQ.decode_attn_pq_lut_asym, lut, ki, ko, qo, vv)
    bs, nb = 16, 40
    kp = torch.randint(0, K, (nb, Hk, bs, M), generator=g, device=dev).to(torch.uint8)
    kop = torch.randn(nb, Hk, bs, 2, generator=g, device=dev).to(torch.bfloat16)
    vp = torch.randn(nb, Hk, bs, D, generator=g, device=dev).to(torch.bfloat16)
    bt = torch.randperm(nb, generator=g, device=dev).to(torch.int32).reshape(B, nb // 2)
    cl = torch.tensor([300, 17], dtype=torch.int32, device=dev)
    qo = qo[..., :2].contiguous()
    _both(monkeypatch, PQ.paged_attn_pq_lut_asym, lut, kp, kop, qo, vp, bt, cl, bs)
    _both(monkeypatch, PQ.paged_attn_pq_lut_asym, lut, kp, kop, qo, vp, bt.long(), cl, bs, taken=False)
    with pytest.raises(ValueError):
        PQ.paged_attn_pq_lut_asym(lut, kp, kop, qo, vp, bt, cl, 32)
    with pytest.raises(ValueError):                                             # as many blocks as sequences
        PQ.paged_attn_pq_lut_asym(lut, kp[:B], kop[:B], qo, vp[:B], None, None, bs)
    for tables in ((bt, None), (None, cl)):
        with pytest.raises(ValueError):
            PQ.paged_attn_pq_lut_asym(lut, kp, kop, qo, vp, *tables, bs)
    cb = torch.randn(3, M, K, 8, generator=g, device=dev)
    x = torch.randn(3, 2, 77, D, generator=g, device=dev)
    for dt in (torch.float32, torch.bfloat16, torch.float16):
        _both(monkeypatch, PQ.pq_encode, x.to(dt), cb)
        _both(monkeypatch, PQ.pq_encode, x.to(dt), cb.half())
        _both(monkeypatch, PQ.pq_encode, x.to(dt)[0], cb[1])
    _both(monkeypatch, PQ.pq_encode, x, cb.double(), taken=False)


@pytest.mark.parametrize("B,Hq,Hk,S,D", [(2, 8, 2, 1000, 128), (1, 3, 3, 515, 64)])
def test_sparse_and_quest(dev, monkeypatch, B, Hq, Hk, S, D):
    q, k, v = _qkv(dev, B, Hq, Hk, S, D)
    k8 = k.to(F8)
    for frac in (0.0001, 0.0505, 1.0):
        _both(monkeypatch, SP.sparse_decode_scalar, q, k, None, None, k, v, frac, 0.1, score_bits=16)
        _both(monkeypatch, SP.sparse_decode_scalar, q, k8, None, None, k, v, frac, 0.1, score_bits=8)
    for bits in (4, 2):
        p, sc, zr = SP.quantize_and_pack_score_keys(k, bits, 32)
        _both(monkeypatch, SP.sparse_decode_scalar, q, p, sc, zr, k, v, 0.1, 0.1, score_bits=bits)
        _both(monkeypatch, SP.token_topk_decode, q, k, v, 33, 0.1, k_score=p, score_scale=sc, score_zero=zr,
              score_bits=bits, taken=True)
    _both(monkeypatch, SP.token_topk_decode, q, k, v, 100, 0.1)
    _both(monkeypatch, SP.token_topk_decode, q, k, v, 1, 0.1, k_score=k8)
    with pytest.raises(RuntimeError):
        SP.token_topk_decode(q, k, v, S + 1, 0.1)
    with pytest.raises(ValueError):
        SP.sparse_decode_scalar(q, k8, None, None, k, v, 0.1, 0.1, score_bits=16)
    s = torch.randn(5, 700, device=dev)
    for so in (True, False, 1, 0):
        _both(monkeypatch, SP.topk_indices, s, 50, sorted=so)
    _both(monkeypatch, SP.topk_indices, s.t(), 3, taken=False)
    idx = SP.topk_indices(torch.randn(B, Hq, S, device=dev), 64)
    _both(monkeypatch, SP.sparse_gather_attn, q, k, v, idx, 0.1)
    _both(monkeypatch, SP.sparse_gather_attn, q, k8, v.to(F8), idx, 0.1, limit=S // 2)
    _both(monkeypatch, SP.sparse_gather_attn, q, k, v, idx[..., ::2], 0.1, taken=False)
    _both(monkeypatch, SP.sparse_gather_attn, q, k, v, idx.long(), 0.1, taken=False)
    _both(monkeypatch, SP.sparse_gather_attn, q, k, v, idx % (S // 16), 0.1, page=16)
    with pytest.raises(ValueError):
        SP.sparse_gather_attn(q, k, v, idx, 0.1, limit=S + 1)
    meta = QU.quest_page_minmax(k, 16)
    for kw in ({}, {"pos": S - 9}, {"local_w": 40}, {"pos": 20, "local_w": 7}):
        _both(monkeypatch, QU.quest_decode, q, k, v, 100, 0.1, meta=meta, **kw)
    _both(monkeypatch, QU.quest_decode, q, k, v, 100, 0.1)
    with pytest.raises(ValueError):
        QU.quest_decode(q, k, v, 100, 0.1, meta=meta, pos=S)
    qb = torch.randn(B, Hq, 5, D, device=dev).to(torch.bfloat16)
    pos = torch.tensor([0, 3, S // 3, S // 2, S - 1])
    for p in (pos, pos.to(dev), pos.tolist()):
        _both(monkeypatch, SA.select_topk, "exact", qb, k, p, S, 90, 256, 0.1)


def test_first_call_and_other_streams(dev, monkeypatch):
    """Without a workspace yet, the wrapper allocates it; later calls, on any
    stream, run on the current one."""
    q, k, v = _qkv(dev, 1, 4, 2, 4000, 64)
    want = AK.decode_attn_bf16(q, k, v)
    key = (dev.index or 0, "splitk")
    _lib._retired.append(_lib._ws.pop(key))
    assert _lib.native().dense(q, k, v, 1.0, 0, False) is None
    assert torch.equal(AK.decode_attn_bf16(q, k, v), want)
    torch.cuda.synchronize()
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        k2 = k * 2
        got = _lib.native().dense(q, k2, v, 0.5, 0, False)
    st.synchronize()
    assert torch.equal(got, want)


def test_gather_refuses_keys_of_other_ranks(dev):
    """With no limit given, keys that are not [B, Hk, S, D] are refused as
    they are with one."""
    q, k, v = _qkv(dev, 1, 4, 2, 100, 64)
    idx = torch.zeros(1, 4, 3, dtype=torch.int32, device=dev)
    for bad in (k[0, 0], k[0, 0, 0]):
        with pytest.raises(ValueError, match="expected 4 dims"):
            SP.sparse_gather_attn(q, bad, bad, idx, 0.1)


def test_dispatch_mode_without_storage_is_refused(dev):
    """Under a mode whose allocations have no memory to point to, a call raises
    before anything is launched, and the next call outside it works."""
    from torch.utils._python_dispatch import TorchDispatchMode

    class NoMemory(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            if func is torch.ops.aten.empty.memory_format:
                return torch.sparse_coo_tensor(size=args[0], dtype=kwargs.get("dtype"), device=dev)
            return func(*args, **(kwargs or {}))

    q, k, v = _qkv(dev, 1, 4, 2, 1000, 64)
    x = torch.randn(3, 64, device=dev)
    s = torch.randn(3, 640, device=dev)
    want = AK.decode_attn_bf16(q, k, v), SP.topk_indices(s, 5)
    n = _lib.native()
    with NoMemory():
        assert n.dense(q, k, v, 1.0, 0, False) is None
        assert n.kivi_pack(x, 32, 2) is None
        assert n.topk(s, 5, True) is None
        assert n.token_topk(q, k, v, 5, 0.1, k, None, None, None) is None
        with pytest.raises(RuntimeError):
            AK.decode_attn_bf16(q, k, v)
    assert torch.equal(AK.decode_attn_bf16(q, k, v), want[0]) and torch.equal(SP.topk_indices(s, 5), want[1])


def test_token_topk_counts_and_selects_in_one_buffer(dev):
    """The selection reads the histogram from the buffer that the score kernel
    counted into, also where another thread replaces the table's buffer in
    between: the table is asked for it once."""
    q, k, v = _qkv(dev, 1, 8, 2, 40000, 64)
    want = SP.token_topk_decode(q, k, v, 50, 0.1)
    asked = []

    class Key(tuple):
        __hash__ = tuple.__hash__

        def __eq__(self, other):
            asked.append(self[1])
            return tuple.__eq__(self, other)

    native = _lib.native()
    native.set_workspaces({Key(n): b for n, b in _lib._ws.items()})
    try:
        got = native.token_topk(q, k, v, 50, 0.1, k, None, None, None)
    finally:
        native.set_workspaces(_lib._ws)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    assert asked.count("topk") == 1


@pytest.mark.parametrize("shift", ["keys", "scale"])
def test_composites_refuse_before_they_allocate(dev, shift):
    """Score keys whose layout needs a copy are left to the wrapper before the
    score tensor is made."""
    q, k, v = _qkv(dev, 2, 8, 2, 1000, 64)
    p, sc, zr = SP.quantize_and_pack_score_keys(k, 4, 32)
    want = SP.sparse_decode_scalar(q, p, sc, zr, k, v, 0.1, 0.1, score_bits=4)
    want_t = SP.token_topk_decode(q, k, v, 33, 0.1, k_score=p, score_scale=sc, score_zero=zr, score_bits=4)
    if shift == "keys":                        # rows off their 16-byte boundary
        wide = torch.zeros(*p.shape[:3], p.shape[3] + 1, dtype=p.dtype, device=dev)
        wide[..., 1:] = p
        p = wide[..., 1:]
    else:                                      # scale and minimum with strides of their own
        wide = torch.zeros(*sc.shape[:2], 2 * sc.shape[2], sc.shape[3], dtype=sc.dtype, device=dev)
        wide[:, :, ::2] = sc
        sc = wide[:, :, ::2]
    native = _lib.native()
    made = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]        # noqa: E731
    at = made()
    assert native.sparse_decode(q, p, sc, zr, k, v, 0.1, 0.1, 4) is None
    assert native.token_topk(q, k, v, 33, 0.1, p, sc, zr, 4) is None
    assert made() == at
    assert torch.equal(SP.sparse_decode_scalar(q, p, sc, zr, k, v, 0.1, 0.1, score_bits=4), want)
    got = SP.token_topk_decode(q, k, v, 33, 0.1, k_score=p, score_scale=sc, score_zero=zr, score_bits=4)
    assert torch.equal(got[0], want_t[0]) and torch.equal(got[1], want_t[1])
