"""Attention of many query rows per kv head (the prefill kernel) against softmax
attention in 64 bits over the store's own codes: every head dim, key and value
width, query and output dtype, GQA group, remainders of the 128-row and 32-token
tiles, causal and full, key ranges, splits, paged stores, large logits.

The shapes have enough (sequence, kv head) groups that the dispatch's cost rule
sends them to the prefill kernel (smaller calls stay on the decode kernels), which
each test asserts.

Bar for fp32 outputs: 3e-5 relative (2-norm), the decode kernels' own (their
large-logit bar is 1e-4, measured 2.2e-5)."""

import math

import pytest
import torch

import quashkv_amd as quashkv
from quashkv_amd import _native as N
from quashkv_amd.kernels import attention_store
from quashkv_amd.paged import PagedQuashKVEngine

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(autouse=True, scope="module")
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    N.lib()


def exact(e, q, causal, lo=None, hi=None, q_end=0, signs=None, logits=False, kcent=None,
          vcent=None, qjl=None):
    b0 = e._cache[0]
    kc = torch.cat([b.mse_indices for b in e._cache], 2).long()
    vc = torch.cat([b.val_indices for b in e._cache], 2).long()
    kn = torch.cat([b.key_norms for b in e._cache], 2).double()
    vn = torch.cat([b.val_norms for b in e._cache], 2).double()
    qs = torch.cat([b.qjl_signs for b in e._cache], 2).double()
    assert b0.qjl_signs is not None
    kq, vq = e.key_quantizer, e.value_quantizer
    mq = kq.mse_quantizer
    S = (kq.S if signs is None else signs).double()
    B, Hq, Q, d = q.shape
    Hkv, T = kc.shape[1:3]
    G = Hq // Hkv
    table = lambda c, own: own if c is None else torch.tensor(c, device=q.device)  # noqa: E731
    k = table(kcent, mq.codebook.centroids).double()[kc].repeat_interleave(G, 1)
    sg = ((2 * qs - 1) * S).repeat_interleave(G, 1)
    v = (table(vcent, vq.codebook.centroids).double()[vc] * vn[..., None]).repeat_interleave(G, 1)
    qr = q.double() @ mq.Pi.double().T
    s = qr @ k.transpose(2, 3) + (kq.qjl_scale if qjl is None else qjl) * (
        qr.abs() @ sg.transpose(2, 3))
    s = s * kn.repeat_interleave(G, 1)[:, :, None] / math.sqrt(d)
    top = float(s.abs().max())
    t = torch.arange(T, device=q.device)
    lo = torch.zeros(B, device=q.device) if lo is None else lo
    hi = torch.full((B,), T, device=q.device) if hi is None else hi
    end = hi if q_end == 0 else torch.full_like(hi, q_end)
    dead = (t[None, :] < lo[:, None]) | (t[None, :] >= hi[:, None])
    dead = dead[:, None, None, :].expand(B, 1, Q, T)
    if causal:
        pos = end[:, None] - Q + torch.arange(Q, device=q.device)[None]
        dead = dead | (t[None, None, :] > pos[:, :, None])[:, None]
    s = s.masked_fill(dead, -math.inf)
    p = torch.nan_to_num(torch.softmax(s, -1))   # a row with no keys: zeros
    out = (p @ v) @ vq.Pi.double()
    return (out, top) if logits else out


def prefills(e, q, ranges=False, n_splits=None, kcent=None, vcent=None, qjl=None):
    """Whether the prefill kernel takes the call."""
    L, kq, vq = N.lib(), e.key_quantizer, e.value_quantizer
    B, Hq, Q, d = q.shape
    H, T, cap = e._store.H, e.total_tokens, e._store.capacity
    ns = L.qkv_attention_splits(B, Hq, H, Q, d, T)
    kc = N.HostFloats(kcent or kq.mse_quantizer.codebook.centroids_host)
    vc = N.HostFloats(vcent or vq.codebook.centroids_host)
    n = L.qkv_attention_prefills(B, Hq, H, Q, d, T, kq.mse_bits, vq.bits, kc.ptr, vc.ptr,
                                 kq.qjl_scale if qjl is None else qjl, cap, ranges,
                                 L.qkv_attention_workspace_bytes(B, Hq, H, Q, d, n_splits or ns),
                                 n_splits or ns)
    assert n >= 0
    return n > 0


def check(out, ref, bar=3e-5):
    err = float((out.double() - ref).norm() / ref.norm())
    assert err <= bar, err


def filled(B, H, T, d, kb, vb, seed, dtype=torch.bfloat16, cls=quashkv.QuashKVEngine, **kw):
    g = torch.Generator(device=DEV).manual_seed(seed)
    e = cls(head_dim=d, key_bits=kb, value_bits=vb, seed=11, device=DEV, **kw)
    k = torch.randn(B, H, T, d, device=DEV, generator=g)
    k[..., ::32] *= 10.0
    v = torch.randn(B, H, T, d, device=DEV, generator=g)
    e.append(k.to(dtype), v.to(dtype))
    return e, g


@pytest.mark.parametrize("d", [64, 96, 128])
@pytest.mark.parametrize("kb,vb", [(2, 1), (2, 2), (3, 3), (3, 4), (4, 4), (4, 2)])
@pytest.mark.parametrize("B,G,H,T,Q,causal,dtype", [
    (8, 4, 8, 160, 33, True, torch.bfloat16),   # 132 rows: a 4-row remainder
    (20, 7, 5, 95, 41, False, torch.float16),   # (d = 64, 2 key MSE bits: decode_small's)
    (20, 7, 5, 500, 41, False, torch.float16),
    (11, 1, 9, 300, 129, True, torch.float32),
])
def test_prefill_matches_64_bits(d, kb, vb, B, G, H, T, Q, causal, dtype):
    e, g = filled(B, H, T, d, kb, vb, T + Q)
    q = torch.randn(B, H * G, Q, d, device=DEV, generator=g).to(dtype)
    assert prefills(e, q) == (d != 64 or kb > 3 or T != 95)
    ref = exact(e, q, causal)
    check(e.attention(q, causal=causal), ref)
    check(e.attention(q, causal=causal, out_dtype=torch.bfloat16).float(), ref, 4e-3)
    check(e.attention(q, causal=causal, out_dtype=torch.float16).float(), ref, 6e-4)


@pytest.mark.parametrize("T,Q,G", [(48, 48, 1), (64, 12, 4), (31, 31, 2), (1024, 16, 8),
                                   (2048, 300, 1), (1500, 1500, 2)])
def test_prefill_sizes(T, Q, G):
    """The smallest calls, whole and odd numbers of tiles, Q = T."""
    e, g = filled(8, 8, T, 128, 3, 3, T)
    q = torch.randn(8, 8 * G, Q, 128, device=DEV, generator=g)
    assert prefills(e, q)
    check(e.attention(q, causal=True), exact(e, q, True))


@pytest.mark.parametrize("d,splits", [(128, 2), (128, 7), (96, 3), (64, 64)])
def test_prefill_splits(d, splits):
    e, g = filled(8, 8, 700, d, 3, 3, splits)
    q = torch.randn(8, 32, 60, d, device=DEV, generator=g)
    assert prefills(e, q, n_splits=splits)
    kq, vq = e.key_quantizer, e.value_quantizer
    for causal in (False, True):
        out = attention_store(q, e._store, 700, kq.mse_quantizer.Pi,
                              kq.mse_quantizer.codebook.centroids_host,
                              vq.codebook.centroids_host, kq.S, kq.qjl_scale, causal=causal,
                              n_splits=splits)
        check(out, exact(e, q, causal))


def test_prefill_ranges_and_positions():
    e, g = filled(4, 16, 333, 128, 3, 3, 5)
    q = torch.randn(4, 64, 40, 128, device=DEV, generator=g)
    lo = torch.tensor([0, 31, 32, 200], device=DEV, dtype=torch.int32)
    hi = torch.tensor([333, 300, 97, 200], device=DEV, dtype=torch.int32)   # the last: no keys
    assert prefills(e, q, ranges=True)
    for causal, q_end in ((False, 0), (True, 0), (True, 333), (True, 60)):
        out = e.attention(q, causal=causal, kv_start=lo, kv_end=hi, q_end=q_end)
        check(out, exact(e, q, causal, lo, hi, q_end))
        assert float(out[3].abs().max()) == 0.0


@pytest.mark.parametrize("d,kb,page", [(128, 3, 64), (96, 4, 256), (64, 3, 2048)])
def test_prefill_paged_equals_contiguous(d, kb, page):
    args = (8, 8, 515, d, kb, 3, 7)
    a, g = filled(*args)
    b, _ = filled(*args, cls=PagedQuashKVEngine, page_tokens=page)
    q = torch.randn(8, 32, 60, d, device=DEV, generator=g)
    assert prefills(a, q)
    assert torch.equal(a.attention(q, causal=True), b.attention(q, causal=True))


@pytest.mark.parametrize("kb,vb", [(2, 2), (3, 3), (4, 4)])
def test_prefill_large_logits_and_norms(kb, vb):
    """Key and value norms over eight decades, tiny and huge queries."""
    g = torch.Generator(device=DEV).manual_seed(9)
    e = quashkv.QuashKVEngine(head_dim=128, key_bits=kb, value_bits=vb, seed=3, device=DEV)
    T = 777
    k = torch.randn(8, 8, T, 128, device=DEV, generator=g)
    v = torch.randn(8, 8, T, 128, device=DEV, generator=g)
    k *= torch.exp(1.5 * torch.randn(8, 8, T, 1, device=DEV, generator=g))
    v *= torch.logspace(-4, 4, T, device=DEV)[torch.randperm(T, device=DEV, generator=g)][:, None]
    e.append(k, v)
    q = torch.randn(8, 32, 50, 128, device=DEV, generator=g)
    q[:, :, 1] *= 1e-6
    q[:, :, 2, 1:] = 0.0
    q[:, :, 3] = 0.0
    assert prefills(e, q)
    ref, top = exact(e, q, True, logits=True)
    out = e.attention(q, causal=True)
    err = (out.double() - ref).norm(dim=-1) / ref.norm(dim=-1).clamp(min=1e-30)
    # a score good to 4e-6 of itself moves a row by at most that of the largest logit
    # (key levels are good to 5e-7); the decode kernels' error here is 3e-2 on average
    assert float(err.max()) <= 4e-6 * top + 2e-5 and float(err.mean()) <= 2e-5


def test_prefill_other_signs():
    """S that f16 does not hold exactly (and of size 0): the third QJL product."""
    e, g = filled(8, 8, 200, 128, 3, 3, 5)
    q = torch.randn(8, 32, 30, 128, device=DEV, generator=g)
    kq, vq = e.key_quantizer, e.value_quantizer
    signs = kq.S * (0.5 + torch.rand(128, device=DEV, generator=g))
    signs[5] = 0.0
    assert prefills(e, q)
    out = attention_store(q, e._store, 200, kq.mse_quantizer.Pi,
                          kq.mse_quantizer.codebook.centroids_host, vq.codebook.centroids_host,
                          signs, kq.qjl_scale, causal=True)
    check(out, exact(e, q, True, signs=signs))


@pytest.mark.parametrize("d,T", [(64, 200), (128, 333)])
def test_prefill_extremes(d, T):
    """Value norms of zero (rows that see no other among them), queries below 1e-38,
    and slots outside the key range whose norms are not finite."""
    e, g = filled(8, 8, T, d, 3, 3, 13, dtype=torch.float32)
    st = e._store
    st.vnorm.view(8, 8, -1)[:, :, :40] = 0.0
    q = torch.randn(8, 32, 80, d, device=DEV, generator=g)
    q[:, :, 45] *= 1e-39
    lo = torch.full((8,), 5, device=DEV, dtype=torch.int32)
    hi = torch.full((8,), T - 13, device=DEV, dtype=torch.int32)
    assert prefills(e, q, ranges=True)
    refs = [exact(e, q, True, lo, hi, end) for end in (0, 80)]
    assert float(refs[1][:, :, :40].abs().max()) == 0.0
    st.vnorm.view(8, 8, -1)[:, :, :5] = math.inf
    st.vnorm.view(8, 8, -1)[:, :, T - 13:T] = math.nan
    st.knorm.view(8, 8, -1)[:, :, T - 13:T] = math.nan
    for end, ref in zip((0, 80), refs):
        out = e.attention(q, causal=True, kv_start=lo, kv_end=hi, q_end=end)
        check(out, ref)
        check(out[:, :, 45], ref[:, :, 45])   # uniform weights
        assert not out[:, :, (ref == 0).all(-1).all(0).all(0)].any()


@pytest.mark.parametrize("d,splits", [(128, 1), (128, 4), (96, 3), (64, 4)])
def test_prefill_split_large_value_norms(d, splits):
    """Value norms to 1e12 (and 1e-12) over several splits: the merge's floor on the
    weights' sum is no part of the result."""
    e, g = filled(8, 8, 700, d, 3, 3, 21, dtype=torch.float32)
    q = torch.randn(8, 32, 60, d, device=DEV, generator=g)
    kq, vq = e.key_quantizer, e.value_quantizer
    e._store.vnorm *= torch.tensor([1e12, 1e-12] * 4, device=DEV)[:, None]
    assert prefills(e, q, n_splits=splits)
    ref = exact(e, q, True)
    out = attention_store(q, e._store, 700, kq.mse_quantizer.Pi,
                          kq.mse_quantizer.codebook.centroids_host,
                          vq.codebook.centroids_host, kq.S, kq.qjl_scale, causal=True,
                          n_splits=splits)
    for h in range(8):   # one norm each
        check(out[:, 4 * h:4 * h + 4], ref[:, 4 * h:4 * h + 4])


def _call(e, q, causal, form):
    """qkv_decode_attention by its workspace, no-allocation or three-call form."""
    st, kq, vq = e._store, e.key_quantizer, e.value_quantizer
    mq = kq.mse_quantizer
    B, Hq, Q, d = q.shape
    T = e.total_tokens
    L, s = N.lib(), N.stream(q.device)
    kc = N.HostFloats(mq.codebook.centroids_host)
    vc = N.HostFloats(vq.codebook.centroids_host)
    out = torch.full((B, Hq, Q, d), math.nan, device=DEV)
    ns = L.qkv_attention_splits(B, Hq, st.H, Q, d, T)
    ws = torch.empty(L.qkv_attention_workspace_bytes(B, Hq, st.H, Q, d, ns), dtype=torch.uint8,
                     device=DEV)
    qa = (q.data_ptr(), N.dtype_code(q.dtype))
    kv = (st.kst.data_ptr(), st.knorm.data_ptr(), st.vst.data_ptr(), st.vnorm.data_ptr(),
          st.capacity, T)
    dims = (B, Hq, st.H, Q, d, st.mbits, st.vbits)
    tail = (1.0 / math.sqrt(d), int(causal), out.data_ptr(), N.QKV_F32)
    w = (ws.data_ptr(), ws.numel(), ns, s)
    if form == "phases":
        N.check(L.qkv_attention_prepare(*qa, *dims, mq.Pi.data_ptr(), kc.ptr, vc.ptr,
                                        kq.S.data_ptr(), kq.qjl_scale, *w))
        N.check(L.qkv_attention_run(*kv, *dims, mq.Pi.data_ptr(), kc.ptr, vc.ptr, *tail, *w))
    else:
        args = (*qa, *kv, *dims, mq.Pi.data_ptr(), kc.ptr, vc.ptr, kq.S.data_ptr(), kq.qjl_scale,
                *tail)
        if form == "noalloc":
            N.check(L.qkv_decode_attention_noalloc(*args, ns, s))
        else:
            N.check(L.qkv_decode_attention(*args, *w))
    return out


@pytest.mark.parametrize("B,H,G,Q,d,T", [(8, 8, 4, 64, 64, 8192), (1, 8, 1, 128, 128, 8200),
                                         (2, 4, 2, 300, 96, 4096)])
def test_many_rows_by_every_form(B, H, G, Q, d, T):
    """The split count of the library in the single call (the prefill kernel's own
    splits, also where the no-allocation array holds fewer than it asks for) and in
    the three-call form, whose kernels it is for."""
    e, g = filled(B, H, T, d, 3, 3, 17)
    q = torch.randn(B, H * G, Q, d, device=DEV, generator=g)
    assert prefills(e, q)
    ref = exact(e, q, True)
    a = _call(e, q, True, "workspace")
    check(a, ref)
    assert torch.equal(a, e.attention(q, causal=True))
    check(_call(e, q, True, "phases"), ref)
    if B * H * G * Q * (12 * d + 1552) < N.NOALLOC_SCRATCH_BYTES:
        check(_call(e, q, True, "noalloc"), ref)


@pytest.mark.parametrize("kb,vb,kc,vc,qjl", [
    (3, 2, (0.0011, 0.1), None, 95.0),            # a QJL weight past f16 at the levels' scale
    (3, 2, None, (1.0, 2e5), None),               # value levels of such a ratio
    (3, 3, (0.15, 0.05), (3e5, 0.9, 0.3, 1.0), None),   # levels in no order
    (4, 4, (0.05, 0.2, 0.1, 0.15), (.4, .1, .3, .2, .8, .5, .7, .6), None),
])
def test_prefill_other_codebooks(kb, vb, kc, vc, qjl):
    """Symmetric codebooks beyond the library's own, of the magnitudes given."""
    e, g = filled(8, 8, 333, 128, kb, vb, 3)
    e._store.knorm *= 0.01
    q = torch.randn(8, 32, 40, 128, device=DEV, generator=g)
    kq, vq = e.key_quantizer, e.value_quantizer
    both = lambda m, own: [-x for x in m[::-1]] + list(m) if m else own   # noqa: E731
    kc = both(kc, kq.mse_quantizer.codebook.centroids_host)
    vc = both(vc, vq.codebook.centroids_host)
    qjl = kq.qjl_scale if qjl is None else qjl
    assert prefills(e, q, kcent=kc, vcent=vc, qjl=qjl) == (qjl < 90.0)
    out = attention_store(q, e._store, 333, kq.mse_quantizer.Pi, kc, vc, kq.S, qjl, causal=True)
    check(out, exact(e, q, True, kcent=kc, vcent=vc, qjl=qjl))


@pytest.mark.parametrize("d,splits", [(64, 1), (128, 1), (128, 3)])
def test_prefill_non_finite_norms_behind_the_mask(d, splits):
    """Slots that are not finite: rows before them do not notice, rows that see them
    are not finite either."""
    T, Q = 700, 60
    e, g = filled(8, 8, T, d, 3, 3, 23)
    q = torch.randn(8, 32, Q, d, device=DEV, generator=g)
    kq, vq = e.key_quantizer, e.value_quantizer
    assert prefills(e, q, n_splits=splits)
    ref = exact(e, q, True)
    for slot, bad in ((T - 20, math.inf), (T - 33, math.nan)):
        norm = e._store.vnorm if bad == math.inf else e._store.knorm
        norm[:, :, slot] = bad
        if bad != math.inf:
            e._store.vnorm[:, :, slot] = bad
        out = attention_store(q, e._store, T, kq.mse_quantizer.Pi,
                              kq.mse_quantizer.codebook.centroids_host,
                              vq.codebook.centroids_host, kq.S, kq.qjl_scale, causal=True,
                              n_splits=splits)
        i = slot - (T - Q)   # the first query that sees it
        check(out[:, :, :i], ref[:, :, :i])
        assert not torch.isfinite(out[:, :, i:]).all(-1).any()


@pytest.mark.parametrize("d,kb,vb,scale,bar", [
    # logits up to ~130: the QJL weight in one f16 (2.5e-5 off) gave 1.5e-5
    (128, 3, 3, 8.0, 3e-6), (96, 3, 3, 8.0, 3e-6),
    # logits near 0: two value magnitudes in one f16 each gave 4.5e-7 - 6e-7; the
    # rounding of ~150 fp32 additions per output, 2^-24 sqrt(150 / 12), is 2e-7
    (64, 2, 2, 0.05, 3.5e-7), (96, 3, 2, 0.05, 3.5e-7), (128, 3, 2, 0.05, 3.5e-7),
])
def test_prefill_precision(d, kb, vb, scale, bar):
    e, g = filled(4, 8, 777, d, kb, vb, 29, dtype=torch.float32)
    q = scale * torch.randn(4, 32, 64, d, device=DEV, generator=g)
    assert prefills(e, q)
    check(e.attention(q, causal=True), exact(e, q, True), bar)


@pytest.mark.parametrize("d,dtype", [(128, torch.float32), (128, torch.bfloat16),
                                     (96, torch.float16), (64, torch.float32)])
def test_prefill_unaligned_queries(d, dtype):
    e, g = filled(8, 8, 200, d, 3, 3, 37)
    n = 8 * 32 * 80 * d
    q = torch.randn(n + 1, device=DEV, generator=g).to(dtype)[1:].view(8, 32, 80, d)
    assert prefills(e, q) and q.is_contiguous() and q.data_ptr() % 16
    out = e.attention(q, causal=True)
    assert torch.equal(out, e.attention(q.clone(), causal=True))
    check(out, exact(e, q, True))
