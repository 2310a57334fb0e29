"""Timed cases of the framework: the calls a serving or search program makes.

``listed()`` names the cases, ``draw`` gives more of the same ranges,
``prepare`` builds what a program holds before the call (seeded inputs, the
engine with its compressed cache, the index), ``run`` is one pass through the
public entry points, ``exact`` the same result in 64 bits by plain torch from
the same stored codes, and ``work`` the bytes and operations of one pass that
no implementation avoids.

Kinds of case:

* ``attend``  QuashKVEngine / PagedQuashKVEngine.attention over a cached
  context: decode (one query token, or a few speculative ones) and causal
  prefill (a prompt, or a chunk of one, over the cache that holds it);
* ``layers``  LayerBatch, a whole model's decode attention in one call;
* ``append``  QuashKVEngine.append into an empty cache: a prompt, a chunk;
* ``append_layers``  LayerBatch.append of a decode step's tokens;
* ``codec``   the quantizer operators: compress of rows, decompress of codes;
* ``rebuild`` QuashKVCache[layer]: the reconstructed K and V of a layer;
* ``search``  QuashIndex.search.
"""

import math

import torch

import quashkv_amd as quashkv
from quashkv_amd.integrations.hf_cache import QuashKVCache
from quashkv_amd.kernels import LayerBatch
from quashkv_amd.nn_search import QuashIndex
from quashkv_amd.paged import PagedQuashKVEngine

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
SEED = 42   # the quantizers' default seed


def attend(name, B, Hq, Hkv, d, T, Q=1, kb=3, vb=3, dtype="bf16", out="fp32", store="flat",
           causal=False):
    return dict(name=name, kind="attend", B=B, Hq=Hq, Hkv=Hkv, d=d, T=T, Q=Q, kb=kb, vb=vb,
                dtype=dtype, out=out, store=store, causal=causal)


def listed():
    return [
        # the README's quickstart: one fp32 query over a 512-token context
        attend("decode_quickstart", 1, 8, 8, 128, 512, dtype="fp32"),
        # a Llama-3-8B layer serving 32 sequences of 8k tokens
        attend("decode_serving", 32, 32, 8, 128, 8192),
        # Qwen2.5-0.5B: the 24 layers of a decode step, 16 sequences
        dict(name="decode_layers", kind="layers", L=24, B=16, Hq=14, Hkv=2, d=64, T=2048, kb=3,
             vb=3, dtype="bf16"),
        # one 128k-token document, mixed-precision keys (32 outlier channels), 4-bit values
        attend("decode_long_mixed", 1, 32, 8, 128, 131072, vb=4, store="kmixed32"),
        # a paged cache at head_dim 96, 4-bit keys and values, an odd context length
        attend("decode_paged", 12, 24, 8, 96, 3001, kb=4, vb=4, dtype="fp16", store="paged"),
        # the prompt pass of a Llama-3-8B layer: 2048 causal queries, in the model's type
        attend("prefill_prompt", 1, 32, 8, 128, 2048, Q=2048, out="bf16", causal=True),
        # a chunk of a longer prompt at head_dim 64, 7 query heads per kv head, odd sizes
        attend("prefill_chunk", 4, 14, 2, 64, 1501, Q=301, causal=True),
        # the prompts of 32 sequences of 8k tokens into a Llama-3-8B layer's cache
        dict(name="append_prompt", kind="append", B=32, H=8, S=8192, d=128, kb=3, vb=3,
             dtype="bf16", store="flat"),
        # a decode step's token of 16 sequences into the 24 layers of Qwen2.5-0.5B
        dict(name="append_token", kind="append_layers", L=24, B=16, H=2, S=1, d=64, kb=3, vb=3,
             dtype="bf16"),
        # the quantizer operators on fp32 rows, a row count that no tile divides
        dict(name="codec_rows", kind="codec", n=200003, d=128, bits=3, dtype="fp32"),
        # a Llama-3-8B layer's reconstructed K and V, 8 sequences of 8k tokens
        dict(name="rebuild_layer", kind="rebuild", B=8, H=8, T=8192, d=128, kb=3, vb=3),
        # top-10 of a million 128-dim vectors for 10,000 queries
        dict(name="search_million", kind="search", N=1000000, M=10000, d=128, bits=3, k=10),
    ]


def _lu(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "paged", "mixed", "prefill", "prefill", "layers",
                       "append", "append_layers", "codec", "rebuild", "search", "search"])
    d = rng.choice([64, 96, 128, 128])
    kb, vb = rng.choice([(3, 3), (3, 3), (2, 2), (4, 4), (3, 4)])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    Hkv = rng.choice([1, 2, 4, 8])
    G = rng.choice([1, 2, 3, 4, 4, 7, 8])
    if kind in ("decode", "paged"):
        T = _lu(rng, 64, 16384)
        B = max(1, min(_lu(rng, 1, 32), (1 << 21) // (Hkv * T)))
        c = attend("", B, Hkv * G, Hkv, d, T, Q=rng.choice([1, 1, 1, 4]), kb=kb, vb=vb,
                   dtype=dtype, store="paged" if kind == "paged" else "flat")
        c["causal"] = c["Q"] > 1
    elif kind == "mixed":
        T = _lu(rng, 1024, 131072)
        c = attend("", 1, Hkv * G, Hkv, 128, T, vb=rng.choice([2, 3, 4]), dtype=dtype,
                   store=rng.choice(["kmixed32", "kmixed64", "kipmixed32"]))
    elif kind == "prefill":
        Q = _lu(rng, 16, 2048)
        T = Q if rng.random() < 0.5 else Q + _lu(rng, 16, 4096)
        B = max(1, min(rng.choice([1, 1, 2, 4]), (1 << 27) // (Hkv * G * Q * T)))
        c = attend("", B, Hkv * G, Hkv, d, T, Q=Q, kb=kb, vb=vb, dtype=dtype,
                   out=rng.choice([dtype, "fp32"]), causal=True)
    elif kind == "layers":
        T = _lu(rng, 64, 4096)
        L = rng.choice([12, 24, 28, 32])
        B = max(1, min(_lu(rng, 1, 16), (1 << 21) // (Hkv * T * L)))
        c = dict(kind="layers", L=L, B=B, Hq=Hkv * G, Hkv=Hkv, d=d, T=T, kb=kb, vb=vb,
                 dtype=dtype)
    elif kind == "append":
        S = _lu(rng, 1, 8192)
        c = dict(kind="append", B=max(1, min(_lu(rng, 1, 32), (1 << 20) // (Hkv * S))), H=Hkv,
                 S=S, d=d, kb=kb, vb=vb, dtype=dtype, store="flat")
        if d == 128 and rng.random() < 0.4:
            c["store"] = rng.choice(["kmixed32", "kmixed64", "kipmixed32"])
    elif kind == "append_layers":
        c = dict(kind="append_layers", L=rng.choice([12, 24, 28, 32]), B=_lu(rng, 1, 32), H=Hkv,
                 S=rng.choice([1, 1, 1, 4]), d=d, kb=kb, vb=vb, dtype=dtype)
    elif kind == "codec":
        c = dict(kind="codec", n=_lu(rng, 1000, 400000), d=d, bits=rng.choice([2, 3, 4]),
                 dtype=dtype)
    elif kind == "rebuild":
        T = _lu(rng, 64, 8192)
        c = dict(kind="rebuild", B=max(1, min(_lu(rng, 1, 16), (1 << 19) // (Hkv * T))), H=Hkv,
                 T=T, d=d, kb=kb, vb=vb)
    else:
        c = dict(kind="search", N=_lu(rng, 10000, 1000000), M=_lu(rng, 1, 4000), d=d, bits=kb,
                 k=rng.choice([1, 10, 10, 32]))
    c.pop("name", None)
    return c


# ------------------------------------------------------------------ preparation

def _randn(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g, dtype=torch.float32)


def _keys_values(g, B, H, S, d, dtype):
    """N(0, 1) keys and values; every 32nd key channel is an outlier (x10), as keys have them."""
    k, v = _randn(g, B, H, S, d), _randn(g, B, H, S, d)
    k[..., ::32] *= 10.0
    return k.to(DTYPES[dtype]), v.to(DTYPES[dtype])


def _engine(g, store, d, kb, vb, capacity=0, seed=SEED):
    if store == "paged":
        return PagedQuashKVEngine(head_dim=d, key_bits=kb, value_bits=vb, seed=seed, device="cuda")
    kq = None
    if store.startswith("k"):
        cls = (quashkv.MixedPrecisionIPQuantizer if store.startswith("kip")
               else quashkv.MixedPrecisionMSEQuantizer)
        kq = cls(d, 3, 2, int(store[-2:]), seed=seed, device="cuda")
        cal = _randn(g, 8192, d)
        cal[:, ::32] *= 10.0
        kq.calibrate(cal)
    return quashkv.QuashKVEngine(head_dim=d, key_bits=kb, value_bits=vb, seed=seed, device="cuda",
                                 capacity=capacity, key_quantizer=kq)


def prepare(case, seed):
    c = dict(case)
    g = torch.Generator(device="cuda").manual_seed(seed)
    st = {"case": c}
    if c["kind"] == "attend":
        e = st["engine"] = _engine(g, c["store"], c["d"], c["kb"], c["vb"], c["T"])
        e.append(*_keys_values(g, c["B"], c["Hkv"], c["T"], c["d"], c["dtype"]))
        st["q"] = _randn(g, c["B"], c["Hq"], c["Q"], c["d"]).to(DTYPES[c["dtype"]])
    elif c["kind"] == "layers":
        engines = [_engine(g, "flat", c["d"], c["kb"], c["vb"], c["T"], SEED + i)
                   for i in range(c["L"])]
        for e in engines:
            e.append(*_keys_values(g, c["B"], c["Hkv"], c["T"], c["d"], c["dtype"]))
        st["engines"], st["batch"] = engines, LayerBatch(engines)
        st["q"] = [_randn(g, c["B"], c["Hq"], 1, c["d"]).to(DTYPES[c["dtype"]]) for _ in engines]
    elif c["kind"] == "append":
        e = st["engine"] = _engine(g, c["store"], c["d"], c["kb"], c["vb"], c["S"])
        st["k"], st["v"] = _keys_values(g, c["B"], c["H"], c["S"], c["d"], c["dtype"])
        e.append(st["k"][:, :, :1], st["v"][:, :, :1])   # the store exists, as in a reused cache
    elif c["kind"] == "append_layers":
        engines = [_engine(g, "flat", c["d"], c["kb"], c["vb"], 64, SEED + i)
                   for i in range(c["L"])]
        kv = [_keys_values(g, c["B"], c["H"], c["S"], c["d"], c["dtype"]) for _ in engines]
        for e, (k, v) in zip(engines, kv):
            e.append(k[:, :, :1], v[:, :, :1])
        st["engines"], st["batch"] = engines, LayerBatch(engines)
        st["k"], st["v"] = [k for k, _ in kv], [v for _, v in kv]
    elif c["kind"] == "codec":
        st["kq"] = quashkv.InnerProductQuantizer(c["d"], max(c["bits"], 2), seed=SEED,
                                                 device="cuda")
        st["vq"] = quashkv.MSEQuantizer(c["d"], c["bits"], seed=SEED, device="cuda")
        st["x"] = _randn(g, c["n"], c["d"]).to(DTYPES[c["dtype"]])
        st["codes"] = torch.randint(0, 1 << c["bits"], (c["n"], c["d"]), device="cuda",
                                    generator=g).to(torch.uint8)
        st["norms"] = _randn(g, c["n"]).abs() + 1.0
    elif c["kind"] == "rebuild":
        cache = st["cache"] = QuashKVCache(1, c["d"], device="cuda")
        e = quashkv.QuashKVEngine(head_dim=c["d"], key_bits=c["kb"], value_bits=c["vb"],
                                  seed=SEED, device="cuda", capacity=c["T"])
        cache.engines[0] = e
        e.append(*_keys_values(g, c["B"], c["H"], c["T"], c["d"], "bf16"))
    else:
        idx = st["index"] = QuashIndex(c["d"], bits=c["bits"], seed=SEED, device="cuda")
        db = _randn(g, c["N"], c["d"])
        idx.add(db / db.norm(dim=1, keepdim=True))
        q = _randn(g, c["M"], c["d"])
        st["q"] = q / q.norm(dim=1, keepdim=True)
    return st


# ------------------------------------------------------------------ one pass

def _store_arrays(e):
    s = e._store
    return {"krows": s.kst, "knorm": s.knorm, "vtiles": s.vst, "vnorm": s.vnorm}


def run(st):
    c = st["case"]
    if c["kind"] == "attend":
        return st["engine"].attention(st["q"], causal=c["causal"], out_dtype=DTYPES[c["out"]])
    if c["kind"] == "layers":
        return st["batch"](st["q"])
    if c["kind"] == "append":
        st["engine"].clear()
        st["engine"].append(st["k"], st["v"])
        return _store_arrays(st["engine"])
    if c["kind"] == "append_layers":
        for e in st["engines"]:
            e.clear()
        st["batch"].append(st["k"], st["v"])
        outs = [_store_arrays(e) for e in st["engines"]]
        # the first and the last layers' whole stores (64 outputs at most)
        return outs[:6] + outs[-6:]
    if c["kind"] == "codec":
        codes, bits, norms = st["kq"].compress(st["x"])
        return {"codes": codes, "bits": bits, "norms": norms,
                "rows": st["vq"].decompress(st["codes"], st["norms"])}
    if c["kind"] == "rebuild":
        return st["cache"][0]
    scores, indices = st["index"].search(st["q"], c["k"])
    return {"scores": scores, "indices": indices}


# ------------------------------------------------------------------ what it takes

def _store_bytes(d, kb, vb, store):
    """Packed bytes of one token of one kv head: K row, V bits, two norms."""
    if store.startswith("kmixed"):
        krow = 2 * d / 8 + int(store[-2:]) / 8
    elif store.startswith("kipmixed"):
        krow = 2 * d / 8 + int(store[-2:]) / 8
    else:
        krow = kb * d / 8
    return krow + vb * d / 8 + 8


def work(case):
    c = case
    size = {"fp32": 4, "bf16": 2, "fp16": 2}
    if c["kind"] in ("attend", "layers"):
        L, Q = c.get("L", 1), c.get("Q", 1)
        kv = c["B"] * c["Hkv"] * c["T"] * _store_bytes(c["d"], c["kb"], c["vb"],
                                                       c.get("store", "flat"))
        rows = c["B"] * c["Hq"] * Q
        keys = c["T"] - (Q - 1) / 2 if c.get("causal") else c["T"]
        io = rows * c["d"] * (size[c["dtype"]] + size[c.get("out", "fp32")])
        return {"bytes": L * (kv + io), "flops": L * rows * (keys * 4 * c["d"] + 4 * c["d"] ** 2)}
    if c["kind"] in ("append", "append_layers"):
        n = c.get("L", 1) * c["B"] * c["H"] * c["S"]
        return {"bytes": n * (2 * c["d"] * size[c["dtype"]]
                              + _store_bytes(c["d"], c["kb"], c["vb"], c.get("store", "flat"))),
                "flops": n * 4 * c["d"] ** 2}
    if c["kind"] == "codec":
        return {"bytes": c["n"] * (c["d"] * (size[c["dtype"]] + 2 + 1 + 4) + 8),
                "flops": c["n"] * 4 * c["d"] ** 2}
    if c["kind"] == "rebuild":
        n = c["B"] * c["H"] * c["T"]
        return {"bytes": n * (c["d"] * ((c["kb"] - 1 + c["vb"]) / 8 + 8) + 8),
                "flops": n * 4 * c["d"] ** 2}
    return {"bytes": c["N"] * (c["bits"] * c["d"] / 8 + 4) + c["M"] * (4 * c["d"] + 12 * c["k"]),
            "flops": 4.0 * c["N"] * c["M"] * c["d"]}


def tolerance(case):
    """About four times what the results were measured to be off their 64-bit values."""
    c = case
    if c["kind"] in ("attend", "layers"):
        # 16-bit results: their rounding (bf16 1.7e-3); fp32 ones: 8e-6, the score path's rounding
        out = c.get("out", "fp32")
        return {"rel": {"fp32": 4e-5, "fp16": 1e-3, "bf16": 6e-3}[out]}
    if c["kind"] in ("append", "append_layers"):
        # norms to fp32 rounding; a coordinate within the rotation's rounding of a threshold may
        # take the neighbouring code (up to 7e-6 of them; 8 share a byte, 32 a word)
        return {"rel": 1e-6, "differ": 6e-4}
    if c["kind"] == "codec":
        return {"rel": 1e-6, "differ": 3e-5}
    if c["kind"] == "rebuild":
        return {"rel": 1e-6}
    # scores 1.6e-7 off; equal or nearly equal ones may change places (none did in 60,000)
    return {"rel": 1e-6, "differ": 1e-4}


# ------------------------------------------------------------------ in 64 bits

def _codes_exact(x, pi, bounds):
    """(rotated unit rows, codes, norms) in 64 bits."""
    x = x.double()
    n = x.norm(dim=-1, keepdim=True).clamp(min=1e-8)
    y = (x / n) @ pi.double().T
    return y, torch.bucketize(y, bounds.double()), n.squeeze(-1)


def _attend_exact(e, q, causal):
    """softmax(scores) V of the engine's stored codes, in the dtype float64."""
    kc = torch.cat([b.mse_indices for b in e._cache], dim=2).long()
    vc = torch.cat([b.val_indices for b in e._cache], dim=2).long()
    kn = torch.cat([b.key_norms for b in e._cache], dim=2).double()
    vn = torch.cat([b.val_norms for b in e._cache], dim=2).double()
    ks = [b.qjl_signs for b in e._cache]
    ks = None if ks[0] is None else torch.cat(ks, dim=2)
    kq, vq = e.key_quantizer, e.value_quantizer
    mq = getattr(kq, "mse_quantizer", kq)
    pi, piv = mq.Pi.double(), vq.Pi.double()
    cv = vq.codebook.centroids.double()
    B, Hq, Q, d = q.shape
    Hkv, T = kc.shape[1], kc.shape[2]
    G = Hq // Hkv
    out = torch.empty(B, Hq, Q, d, dtype=torch.float64, device=q.device)
    mask = None
    if causal:
        pos = torch.arange(T, device=q.device)
        mask = pos[None, :] > (T - Q + torch.arange(Q, device=q.device))[:, None]
    if hasattr(mq, "outlier_codebook"):
        oc, rc = mq.outlier_codebook.centroids.double(), mq.regular_codebook.centroids.double()
    for b in range(B):
        for h in range(Hkv):
            if hasattr(mq, "outlier_codebook"):
                code = kc[b, h]
                kh = torch.where(mq._outlier_mask, oc[code], rc[code.clamp(max=rc.numel() - 1)])
            else:
                kh = mq.codebook.centroids.double()[kc[b, h]]
            vh = cv[vc[b, h]] * vn[b, h, :, None]
            for j in range(G):
                qr = q[b, h * G + j].double() @ pi.T
                s = qr @ kh.T
                if ks is not None:
                    sg = (2.0 * ks[b, h].double() - 1.0) * kq.S.double()
                    s = s + kq.qjl_scale * (qr.abs() @ sg.T)
                s = s * kn[b, h] / math.sqrt(d)
                if mask is not None:
                    s = s.masked_fill(mask, -math.inf)
                out[b, h * G + j] = (torch.softmax(s, dim=-1) @ vh) @ piv
    return out


def _search_exact(idx, q, k):
    codes, bits = idx._get_unpacked()
    norms = idx._norms[:codes.shape[0]].double()
    quant = idx.quantizer
    mq = quant.mse_quantizer
    c, s = mq.codebook.centroids.double(), quant.S.double()
    qr = q.double() @ mq.Pi.double().T
    qa = torch.cat([qr, quant.qjl_scale * qr.abs()], dim=1)
    best = idx_best = None
    step = max(1, int(4e8) // max(q.shape[0], 1))
    for a in range(0, codes.shape[0], step):
        rows = torch.cat([c[codes[a:a + step].long()],
                          (2.0 * bits[a:a + step].double() - 1.0) * s], dim=1)
        sc = (qa @ rows.T) * norms[a:a + step]
        v, i = torch.topk(sc, min(k, sc.shape[1]), dim=1)
        i = i + a
        if best is not None:
            v, i = torch.cat([best, v], dim=1), torch.cat([idx_best, i], dim=1)
            v, j = torch.topk(v, min(k, v.shape[1]), dim=1)
            i = i.gather(1, j)
        best, idx_best = v, i
    return {"scores": best, "indices": idx_best}


def exact(case, seed):
    c = dict(case)
    st = prepare(c, seed)
    if c["kind"] == "attend":
        return _attend_exact(st["engine"], st["q"], c["causal"])
    if c["kind"] == "layers":
        return [_attend_exact(e, q, False) for e, q in zip(st["engines"], st["q"])]
    if c["kind"] == "append":
        e, S = st["engine"], st["k"].shape[2]
        out = {"krows": None, "vtiles": None}
        for name, x in (("knorm", st["k"]), ("vnorm", st["v"])):
            n = torch.zeros(*x.shape[:2], e._store.capacity, dtype=torch.float64, device=x.device)
            n[:, :, :S] = x.double().norm(dim=-1).clamp(min=1e-8)
            out[name] = n
        return out
    if c["kind"] == "append_layers":
        outs = []
        for e, k, v in zip(st["engines"], st["k"], st["v"]):
            out = {"krows": None, "vtiles": None}
            for name, x in (("knorm", k), ("vnorm", v)):
                n = torch.zeros(*x.shape[:2], e._store.capacity, dtype=torch.float64,
                                device=x.device)
                n[:, :, :x.shape[2]] = x.double().norm(dim=-1).clamp(min=1e-8)
                out[name] = n
            outs.append(out)
        return outs[:6] + outs[-6:]
    if c["kind"] == "codec":
        kq, vq = st["kq"], st["vq"]
        mq = kq.mse_quantizer
        y, codes, norms = _codes_exact(st["x"], mq.Pi, mq.codebook.boundaries)
        r = y - mq.codebook.centroids.double()[codes]
        bits = (r * kq.S.double() >= 0).to(torch.uint8)
        rows = (vq.codebook.centroids.double()[st["codes"].long()] @ vq.Pi.double()) \
            * st["norms"].double()[:, None]
        return {"codes": codes.to(torch.uint8), "bits": bits, "norms": norms, "rows": rows}
    if c["kind"] == "rebuild":
        e = st["cache"].engines[0]
        b = e._cache[0]
        mq, vq = e.key_quantizer.mse_quantizer, e.value_quantizer
        k = (mq.codebook.centroids.double()[b.mse_indices.long()] @ mq.Pi.double()) \
            * b.key_norms.double()[..., None]
        v = (vq.codebook.centroids.double()[b.val_indices.long()] @ vq.Pi.double()) \
            * b.val_norms.double()[..., None]
        return [k, v]
    return _search_exact(st["index"], st["q"], c["k"])
