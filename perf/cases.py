"""The work this framework is timed on: attention calls through its public entry points.

Each case is a dict of plain values.  ``kind`` names the call:

* ``dense``   one ``flash_attn_func`` forward, ``[B, S, H, D]`` inputs (inference prefill, encoders);
* ``train``   forward and backward of ``flash_attn_func`` / ``flash_attn_qkvpacked_func``, every gradient returned;
* ``varlen``  ``flash_attn_varlen_func`` on packed sequences, forward, or forward and backward with ``backward``;
* ``cache``   ``flash_attn_with_kvcache``: single-token decode, decode with append and rotary, chunked prefill;
* ``int8``    ``attention_int8`` on ``[B, H, S, D]`` inputs, K quantization included.

``prepare`` builds what a program holds before the call, ``run`` is one pass, ``exact`` the same outputs in float64
torch without this package, ``work`` the bytes and flops a pass cannot do without, ``tolerance`` the error another
correct implementation with 16-bit operands and fp32 accumulation would show.
"""
import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.getcwd(), "flash-attn-triton_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
DEV = "cuda"


# ----------------------------------------------------------------------------- the cases
def listed():
    return [
        # Smallest: one attention call of a small model; launches and host latency decide.
        dict(name="dense_small", kind="dense", dtype="fp16", B=2, Sq=256, Sk=256, Hq=4, Hk=4, D=64, causal=False),
        # An ordinary encoder layer at head dim 64 (a row of the reference's published table).
        dict(name="dense_d64", kind="dense", dtype="fp16", B=4, Sq=1024, Sk=1024, Hq=32, Hk=32, D=64, causal=False),
        # Prompt prefill of a grouped-query decoder, ragged length.
        dict(name="prefill_gqa", kind="dense", dtype="bf16", B=2, Sq=3001, Sk=3001, Hq=32, Hk=8, D=128, causal=True),
        # The headline benchmark: long causal prefill.
        dict(name="prefill_long", kind="dense", dtype="fp16", B=4, Sq=4096, Sk=4096, Hq=32, Hk=32, D=128, causal=True),
        # Training step of one attention layer at head dim 64 on packed QKV.
        dict(name="train_d64", kind="train", dtype="bf16", B=8, S=1024, Hq=16, Hk=16, D=64, causal=True, packed=True),
        # The same at head dim 128 and long sequences (the largest case).
        dict(name="train_d128", kind="train", dtype="fp16", B=4, S=4096, Hq=32, Hk=32, D=128, causal=True, packed=False),
        # Packed prefill with a sliding window, ALiBi and softcap.
        dict(name="varlen_features", kind="varlen", dtype="fp16", n=32, lo=128, hi=4096, lens=0, Hq=16, Hk=16, D=128,
             causal=True, window=1024, alibi=True, softcap=30.0, backward=False),
        # Training on packed documents of uneven length, grouped KV heads.
        dict(name="varlen_train", kind="varlen", dtype="bf16", n=8, lo=100, hi=2048, lens=1, Hq=16, Hk=4, D=128,
             causal=True, window=-1, alibi=False, softcap=0.0, backward=True),
        # Serving: one decode step of a full batch on a paged cache.
        dict(name="decode_paged", kind="cache", dtype="fp16", B=64, Sq=1, Hq=32, Hk=8, D=128, page=256, cap=8192,
             lo=512, hi=8192, lens=0, append=False, causal=False),
        # Serving: one decode step of a small batch that rotates and appends the new token.
        dict(name="decode_append", kind="cache", dtype="bf16", B=8, Sq=1, Hq=32, Hk=8, D=128, page=0, cap=2048,
             lo=100, hi=2000, lens=2, append=True, causal=True),
        # Serving: a chunk of a long prompt against the pages already cached.
        dict(name="chunk_prefill", kind="cache", dtype="bf16", B=4, Sq=512, Hq=32, Hk=8, D=128, page=256, cap=8192,
             lo=512, hi=8192, lens=3, append=False, causal=True),
        # The quantized-QK forward at the headline shape.
        dict(name="int8_long", kind="int8", dtype="fp16", B=4, S=4096, Hq=32, D=128, causal=True),
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heads(rng):
    hq = rng.choice([4, 8, 16, 32])
    return hq, rng.choice([h for h in (hq, hq // 2, hq // 4) if h >= 1])


def _draw(rng):
    kind = rng.choice(["dense", "dense", "dense", "train", "train", "varlen", "varlen", "cache", "cache", "cache", "int8"])
    dtype = "fp16" if kind == "int8" else rng.choice(["fp16", "bf16"])
    D = rng.choice([64, 128])
    hq, hk = _heads(rng)
    if kind == "dense":
        s = _log(rng, 64, 8192)
        # mostly self attention; now and then a query block shorter or longer than its keys
        sk = s if rng.random() < 0.75 else _log(rng, 64, 8192)
        return dict(kind=kind, dtype=dtype, B=rng.randint(1, 8), Sq=s, Sk=sk, Hq=hq, Hk=hk, D=D,
                    causal=sk == s and rng.random() < 0.6)
    if kind == "train":
        packed = rng.random() < 0.4
        return dict(kind=kind, dtype=dtype, B=rng.randint(1, 8), S=_log(rng, 128, 4096), Hq=hq, Hk=hq if packed else hk,
                    D=D, causal=rng.random() < 0.7, packed=packed)
    if kind == "varlen":
        hi = _log(rng, 256, 4096)
        features = rng.random() < 0.4
        return dict(kind=kind, dtype=dtype, n=rng.randint(2, 32), lo=max(1, hi // 32), hi=hi, lens=rng.randint(0, 999),
                    Hq=hq, Hk=hk, D=D, causal=features or rng.random() < 0.8, window=1024 if features else -1,
                    alibi=features, softcap=30.0 if features else 0.0, backward=not features and rng.random() < 0.5)
    if kind == "cache":
        hi = _log(rng, 256, 8192)
        mode = rng.choice(["decode", "append", "chunk"])
        paged = mode != "append" or rng.random() < 0.5
        sq = 1 if mode != "chunk" else _log(rng, 32, 1024)
        hi = max(hi, sq)
        cap = -(-(hi + sq) // 256) * 256
        return dict(kind=kind, dtype=dtype, B=_log(rng, 1, 64) if mode != "chunk" else rng.randint(1, 4), Sq=sq, Hq=hq,
                    Hk=hk, D=D, page=rng.choice([64, 256]) if paged else 0, cap=cap, lo=max(sq, hi // 16), hi=hi,
                    lens=rng.randint(0, 999), append=mode == "append", causal=mode != "decode")
    return dict(kind=kind, dtype=dtype, B=rng.randint(1, 4), S=64 * _log(rng, 2, 64), Hq=hq, D=D,
                causal=rng.random() < 0.6)


def draw(rng):
    top = work(next(c for c in listed() if c["name"] == "train_d128"))["flops"]
    while True:
        case = _draw(rng)
        if work(case)["flops"] <= top:
            return case


# ----------------------------------------------------------------------------- shared pieces
def _lengths(case):
    rng = random.Random(case["lens"])
    n = case["n"] if case["kind"] == "varlen" else case["B"]
    return [rng.randint(case["lo"], case["hi"]) for _ in range(n)]


def _cu(case):
    lengths = _lengths(case)
    cu = [0]
    for n in lengths:
        cu.append(cu[-1] + n)
    return lengths, cu


def _randn(gen, *shape, dtype):
    return torch.randn(*shape, generator=gen, device=DEV, dtype=torch.float32).to(dtype)


def _slopes(heads):
    return (2.0 ** (-8.0 * (torch.arange(heads) + 1) / heads)).float().to(DEV)


def _visible(sq, sk, causal, offset=0, window=-1):
    """Visible (query, key) pairs of one head."""
    if not causal:
        return sq * sk
    total = 0
    for i in range(sq):
        last = min(sk - 1, i + offset)
        first = max(0, i + offset - window) if window >= 0 else 0
        total += max(0, last - first + 1)
    return total


def work(case):
    kind, D, hq = case["kind"], case["D"], case["Hq"]
    hk = case.get("Hk", hq)
    if kind == "dense":
        pairs = case["B"] * _visible(case["Sq"], case["Sk"], case["causal"])
        nbytes = 2 * D * case["B"] * (2 * case["Sq"] * hq + 2 * case["Sk"] * hk)
        return dict(bytes=nbytes, flops=4 * D * hq * pairs)
    if kind == "train":
        # forward 2 products a pair, backward 5; q, k, v, out, dout, dq, dk, dv
        pairs = case["B"] * _visible(case["S"], case["S"], case["causal"])
        nbytes = 2 * D * case["B"] * case["S"] * (4 * hq + 4 * hk)
        return dict(bytes=nbytes, flops=14 * D * hq * pairs)
    if kind == "varlen":
        lengths, cu = _cu(case)
        pairs = sum(_visible(n, n, case["causal"], 0, case["window"]) for n in lengths)
        if case["backward"]:
            return dict(bytes=2 * D * cu[-1] * (4 * hq + 4 * hk), flops=14 * D * hq * pairs)
        return dict(bytes=2 * D * cu[-1] * (2 * hq + 2 * hk), flops=4 * D * hq * pairs)
    if kind == "cache":
        new = 1 if case["append"] else 0
        lengths = [n + new for n in _lengths(case)]
        pairs = sum(_visible(case["Sq"], n, case["causal"], n - case["Sq"]) for n in lengths)
        nbytes = 2 * D * (2 * hk * sum(lengths) + 2 * hq * case["B"] * case["Sq"] + 4 * hk * case["B"] * new)
        return dict(bytes=nbytes, flops=4 * D * hq * pairs)
    pairs = case["B"] * _visible(case["S"], case["S"], case["causal"])
    return dict(bytes=2 * D * hq * case["B"] * case["S"] * 4, flops=4 * D * hq * pairs)


def tolerance(case):
    # About four times the measured distance to float64 (fp16 3.2e-4, bf16 2.6e-3: the operands' and P's rounding),
    # gradients included.
    return {"rel": 1.3e-3 if case["dtype"] == "fp16" else 1e-2}


# ----------------------------------------------------------------------------- inputs
def _cache_tables(case):
    """Block table (rows of page numbers) of a paged case: the used pages in a shuffled pool."""
    page, per = case["page"], -(-case["cap"] // case["page"])
    new = 1 if case["append"] else 0
    used = [-(-(n + new) // page) for n in _lengths(case)]
    pool = list(range(sum(used)))
    random.Random(case["lens"] + 1).shuffle(pool)
    rows, at = [], 0
    for n in used:
        rows.append(pool[at:at + n] + [0] * (per - n))
        at += n
    return rows, sum(used)


def prepare(case, seed):
    dt = DTYPES[case["dtype"]]
    gen = torch.Generator(device=DEV).manual_seed(seed)
    kind, D, hq = case["kind"], case["D"], case["Hq"]
    hk = case.get("Hk", hq)
    st = {"case": case}
    if kind == "dense":
        st["q"] = _randn(gen, case["B"], case["Sq"], hq, D, dtype=dt)
        st["k"] = _randn(gen, case["B"], case["Sk"], hk, D, dtype=dt)
        st["v"] = _randn(gen, case["B"], case["Sk"], hk, D, dtype=dt)
    elif kind == "train":
        B, S = case["B"], case["S"]
        if case["packed"]:
            st["qkv"] = _randn(gen, B, S, 3, hq, D, dtype=dt).requires_grad_()
        else:
            st["q"] = _randn(gen, B, S, hq, D, dtype=dt).requires_grad_()
            st["k"] = _randn(gen, B, S, hk, D, dtype=dt).requires_grad_()
            st["v"] = _randn(gen, B, S, hk, D, dtype=dt).requires_grad_()
        st["dout"] = _randn(gen, B, S, hq, D, dtype=dt)
    elif kind == "varlen":
        lengths, cu = _cu(case)
        st["q"] = _randn(gen, cu[-1], hq, D, dtype=dt)
        st["k"] = _randn(gen, cu[-1], hk, D, dtype=dt)
        st["v"] = _randn(gen, cu[-1], hk, D, dtype=dt)
        if case["backward"]:
            for name in ("q", "k", "v"):
                st[name].requires_grad_()
            st["dout"] = _randn(gen, cu[-1], hq, D, dtype=dt)
        st["cu"] = torch.tensor(cu, dtype=torch.int32, device=DEV)
        st["max"] = max(lengths)
        st["slopes"] = _slopes(hq) if case["alibi"] else None
    elif kind == "cache":
        lengths = _lengths(case)
        st["q"] = _randn(gen, case["B"], case["Sq"], hq, D, dtype=dt)
        st["lens"] = torch.tensor(lengths, dtype=torch.int32, device=DEV)
        st["table"] = None
        if case["page"]:
            rows, pages = _cache_tables(case)
            st["table"] = torch.tensor(rows, dtype=torch.int32, device=DEV)
            shape = (pages, case["page"], hk, D)
        else:
            shape = (case["B"], case["cap"], hk, D)
        st["kc"] = _randn(gen, *shape, dtype=dt)
        st["vc"] = _randn(gen, *shape, dtype=dt)
        if case["append"]:
            st["kn"] = _randn(gen, case["B"], 1, hk, D, dtype=dt)
            st["vn"] = _randn(gen, case["B"], 1, hk, D, dtype=dt)
            pos = torch.arange(case["cap"], dtype=torch.float32)[:, None]
            ang = pos * (10000.0 ** (-torch.arange(0, D, 2, dtype=torch.float32) / D))[None, :]
            st["cos"], st["sin"] = ang.cos().to(DEV).to(dt), ang.sin().to(DEV).to(dt)
    else:
        B, S = case["B"], case["S"]
        for name in ("q", "k", "v"):
            st[name] = _randn(gen, B, hq, S, D, dtype=dt)
        # one key row in a hundred is an outlier, as per-token quantization meets them
        rows = torch.rand(B, hq, S, 1, generator=gen, device=DEV) < 0.01
        st["k"] = torch.where(rows, st["k"] * 8, st["k"])
    return st


# ----------------------------------------------------------------------------- one pass
def run(st):
    import flash_attn_triton as fa

    case = st["case"]
    kind = case["kind"]
    if kind == "dense":
        return fa.flash_attn_func(st["q"], st["k"], st["v"], causal=case["causal"])
    if kind == "train":
        if case["packed"]:
            out = fa.flash_attn_qkvpacked_func(st["qkv"], causal=case["causal"])
            return (out,) + torch.autograd.grad(out, (st["qkv"],), st["dout"])
        out = fa.flash_attn_func(st["q"], st["k"], st["v"], causal=case["causal"])
        return (out,) + torch.autograd.grad(out, (st["q"], st["k"], st["v"]), st["dout"])
    if kind == "varlen":
        window = (case["window"], 0) if case["window"] >= 0 else (-1, -1)
        out = fa.flash_attn_varlen_func(st["q"], st["k"], st["v"], st["cu"], st["cu"], st["max"], st["max"],
                                        causal=case["causal"], window_size=window, softcap=case["softcap"],
                                        alibi_slopes=st["slopes"])
        if not case["backward"]:
            return out
        return (out,) + torch.autograd.grad(out, (st["q"], st["k"], st["v"]), st["dout"])
    if kind == "cache":
        if case["append"]:
            out = fa.flash_attn_with_kvcache(st["q"], st["kc"], st["vc"], k=st["kn"], v=st["vn"], rotary_cos=st["cos"],
                                             rotary_sin=st["sin"], cache_seqlens=st["lens"], block_table=st["table"],
                                             causal=case["causal"], rotary_interleaved=False)
            return out, st["kc"], st["vc"]
        return fa.flash_attn_with_kvcache(st["q"], st["kc"], st["vc"], cache_seqlens=st["lens"],
                                          block_table=st["table"], causal=case["causal"])
    from flash_attn_triton.triton_kernel.attention_kernel_int8 import attention_int8

    return attention_int8(st["q"], st["k"], st["v"], causal=case["causal"])


# ----------------------------------------------------------------------------- float64
def _keep(sq, sk, causal, offset=0, window=-1):
    i = torch.arange(sq, device=DEV)[:, None] + offset
    j = torch.arange(sk, device=DEV)[None, :]
    keep = torch.ones(sq, sk, dtype=torch.bool, device=DEV)
    if causal:
        keep &= j <= i
    if window >= 0:
        keep &= j >= i - window
    return keep, (i - j).abs()


def _head64(q, k, v, keep, dist=None, slope=0.0, softcap=0.0, scores=None, dout=None):
    """One head in float64: q [Sq, D], k / v [Sk, D]; the output, and with dout the gradients of q, k and v."""
    scale = 1.0 / math.sqrt(q.shape[-1])
    s = (q @ k.t().contiguous()) * scale if scores is None else scores
    if slope:
        s -= slope * dist
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    s.masked_fill_(~keep, -math.inf)
    top = s.amax(1, keepdim=True)
    s.sub_(torch.where(torch.isfinite(top), top, torch.zeros_like(top))).exp_()
    p = s.div_(s.sum(1, keepdim=True).clamp_min(1e-300))
    out = p @ v
    if dout is None:
        return out
    dv = p.t().contiguous() @ dout
    ds = dout @ v.t().contiguous()
    ds.sub_((dout * out).sum(1, keepdim=True)).mul_(p).mul_(scale)
    return out, ds @ k, ds.t().contiguous() @ q, dv


def _dense64(q, k, v, causal, dout=None):
    """[B, S, H, D] inputs: the output, with dout (out, dq, dk, dv)."""
    B, sq, hq, D = q.shape
    sk, hk = k.shape[1], k.shape[2]
    keep, _ = _keep(sq, sk, causal)
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    if dout is not None:
        dq = torch.empty_like(out)
        dk = torch.zeros(k.shape, dtype=torch.float64, device=DEV)
        dv = torch.zeros_like(dk)
    for b in range(B):
        for h in range(hq):
            kh = h // (hq // hk)
            args = (q[b, :, h].double(), k[b, :, kh].double(), v[b, :, kh].double(), keep)
            if dout is None:
                out[b, :, h] = _head64(*args)
            else:
                out[b, :, h], dq[b, :, h], gk, gv = _head64(*args, dout=dout[b, :, h].double())
                dk[b, :, kh] += gk
                dv[b, :, kh] += gv
    return out if dout is None else (out, dq, dk, dv)


def _rotate64(x, cos, sin, pos):
    """x [n, H, D] at positions pos [n]; halves rotated against each other."""
    half = x.shape[-1] // 2
    c, s = cos[pos].double()[:, None, :], sin[pos].double()[:, None, :]
    a, b = x[..., :half], x[..., half:]
    return torch.cat((a * c - b * s, a * s + b * c), -1)


def _cache64(st):
    case = st["case"]
    B, sq, hq, D = st["q"].shape
    hk = case["Hk"]
    out = torch.empty(st["q"].shape, dtype=torch.float64, device=DEV)
    kc, vc = st["kc"], st["vc"]
    if case["append"]:
        kc, vc = kc.double(), vc.double()
    for b, n in enumerate(_lengths(case)):
        if case["page"]:
            slots = torch.arange(n + 1, device=DEV)
            page = st["table"][b].long()[(slots // case["page"]).clamp_max(st["table"].shape[1] - 1)]
            at = (page, slots % case["page"])
        else:
            slots = torch.arange(n + 1, device=DEV).clamp_max(kc.shape[1] - 1)
            at = (torch.full_like(slots, b), slots)
        q = st["q"][b].double()
        if case["append"]:
            pos = torch.tensor([n], device=DEV)
            kc[at[0][n], at[1][n]] = _rotate64(st["kn"][b].double(), st["cos"], st["sin"], pos)[0]
            vc[at[0][n], at[1][n]] = st["vn"][b, 0].double()
            q = _rotate64(q, st["cos"], st["sin"], pos)
            n += 1
        k, v = kc[at[0][:n], at[1][:n]].double(), vc[at[0][:n], at[1][:n]].double()
        keep, _ = _keep(sq, n, case["causal"], n - sq)
        for h in range(hq):
            kh = h // (hq // hk)
            out[b, :, h] = _head64(q[:, h].contiguous(), k[:, kh].contiguous(), v[:, kh].contiguous(), keep)
    return (out, kc, vc) if case["append"] else out


def _round_away(x):
    return torch.where(x >= 0, torch.floor(x + 0.5), torch.ceil(x - 0.5))


def _int8_64(st):
    """Per-token int8 Q and K (the quantizer is part of the call's contract), the rest in float64."""
    case = st["case"]
    q, k, v = st["q"], st["k"], st["v"]
    keep, _ = _keep(case["S"], case["S"], case["causal"])
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    scale = 1.0 / math.sqrt(case["D"])
    sq = q.float().abs().amax(-1, keepdim=True).clamp_min(1.0) / 127.0
    sk = k.float().abs().amax(-1, keepdim=True).clamp_min(1.0) / 127.0
    q8 = _round_away(q.float() / sq)
    k8 = _round_away(k.float() * (1.0 / sk))
    for b in range(case["B"]):
        for h in range(case["Hq"]):
            s = q8[b, h].double() @ k8[b, h].double().t().contiguous()
            s *= sq[b, h].double() * scale
            s *= sk[b, h].double().t()
            out[b, h] = _head64(q[b, h].double(), None, v[b, h].double(), keep, scores=s)
    return out


@torch.no_grad()
def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    if kind == "dense":
        return _dense64(st["q"], st["k"], st["v"], case["causal"])
    if kind == "train":
        if case["packed"]:
            q, k, v = st["qkv"].detach().unbind(2)
            out, dq, dk, dv = _dense64(q, k, v, case["causal"], st["dout"])
            return out, torch.stack((dq, dk, dv), 2)
        return _dense64(st["q"].detach(), st["k"].detach(), st["v"].detach(), case["causal"], st["dout"])
    if kind == "varlen":
        lengths, cu = _cu(case)
        q, k, v = (st[n].detach() for n in ("q", "k", "v"))
        back = case["backward"]
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        dq, dk, dv = (torch.zeros(t.shape, dtype=torch.float64, device=DEV) for t in (q, k, v)) if back else (None,) * 3
        group = case["Hq"] // case["Hk"]
        slopes = st["slopes"].double().tolist() if case["alibi"] else [0.0] * case["Hq"]
        for at, n in zip(cu, lengths):
            row = slice(at, at + n)
            keep, dist = _keep(n, n, case["causal"], 0, case["window"])
            for h in range(case["Hq"]):
                kh = h // group
                args = (q[row, h].double(), k[row, kh].double(), v[row, kh].double(), keep, dist, slopes[h],
                        case["softcap"])
                if back:
                    out[row, h], dq[row, h], gk, gv = _head64(*args, dout=st["dout"][row, h].double())
                    dk[row, kh] += gk
                    dv[row, kh] += gv
                else:
                    out[row, h] = _head64(*args)
        return (out, dq, dk, dv) if back else out
    if kind == "cache":
        return _cache64(st)
    return _int8_64(st)
