"""The timed workloads of the framework, each through its public entry points.

A case is one layer's pass over a batch, or one token-selection call:

  gqa        KVCache.AppendAttend of every sequence's new tokens over its
             paged cache, then the Rollback a speculative loop makes (it
             also keeps the context length fixed from pass to pass): decode
             (1 new token), verify (a few drafts) and chunked prefill
  mla        the same over an MLACache's latent rows
  gqa_block  a GQA layer's attention block: ProjectAppend (projection, RoPE,
             append), Attend, OutProject with the residual, Rollback
  mla_block  the same for an MLA layer
  sample     Sampler.SampleAsync on device logits
  accept     spec_accept_async: a batch's speculative acceptance

Sequence lengths are part of the case (drawn from its "mix"), so that work()
is known without a seed; everything else comes from prepare()'s seed.  Pages
are handed out to the sequences a page at a time in random order, as a
serving batch that grows together leaves them.
"""
import math
import random

import numpy as np
import torch

from relux_amd import (KVCache, MLACache, Sampler, pack_mla_proj, pack_out, pack_qkv, rope_tables,
                       spec_accept_async)

DEV = torch.device("cuda", 0)
DC, DR = 512, 64  # MLA latent and rope widths (DeepSeek-V2/V3)
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # One user, a short chat, the API's default f32 rows: launches and host time only.
        dict(name="gqa_decode_one", kind="gqa", B=1, H=32, KVH=8, D=128, P=16, T_lo=200, T_hi=200,
             n_lo=1, n_hi=1, mix=1, dtype="f32"),
        # An ordinary serving batch whose users are at different points of their chats.
        dict(name="gqa_decode_ragged", kind="gqa", B=16, H=32, KVH=8, D=128, P=16, T_lo=512, T_hi=4096,
             n_lo=1, n_hi=1, mix=2, dtype="bf16"),
        # The benchmark's headline: 16 users at 8k of context.
        dict(name="gqa_decode_8k", kind="gqa", B=16, H=32, KVH=8, D=128, P=16, T_lo=8192, T_hi=8192,
             n_lo=1, n_hi=1, mix=3, dtype="bf16"),
        # Speculative verify of 4 drafts for a full batch of 1k to 32k contexts: the most cache bytes.
        dict(name="gqa_verify", kind="gqa", B=64, H=64, KVH=8, D=128, P=16, T_lo=1024, T_hi=32768,
             n_lo=4, n_hi=4, mix=5, dtype="bf16"),
        # Prompts of odd lengths prefilled on top of a shared history, in one call.
        dict(name="gqa_prefill", kind="gqa", B=4, H=32, KVH=8, D=128, P=16, T_lo=1000, T_hi=4000,
             n_lo=700, n_hi=2048, mix=6, dtype="bf16"),
        # A DeepSeek-V2-Lite layer's whole attention block in decode at 8k.
        dict(name="mla_block_decode", kind="mla_block", B=32, H=16, D=128, P=64, T_lo=8192, T_hi=8192,
             n_lo=1, n_hi=1, mix=7, dtype="bf16", d_model=2048),
        # DeepSeek-V3's 128 heads in decode, uneven contexts around 8k.
        dict(name="mla_decode_h128", kind="mla", B=8, H=128, D=128, P=64, T_lo=6000, T_hi=10000,
             n_lo=1, n_hi=1, mix=8, dtype="bf16"),
        # A 2048-token chunk on 6144 cached tokens for 4 users, 128 heads: the most arithmetic.
        dict(name="mla_prefill", kind="mla", B=4, H=128, D=128, P=64, T_lo=6144, T_hi=6144,
             n_lo=2048, n_hi=2048, mix=9, dtype="bf16"),
        # One prompt of an odd length through a layer's attention block, from an empty cache.
        dict(name="gqa_block_prefill", kind="gqa_block", B=1, H=32, KVH=8, D=128, P=16, T_lo=0, T_hi=0,
             n_lo=1531, n_hi=1531, mix=10, dtype="bf16", d_model=4096),
        # A serving batch's sampling step with every stage of the sampler on.
        dict(name="sample_topk", kind="sample", B=64, V=32000, T=0.8, k=50, p=0.9, min_p=0.02, pen=1),
        # Nucleus sampling without top-k, a vocabulary whose rows are not 16-byte aligned.
        dict(name="sample_nucleus", kind="sample", B=16, V=50257, T=0.8, k=0, p=0.95, min_p=0.0, pen=0),
        # Acceptance of 4 drafts for 64 users over a 32k vocabulary.
        dict(name="spec_accept", kind="accept", B=64, K=4, V=32000, T=0.8, k=50, p=0.9),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 5e12, w["flops"] / 8e14)


def draw(rng):
    while True:
        c = _draw(rng)
        if _cost(c) <= 4e-3 and _slots(c) <= 700_000:
            return c


def _draw(rng):
    kind = rng.choice(["gqa", "gqa", "mla", "mla", "gqa_block", "mla_block", "sample", "accept"])
    if kind == "sample":
        mode = rng.choice(["topk", "topk", "nucleus", "plain"])
        return dict(kind=kind, B=_log(rng, 1, 64), V=_log(rng, 4000, 128000),
                    T=round(rng.uniform(0.6, 1.1), 2), k=rng.randint(1, 200) if mode == "topk" else 0,
                    p=1.0 if mode == "plain" else round(rng.uniform(0.7, 0.98), 2),
                    min_p=rng.choice([0.0, 0.02]), pen=rng.choice([0, 1]))
    if kind == "accept":
        return dict(kind=kind, B=_log(rng, 1, 64), K=rng.randint(1, 8), V=_log(rng, 4000, 64000),
                    T=round(rng.uniform(0.6, 1.1), 2), k=rng.randint(1, 200), p=round(rng.uniform(0.7, 0.98), 2))
    block = kind.endswith("_block")
    way = rng.choice(["decode", "verify", "prefill"])
    c = dict(kind=kind, mix=rng.randint(100, 10 ** 6), dtype=rng.choice(["bf16", "bf16", "f32"]))
    if way == "prefill":
        c["B"], n, T = _log(rng, 1, 4), _log(rng, 64, 2048), rng.choice([0, _log(rng, 64, 8192)])
        c["n_lo"], c["n_hi"] = max(1, n // 2), n
    else:
        c["B"], T = _log(rng, 1, 64), _log(rng, 64, 32768)
        c["n_lo"] = c["n_hi"] = 1 if way == "decode" else rng.randint(2, 5)
    c["T_hi"] = T
    c["T_lo"] = rng.choice([T, T // 2, T // 8])
    if kind.startswith("gqa"):
        c["H"], c["KVH"] = rng.choice([(32, 8), (32, 8), (64, 8), (16, 4), (16, 16), (8, 2)])
        c["D"] = rng.choice([128, 128, 64, 80])
        c["P"] = rng.choice([16, 16, 32, 64])
        if block:
            c["d_model"] = rng.choice([1024, 2048, 4096])
    else:
        c["H"] = rng.choice([16, 16, 32, 64, 128]) if not block else rng.choice([16, 32])
        c["D"], c["P"] = 128, rng.choice([16, 64, 64])
        if block:
            c["d_model"] = rng.choice([1024, 2048])
    return c


# ---- shapes and lengths ---------------------------------------------------------------

def _lens(case):
    """(cached tokens, new tokens) of every sequence."""
    r = random.Random(case["mix"])
    lo, hi = case["T_lo"], case["T_hi"]
    wide = lo > 0 and hi > 10 * lo
    T = [_log(r, lo, hi) if wide else r.randint(lo, hi) for _ in range(case["B"])]
    return T, [r.randint(case["n_lo"], case["n_hi"]) for _ in range(case["B"])]


def _slots(case):
    return sum(map(sum, _lens(case))) if "mix" in case else 0


def _rounds(case):
    """The history's appends, a page a sequence in a fresh random order each
    time: [(sequences, tokens of each)]."""
    T, _ = _lens(case)
    r = random.Random(case["mix"] + 1)
    left, out = list(T), []
    while any(left):
        order = [i for i in range(len(T)) if left[i]]
        r.shuffle(order)
        n = [min(case["P"], left[i]) for i in order]
        for i, k in zip(order, n):
            left[i] -= k
        out.append((order, n))
    return out


def _rows_of(case):
    """For every sequence the rows of the history, as appended, that are its."""
    got, at = [[] for _ in range(case["B"])], 0
    for order, n in _rounds(case):
        for i, k in zip(order, n):
            got[i].append(np.arange(at, at + k))
            at += k
    return [torch.from_numpy(np.concatenate(g) if g else np.zeros(0, np.int64)).to(DEV) for g in got]


def _inputs(case, seed):
    """The case's tensors, from the seed."""
    g = torch.Generator(device=DEV).manual_seed(int(seed))

    def randn(*shape, dtype=torch.float32):
        return torch.randn(*shape, device=DEV, dtype=dtype, generator=g)

    kind = case["kind"]
    if kind == "sample":
        B, V = case["B"], case["V"]
        x = randn(B, V) * 3.0
        return dict(x=x, hist=torch.randint(0, V, (B, 256), device=DEV, generator=g, dtype=torch.int32),
                    hist_len=torch.full((B,), 256, dtype=torch.int32, device=DEV),
                    u=torch.rand(B, device=DEV, generator=g))
    if kind == "accept":
        B, K, V = case["B"], case["K"], case["V"]
        d = randn(B, K, V) * 2.0
        t = torch.cat([d + randn(B, K, V) * 0.6, randn(B, 1, V) * 2.0], dim=1)
        tok = torch.multinomial(torch.softmax(d.reshape(B * K, V), dim=-1), 1, generator=g)
        return dict(d=d, t=t, tok=tok.reshape(B, K).to(torch.int32).contiguous(),
                    nd=torch.full((B,), K, dtype=torch.int32, device=DEV),
                    u=torch.rand(B, K + 1, device=DEV, generator=g))
    T, n = _lens(case)
    old, new, H, D, dt = sum(T), sum(n), case["H"], case["D"], DTYPES[case["dtype"]]
    bf = torch.bfloat16
    s = {}
    if kind.startswith("gqa"):
        KVH = case["KVH"]
        s["K"], s["V"] = randn(old, KVH, D, dtype=dt), randn(old, KVH, D, dtype=dt)
    else:
        s["C"], s["R"] = randn(old, DC, dtype=dt), randn(old, DR, dtype=dt)
        s["w_uk"] = (randn(DC, H * D) * 0.02).to(bf)
        s["w_uv"] = (randn(DC, H * D) * 0.02).to(bf)
    if kind.endswith("_block"):
        dm = case["d_model"]
        s["x"] = randn(new, dm, dtype=dt)
        wide = [H * D, KVH * D, KVH * D] if kind == "gqa_block" else [H * D, H * DR, DC, DR]
        s["w"] = [(randn(dm, k) * 0.02).to(bf) for k in wide]
        s["w_o"] = (randn(H * D, dm) * 0.02).to(bf)
    elif kind == "gqa":
        s["k"], s["v"] = randn(new, KVH, D, dtype=dt), randn(new, KVH, D, dtype=dt)
        s["q"] = randn(new, H, D, dtype=dt)
    else:
        s["c"], s["r"] = randn(new, DC, dtype=dt), randn(new, DR, dtype=dt)
        s["qn"], s["qr"] = randn(new, H, D, dtype=dt), randn(new, H, DR, dtype=dt)
    return s


# ---- the cases -------------------------------------------------------------------------

def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"], kind = case, case["kind"]
    if kind in ("sample", "accept"):
        # token selection runs on any cache's stream
        s["cache"] = KVCache(num_layers=1, max_len=16, num_kv_heads=1, head_dim=64)
        s["out"] = torch.empty(case["B"], dtype=torch.int32, device=DEV)
        s["out2"] = torch.empty(case["B"], dtype=torch.int32, device=DEV)
        pen = dict(repeat_penalty=1.1, frequency_penalty=0.1, presence_penalty=0.1, repeat_window=64)
        s["sampler"] = Sampler(temperature=case["T"], top_k=case["k"], top_p=case["p"],
                               min_p=case.get("min_p", 0.0), **(pen if case.get("pen") else {}))
        return s
    T, n = _lens(case)
    P, H, D, rows = case["P"], case["H"], case["D"], sum(n)
    pool = sum(-(-(a + b) // P) for a, b in zip(T, n)) + 8
    size = dict(num_layers=1, max_len=max(a + b for a, b in zip(T, n)), page_tokens=P, max_seqs=case["B"],
                pool_pages=pool)
    at = 0
    if kind.startswith("gqa"):
        c = KVCache(num_kv_heads=case["KVH"], head_dim=D, **size)
        for order, k in _rounds(case):
            m = sum(k)
            c.Append(0, s["K"][at:at + m], s["V"][at:at + m], seq_ids=order, n_tok=k, layout="SHD")
            at += m
        s["K"] = s["V"] = None
    else:
        c = MLACache(d_c=DC, d_r=DR, **size)
        for order, k in _rounds(case):
            m = sum(k)
            c.Append(0, s["C"][at:at + m], s["R"][at:at + m], seq_ids=order, n_tok=k)
            at += m
        s["C"] = s["R"] = None
    dt = DTYPES[case["dtype"]]
    s["cache"], s["seqs"], s["n"] = c, list(range(case["B"])), n
    s["out"] = torch.empty(rows, H, D, dtype=dt, device=DEV)
    if kind.endswith("_block"):
        s["wp"] = (pack_qkv(*s["w"], H, case["KVH"], D) if kind == "gqa_block"
                   else pack_mla_proj(*s["w"], H, D))
        s["wo"] = pack_out(s["w_o"])
        s["w"] = s["w_o"] = None
        s["rope"] = rope_tables(D if kind == "gqa_block" else DR, 10000.0, size["max_len"], DEV)
        s["y"] = torch.empty(rows, case["d_model"], dtype=dt, device=DEV)
    return s


def run(s):
    case, c = s["case"], s["cache"]
    kind = case["kind"]
    if kind == "sample":
        pen = case["pen"]
        return s["sampler"].SampleAsync(s["x"], s["hist"] if pen else None, s["hist_len"] if pen else None,
                                        s["u"], c, out=s["out"])
    if kind == "accept":
        return spec_accept_async(c, s["d"], s["t"], s["tok"], s["nd"], s["u"], s["sampler"],
                                 n_acc=s["out"], next_tok=s["out2"])
    H, D, seqs, n, dt = case["H"], case["D"], s["seqs"], s["n"], DTYPES[case["dtype"]]
    if kind == "gqa":
        got = c.AppendAttend(0, s["k"], s["v"], s["q"], H, seq_ids=seqs, n_tok=n, out=s["out"])
    elif kind == "mla":
        got = c.AppendAttend(0, s["c"], s["r"], s["qn"], s["qr"], s["w_uk"], s["w_uv"], H, D, seq_ids=seqs,
                             n_tok=n, out=s["out"])
    else:
        if kind == "gqa_block":
            q = c.ProjectAppend(0, s["x"], s["wp"], H, rope=s["rope"], seq_ids=seqs, n_tok=n, q_dtype=dt)
            o = c.Attend(0, q, H, seq_ids=seqs, n_q=n, out=s["out"])
            qs = [q]
        else:
            qs = c.ProjectAppend(0, s["x"], s["wp"], H, D, rope=s["rope"], seq_ids=seqs, n_tok=n, q_dtype=dt)
            o = c.Attend(0, *qs, s["w_uk"], s["w_uv"], H, D, seq_ids=seqs, n_q=n, out=s["out"])
        y = c.OutProject(o.view(-1, H * D), s["wo"], case["d_model"], residual=s["x"], out=s["y"])
        got = dict(q=list(qs), attn=o, y=y)
    c.Rollback(seqs, n)
    return got


def work(case):
    kind = case["kind"]
    if kind == "sample":
        return {"bytes": case["B"] * case["V"] * 4, "flops": case["B"] * case["V"] * 4}
    if kind == "accept":
        rows = case["B"] * (2 * case["K"] + 1)
        return {"bytes": rows * case["V"] * 4, "flops": rows * case["V"] * 4}
    T, n = _lens(case)
    live, rows, H, D = sum(T) + sum(n), sum(n), case["H"], case["D"]
    pairs = sum(a * b + b * (b + 1) // 2 for a, b in zip(T, n))
    e = 2 if case["dtype"] == "bf16" else 4
    if kind.startswith("gqa"):
        KVH = case["KVH"]
        byte = live * KVH * D * 4 + 2 * rows * H * D * e
        flops = 4 * pairs * H * D
        feat = (H + 2 * KVH) * D
        new = 2 * rows * KVH * D * e
    else:
        byte = live * (DC + DR) * 2 + rows * H * (2 * D + DR) * e + 2 * DC * H * D * 2
        absorbed = 2 * pairs * H * (2 * DC + DR) + 4 * rows * H * D * DC
        expanded = 2 * pairs * H * (2 * D + DR) + 4 * live * DC * H * D
        flops = min(absorbed, expanded)
        feat = H * (D + DR) + DC + DR
        new = rows * (DC + DR) * e
    if kind.endswith("_block"):
        dm = case["d_model"]
        byte += (feat + H * D) * dm * 2 + 2 * rows * dm * e
        flops += 2 * rows * dm * (feat + H * D)
    else:
        byte += new
    return {"bytes": byte, "flops": flops}


def tolerance(case):
    if case["kind"] in ("sample", "accept"):
        return {"rel": 0.0, "max": 0.0, "differ": 0.01}  # a draw within a few ulp of a boundary
    # bf16 rows and weights of the softmax: 0.002 to 0.003 off the 64-bit result at every shape, a
    # few bf16 steps at the worst element
    return {"rel": 1e-2, "max": 0.1}


# ---- what the results are, in 64 bits --------------------------------------------------

def _mm(a, b):
    return torch.matmul(a.double(), b.double())


def _attend(q, k, v, n, scale):
    """[rows, dk] queries of the last n tokens, `rows // n` heads a token
    (token-major), over k [T, dk], v [T, dv]: causal softmax attention."""
    rows, T = q.shape[0], k.shape[0]
    s = torch.matmul(q, k.t().contiguous()) * scale
    if n > 1:
        last = T - n + torch.arange(n, device=DEV).repeat_interleave(rows // n)
        s.masked_fill_(torch.arange(T, device=DEV)[None, :] > last[:, None], -math.inf)
    return torch.matmul(torch.softmax(s, dim=-1), v)


def _gqa(q, K, V, H, D, n):
    """q [n, H, D] over K, V [T, KVH, D]."""
    KVH = K.shape[1]
    G = H // KVH
    out = torch.empty(n, H, D, dtype=torch.float64, device=DEV)
    for h in range(KVH):
        o = _attend(q[:, h * G:(h + 1) * G].reshape(n * G, D).double(), K[:, h].double(), V[:, h].double(), n,
                    1.0 / math.sqrt(D))
        out[:, h * G:(h + 1) * G] = o.view(n, G, D)
    return out


def _mla(qn, qr, C, R, w_uk, w_uv, H, D, n):
    """qn [n, H, D], qr [n, H, DR] over the latents C [T, DC], R [T, DR]."""
    kr = torch.cat([C, R], dim=1).double()
    uk, uv = w_uk.double().view(DC, H, D), w_uv.double().view(DC, H, D)
    out = torch.empty(n, H, D, dtype=torch.float64, device=DEV)
    step = max(1, min(H, (1 << 27) // max(1, n * C.shape[0])))
    for h in range(0, H, step):
        m = min(step, H - h)
        lat = torch.stack([torch.matmul(qn[:, h + i].double(), uk[:, h + i].t().contiguous()) for i in range(m)],
                          dim=1)
        q = torch.cat([lat, qr[:, h:h + m].double()], dim=2).reshape(n * m, DC + DR)
        o = _attend(q, kr, C.double(), n, 1.0 / math.sqrt(D + DR)).view(n, m, DC)
        for i in range(m):
            out[:, h + i] = torch.matmul(o[:, i].contiguous(), uv[:, h + i].contiguous())
    return out


def _rope(x, pos, tables):
    """Rotates the pairs (2i, 2i + 1) of x [rows, heads, d] by its rows' positions."""
    c, s = (t.double()[pos][:, None, :] for t in tables)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, a * s + b * c], dim=-1).flatten(-2)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("sample", "accept"):
        return None
    s, rows_of = _inputs(case, seed), _rows_of(case)
    T, n = _lens(case)
    H, D, dt, bf = case["H"], case["D"], DTYPES[case["dtype"]], torch.bfloat16
    at = np.concatenate([[0], np.cumsum(n)])
    new = [slice(int(at[i]), int(at[i + 1])) for i in range(case["B"])]
    if kind.endswith("_block"):
        # q and the cached rows are values of their stored types, as the interface states
        pos = torch.cat([torch.arange(a, a + b, device=DEV) for a, b in zip(T, n)])
        p = [_mm(s["x"], w) for w in s["w"]]
        tables = rope_tables(D if kind == "gqa_block" else DR, 10000.0, max(a + b for a, b in zip(T, n)), DEV)
        if kind == "gqa_block":
            KVH = case["KVH"]
            s["q"] = _rope(p[0].view(-1, H, D), pos, tables).to(dt)
            s["k"] = _rope(p[1].view(-1, KVH, D), pos, tables)
            s["v"] = p[2].view(-1, KVH, D)
            qs = [s["q"]]
        else:
            s["qn"] = p[0].view(-1, H, D).to(dt)
            s["qr"] = _rope(p[1].view(-1, H, DR), pos, tables).to(dt)
            s["c"], s["r"] = p[2], _rope(p[3].view(-1, 1, DR), pos, tables).view(-1, DR)
            qs = [s["qn"], s["qr"]]
    out = torch.empty(int(at[-1]), H, D, dtype=torch.float64, device=DEV)
    for i in range(case["B"]):
        def cached(old, fresh):
            return torch.cat([old[rows_of[i]].to(bf), fresh[new[i]].to(bf)])
        if kind.startswith("gqa"):
            out[new[i]] = _gqa(s["q"][new[i]], cached(s["K"], s["k"]), cached(s["V"], s["v"]), H, D, n[i])
        else:
            out[new[i]] = _mla(s["qn"][new[i]], s["qr"][new[i]], cached(s["C"], s["c"]), cached(s["R"], s["r"]),
                               s["w_uk"], s["w_uv"], H, D, n[i])
    if not kind.endswith("_block"):
        return out
    y = _mm(out.to(dt).view(-1, H * D), s["w_o"]) + s["x"].double()
    return dict(q=[q.double() for q in qs], attn=out, y=y)
