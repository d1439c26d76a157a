"""Chunked prefill with its tiles cut along the keys, GQA prefill at stored
head dim 96, and the absorbed MLA kernel past 1024 query rows, against exact
softmax attention in f64 over the rounded cache rows (max-abs 1e-2, mean-abs
1e-3, the bars of the other attention tests), and the cut against the whole
tiles (a handle whose workspace may not grow keeps them whole)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _limit(mask, T, n, i):
    if mask == "causal":
        return T - n + i
    return i if (mask == "ref" and n == T) else T - 1


def _exact(q, k, v, n, mask, scale):
    """q [n, H, dk] over k [T, KVH, dk], v [T, KVH, dv] (f64)."""
    T, KVH, G = k.shape[0], k.shape[1], q.shape[1] // k.shape[1]
    lim = torch.tensor([_limit(mask, T, n, i) for i in range(n)], device=q.device)
    bad = torch.arange(T, device=q.device)[None, :] > lim[:, None]
    out = []
    for h in range(q.shape[1]):
        s = torch.matmul(q[:, h], k[:, h // G].t().contiguous()) * scale
        out.append(torch.matmul(torch.softmax(s.masked_fill(bad, -math.inf), -1), v[:, h // G]))
    return torch.stack(out, 1)


def _check(got, want):
    e = (got.double() - want).abs()
    assert float(e.max()) <= 1e-2 and float(e.mean()) <= 1e-3, (float(e.max()), float(e.mean()))


# few work-groups over long contexts (cut tiles): one row past the decode
# kernel's 32, tile edges (64 tokens x 4 heads), a group that does not divide
# 256, causal tiles of unequal lengths, rows whose first part is all masked
# (the ref mask's whole-prompt case), every stored head dim of the kernel
GQA = [
    (4, 2, 128, 16, [3000], [17], "causal", "SHD", False),
    (8, 2, 128, 16, [2049, 700], [64, 9], "causal", "HSD", True),
    (6, 2, 64, 48, [4000], [65], "none", "SHD", False),
    (4, 1, 128, 16, [0], [1100], "causal", "SHD", False),
    (4, 1, 128, 16, [0], [1100], "ref", "SHD", False),
    (4, 2, 80, 16, [2500, 31], [40, 33], "causal", "SHD", False),
    (4, 2, 96, 32, [0], [1300], "causal", "HSD", True),
    (32, 8, 80, 16, [100] * 4, [600] * 4, "causal", "SHD", False),
    (2, 1, 256, 16, [3001], [40], "causal", "SHD", False),
    (10, 2, 72, 16, [1500], [100], "causal", "SHD", True),
]


@pytest.mark.parametrize("H,KVH,D,P,before,n,mask,layout,f32", GQA)
def test_gqa_parts(gpu, monkeypatch, H, KVH, D, P, before, n, mask, layout, f32):
    from relux_amd import KVCache
    g = torch.Generator(device=gpu).manual_seed(D + sum(before) + H)
    S, dt = len(before), torch.float32 if f32 else torch.bfloat16
    T = [a + b for a, b in zip(before, n)]
    k = torch.randn(sum(T), KVH, D, device=gpu, generator=g).to(torch.bfloat16)
    v = torch.randn(sum(T), KVH, D, device=gpu, generator=g).to(torch.bfloat16)
    q = torch.randn(sum(n), H, D, device=gpu, generator=g).to(dt)
    outs = []
    for whole in (False, True):
        c = KVCache(num_layers=1, max_len=max(T), num_kv_heads=KVH, head_dim=D, page_tokens=P, max_seqs=S,
                    device=gpu.index)
        c.Append(0, k, v, seq_ids=list(range(S)), n_tok=T, layout="SHD")
        if whole:
            monkeypatch.setenv("RLX_WS_MAX_KB", "1")
        qi = q if layout == "SHD" else torch.cat([x.transpose(0, 1).reshape(-1) for x in q.split(n)])
        o = c.Attend(0, qi.contiguous(), H, seq_ids=list(range(S)), n_q=n, mask=mask, layout=layout)
        if layout == "HSD":
            o = torch.cat([x.view(H, m, D).transpose(0, 1) for x, m in
                           zip(o.reshape(-1).split([m * H * D for m in n]), n)])
        outs.append(o.reshape(sum(n), H, D))
        cut = c.MemoryStats()["workspace"] > 0
        assert not (whole and cut)
        if not whole and S == 1:
            assert cut, "the tiles were not cut"
    at = qt = 0
    for i in range(S):
        want = _exact(q[qt:qt + n[i]].float().bfloat16().double() if not f32 else q[qt:qt + n[i]].double(),
                      k[at:at + T[i]].double(), v[at:at + T[i]].double(), n[i], mask, 1.0 / math.sqrt(D))
        for o in outs:
            _check(o[qt:qt + n[i]], want)
        at, qt = at + T[i], qt + n[i]


@pytest.mark.parametrize("H,D,before,n,fa2", [
    (4, 128, [3000], [300], True),         # few heads: cut tiles of the expanded form
    (3, 64, [1000, 0], [270, 257], True),
    (2, 192, [2000], [513], True),         # two launches over halves of V
    (16, 128, [700], [70], False),         # the absorbed kernel past 1024 rows
    (128, 128, [300, 65], [12, 9], False),
])
def test_mla_parts(gpu, monkeypatch, H, D, before, n, fa2):
    from relux_amd import MLACache
    g = torch.Generator(device=gpu).manual_seed(D + sum(before) + H)
    S, bf = len(before), torch.bfloat16
    T = [a + b for a, b in zip(before, n)]
    cl = torch.randn(sum(T), 512, device=gpu, generator=g).to(bf)
    kr = torch.randn(sum(T), 64, device=gpu, generator=g).to(bf)
    w = [(torch.randn(512, H * D, device=gpu, generator=g) * 0.02).to(bf) for _ in range(2)]
    qn, qr = (torch.randn(sum(n), H, d, device=gpu, generator=g) for d in (D, 64))
    c = MLACache(num_layers=1, max_len=max(T), page_tokens=64, max_seqs=S, device=gpu.index)
    c.Append(0, cl, kr, seq_ids=list(range(S)), n_tok=T)
    if fa2:
        monkeypatch.setenv("RLX_MLA_FA2_ROWS", "32")
    o = c.Attend(0, qn, qr, *w, H, D, seq_ids=list(range(S)), n_q=n)
    uk, uv = (x.double().view(512, H, D) for x in w)
    at = qt = 0
    for i in range(S):
        C, R = cl[at:at + T[i]].double(), kr[at:at + T[i]].double()
        K = torch.cat([torch.matmul(C, uk.reshape(512, -1)).view(-1, H, D), R[:, None].expand(-1, H, -1)], 2)
        V = torch.matmul(C, uv.reshape(512, -1)).view(-1, H, D)
        Q = torch.cat([qn, qr], 2)[qt:qt + n[i]].double()
        _check(o[qt:qt + n[i]], _exact(Q, K, V, n[i], "causal", 1.0 / math.sqrt(D + 64)))
        at, qt = at + T[i], qt + n[i]


@pytest.mark.parametrize("D", [80, 96])
@pytest.mark.parametrize("scale", [0.3, 1.0, 3.0])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_hd96_no_less_precise_than_query_tiles(gpu, D, scale, dtype):
    """Stored head dim 96 in the prefill kernel is no further off the 64-bit
    result than as query tiles of the decode kernel (the call that allocates
    nothing takes those)."""
    from relux_amd import KVCache
    H, T, n = 2, 9000, 1800
    g = torch.Generator(device=gpu).manual_seed(D)
    k, v = (torch.randn(T, H, D, device=gpu, generator=g).to(torch.bfloat16) for _ in range(2))
    q = (torch.randn(n, H, D, device=gpu, generator=g) * scale).to(dtype)
    c = KVCache(num_layers=1, max_len=T, num_kv_heads=H, head_dim=D, device=gpu.index)
    c.Append(0, k, v, seq_ids=[0], n_tok=[T], layout="SHD")
    tiles = torch.empty_like(q)
    c.AttendNoAlloc(0, q, H, tiles, seq_ids=[0], n_q=[n], layout="SHD")
    o = c.Attend(0, q, H, seq_ids=[0], n_q=[n], out=torch.empty_like(q))
    assert not torch.equal(o, tiles), "the call took query tiles"
    want = _exact(q.double(), k.double(), v.double(), n, "causal", 1.0 / math.sqrt(D))
    off = [float((x.double() - want).norm()) for x in (o, tiles)]
    assert off[0] <= 1.005 * off[1], off


def _hd96(gpu, H, KVH, D, before, n, dtype):
    from relux_amd import KVCache
    g = torch.Generator(device=gpu).manual_seed(D + H)
    S, T = len(before), [a + b for a, b in zip(before, n)]
    k, v = (torch.randn(sum(T), KVH, D, device=gpu, generator=g).to(torch.bfloat16) for _ in range(2))
    c = KVCache(num_layers=1, max_len=max(T), num_kv_heads=KVH, head_dim=D, max_seqs=S, device=gpu.index)
    c.Append(0, k, v, seq_ids=list(range(S)), n_tok=T, layout="SHD")
    q = torch.randn(sum(n), H, D, device=gpu, generator=g).to(dtype)
    tiles = c.AttendNoAlloc(0, q, H, torch.empty_like(q), seq_ids=list(range(S)), n_q=n)
    return c, q, tiles, dict(seq_ids=list(range(S)), n_q=n)


@pytest.mark.parametrize("H,KVH,D,before,n,fa2", [
    (32, 8, 80, [2000], [100], False),
    (16, 16, 80, [300, 50], [200, 400], False),
    (32, 8, 96, [0], [40], False),
    (8, 2, 72, [8000], [64], False),
    (64, 8, 80, [8000], [128], True),
    (16, 16, 96, [8000], [1000], True),
])
def test_hd96_route(gpu, H, KVH, D, before, n, fa2):
    """Query tiles where they are the faster form, which is most small calls."""
    c, q, tiles, kw = _hd96(gpu, H, KVH, D, before, n, torch.bfloat16)
    assert torch.equal(c.Attend(0, q, H, out=torch.empty_like(q), **kw), tiles) != fa2


def test_hd96_outputs_in_the_queries_memory(gpu):
    """The prefill kernel writes a tile's rows while others still read theirs:
    outputs in the queries' own memory, but not row for row, and outputs off
    their stores' alignment, run as query tiles at any size."""
    H, KVH, D, before, n = 64, 8, 80, [8000], [128]
    c, q, tiles, kw = _hd96(gpu, H, KVH, D, before, n, torch.float32)
    out = torch.empty(q.shape, dtype=torch.bfloat16, device=gpu)
    want = c.AttendNoAlloc(0, q, H, out, **kw).clone()
    m = q.numel()
    buf = q.reshape(-1).clone().view(torch.bfloat16)  # 2 m elements, the queries as f32
    for off in (0, m, 8):
        buf.view(torch.float32).copy_(q.reshape(-1))
        c.Attend(0, buf.view(torch.float32).view(q.shape), H, out=buf[off:off + m].view(q.shape), **kw)
        assert torch.equal(buf[off:off + m].view(q.shape), want), off
    odd = torch.empty(m + 1, dtype=torch.bfloat16, device=gpu)[1:].view(q.shape)
    assert torch.equal(c.Attend(0, q, H, out=odd, **kw), want)
    same = q.clone()  # row for row: as with separate outputs
    assert torch.equal(c.Attend(0, same, H, out=same, **kw), c.Attend(0, q, H, **kw))
    assert not torch.equal(same, tiles), "the call took query tiles"


def test_mla_prefill_weights_off_alignment(gpu):
    """W_UK and W_UV that start at any element: the expansion packs them by
    elements, with the same result."""
    from relux_amd import MLACache
    H, D, T, n = 3, 64, 500, 400
    g = torch.Generator(device=gpu).manual_seed(2)
    w = [(torch.randn(512, H * D, device=gpu, generator=g) * 0.02).to(torch.bfloat16) for _ in range(2)]
    odd = []
    for off, x in zip((1, 3), w):
        buf = torch.empty(x.numel() + 8, dtype=torch.bfloat16, device=gpu)
        odd.append(buf[off:off + x.numel()].view(x.shape).copy_(x))
    c = MLACache(num_layers=1, max_len=T, page_tokens=64, device=gpu.index)
    c.Append(0, torch.randn(T, 512, device=gpu, generator=g), torch.randn(T, 64, device=gpu, generator=g),
             seq_ids=[0], n_tok=[T])
    qn, qr = (torch.randn(n, H, d, device=gpu, generator=g) for d in (D, 64))
    want = c.Attend(0, qn, qr, *w, H, D, seq_ids=[0], n_q=[n])
    assert torch.equal(c.Attend(0, qn, qr, *odd, H, D, seq_ids=[0], n_q=[n]), want)
