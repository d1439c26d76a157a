"""MLA decode and verify with head groups: plans of at most 64 rows travel in
the kernel arguments, larger ones staged.  Against exact softmax attention in
f64 over the rounded cache rows (max-abs 1e-2, mean-abs 1e-3, the bars of the
other attention tests)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


# H x queries over the 16 or 32 rows of a group: 1 to 8 groups a sequence,
# groups that do not fill their last, mixed query counts (one sequence with a
# single group), splits that are no multiple of 8 (ragged lengths); 16
# sequences of 4 groups (the last plan in the arguments) and 17 (staged)
@pytest.mark.parametrize("H,before,n", [
    (128, [1], [1]),
    (128, [5000, 37, 2500], [1, 1, 1]),
    (40, [3000, 900], [1, 1]),
    (16, [4000, 600, 2111], [1, 5, 3]),
    (20, [777, 64, 1500], [4, 1, 2]),
    (64, [2000], [4]),
    (128, [100 + 7 * i for i in range(16)], [1] * 16),
    (128, [100 + 7 * i for i in range(17)], [1] * 17),
])
def test_mla_head_groups(gpu, H, before, n):
    from relux_amd import MLACache
    D, S, bf = 128, len(before), torch.bfloat16
    g = torch.Generator(device=gpu).manual_seed(H + sum(before))
    T = [a + b for a, b in zip(before, n)]
    cl = torch.randn(sum(T), 512, device=gpu, generator=g).to(bf)
    kr = torch.randn(sum(T), 64, device=gpu, generator=g).to(bf)
    w = [(torch.randn(512, H * D, device=gpu, generator=g) * 0.02).to(bf) for _ in range(2)]
    qn, qr = (torch.randn(sum(n), H, d, device=gpu, generator=g) for d in (D, 64))
    c = MLACache(num_layers=1, max_len=max(T), page_tokens=64, max_seqs=S, device=gpu.index)
    c.Append(0, cl, kr, seq_ids=list(range(S)), n_tok=T)
    o = c.Attend(0, qn, qr, *w, H, D, seq_ids=list(range(S)), n_q=n)
    uk, uv = (x.double().view(512, H, D).permute(1, 0, 2).contiguous() for x in w)
    at = qt = 0
    for i in range(S):
        C, R = cl[at:at + T[i]].double(), kr[at:at + T[i]].double()
        hidden = torch.arange(T[i], device=gpu)[None, :] > torch.arange(before[i], T[i], device=gpu)[:, None]
        for h in range(H):
            k = torch.cat([torch.matmul(C, uk[h]), R], 1)
            q = torch.cat([qn[qt:qt + n[i], h], qr[qt:qt + n[i], h]], 1).double()
            s = torch.matmul(q, k.t().contiguous()) / math.sqrt(D + 64)
            want = torch.matmul(torch.softmax(s.masked_fill(hidden, -math.inf), -1), torch.matmul(C, uv[h]))
            e = (o[qt:qt + n[i], h].double() - want).abs()
            assert float(e.max()) <= 1e-2 and float(e.mean()) <= 1e-3, (i, h, float(e.max()), float(e.mean()))
        at, qt = at + T[i], qt + n[i]


@pytest.mark.parametrize("H,before,n", [
    (128, [8144], [48]),                  # one split a row for most rows
    (128, [1000 + 300 * i for i in range(8)], [9] * 8),
    (16, [600, 100], [65, 70]),           # several splits a row, ragged
])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_absorbed_prefill_no_less_precise(gpu, monkeypatch, H, before, n, dtype):
    """Calls past 1024 query rows that run the absorbed kernel: no further off
    the 64-bit result than the expanded form, whose sums are all f32."""
    from relux_amd import MLACache
    D, S, bf = 128, len(before), torch.bfloat16
    dt = torch.float32 if dtype == "f32" else bf
    g = torch.Generator(device=gpu).manual_seed(H + sum(before))
    T = [a + b for a, b in zip(before, n)]
    cl = torch.randn(sum(T), 512, device=gpu, generator=g).to(bf)
    kr = torch.randn(sum(T), 64, device=gpu, generator=g).to(bf)
    w = [(torch.randn(512, H * D, device=gpu, generator=g) * 0.02).to(bf) for _ in range(2)]
    qn, qr = (torch.randn(sum(n), H, d, device=gpu, generator=g).to(dt) for d in (D, 64))
    c = MLACache(num_layers=1, max_len=max(T), page_tokens=64, max_seqs=S, device=gpu.index)
    c.Append(0, cl, kr, seq_ids=list(range(S)), n_tok=T)
    outs = [c.Attend(0, qn, qr, *w, H, D, seq_ids=list(range(S)), n_q=n).double()]
    for rows in ("1000000", "32"):
        monkeypatch.setenv("RLX_MLA_FA2_ROWS", rows)
        outs.append(c.Attend(0, qn, qr, *w, H, D, seq_ids=list(range(S)), n_q=n).double())
    assert torch.equal(outs[0], outs[1]), "the call did not take the absorbed kernel"
    uk, uv = (x.double().view(512, H, D) for x in w)
    off = [0.0, 0.0]
    at = qt = 0
    for i in range(S):
        C, R = cl[at:at + T[i]].double(), kr[at:at + T[i]].double()
        hidden = torch.arange(T[i], device=gpu)[None, :] > torch.arange(before[i], T[i], device=gpu)[:, None]
        for h in range(0, H, H // 8):
            k = torch.cat([torch.matmul(C, uk[:, h].contiguous()), R], 1)
            q = torch.cat([qn[qt:qt + n[i], h], qr[qt:qt + n[i], h]], 1).double()
            s = torch.matmul(q, k.t().contiguous()) / math.sqrt(D + 64)
            p = torch.softmax(s.masked_fill(hidden, -math.inf), -1)
            want = torch.matmul(p, torch.matmul(C, uv[:, h].contiguous()))
            for j, o in enumerate((outs[0], outs[2])):
                off[j] += float((o[qt:qt + n[i], h] - want).pow(2).sum())
        at, qt = at + T[i], qt + n[i]
    assert off[0] <= off[1], off
