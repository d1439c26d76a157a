"""GQA decode calls whose rows each lie in one range: the decode kernel writes
the outputs itself.  Checked against a float64 attention, and bit for bit
against the same call with the outputs in the query's own memory, which is
merged from partials."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

U = 2.0 ** -8  # bf16 unit roundoff: of the probabilities and of a bf16 output


@pytest.mark.parametrize("H,KVH,D,lens,nq", [
    (32, 8, 128, [1], 1),
    (32, 8, 128, [768], 1),               # the longest whole row of 128 dims
    (32, 8, 128, [769], 1),               # cut: merged on both sides
    (32, 8, 128, [512, 64, 65, 3], 5),    # two query tiles a group: the longest whole row
    (32, 8, 128, [500] * 31 + [9] * 17, 1),  # several rows a work-group, the most that keep their ranges
    (32, 8, 128, [70] * 49, 1),           # more rows than the kernel arguments take with their ranges
    (64, 8, 128, [300, 768], 5),          # a row's queries in two tiles
    (16, 16, 64, [1536, 1], 1),
    (16, 4, 80, [1000], 2),               # stored as 96 dims
    (8, 2, 16, [130], 1),
    (4, 4, 24, [90, 64], 3),              # stored as 32 dims
    (8, 2, 256, [384, 100], 2),
])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("layout", ["SHD", "HSD"])
def test_direct_outputs(gpu, H, KVH, D, lens, nq, dtype, layout):
    from relux_amd import KVCache
    g = torch.Generator().manual_seed(D + len(lens) + nq)
    S, dt = len(lens), torch.bfloat16 if dtype == "bf16" else torch.float32
    n_q = [min(nq, t) for t in lens]
    c = KVCache(num_layers=1, max_len=max(lens), num_kv_heads=KVH, head_dim=D, page_tokens=16, max_seqs=S,
                device=gpu.index)
    k, v = (torch.randn(sum(lens), KVH, D, generator=g).to(torch.bfloat16) for _ in range(2))
    c.Append(0, k.to(gpu), v.to(gpu), seq_ids=range(S), n_tok=lens, layout="SHD")
    q = torch.randn(sum(n_q), H, D, generator=g).to(torch.bfloat16)
    per = [t.transpose(0, 1).reshape(-1) if layout == "HSD" else t.reshape(-1) for t in q.split(n_q)]
    qd = torch.cat(per).view(-1, H, D).to(dt).to(gpu)
    kw = dict(seq_ids=range(S), n_q=n_q, layout=layout)
    got = c.Attend(0, qd, H, out=torch.full_like(qd, 7.0), **kw)
    odd = torch.full((qd.numel() + 1,), 7.0, dtype=dt, device=gpu)[1:].view(qd.shape)  # no wide stores
    c.Attend(0, qd, H, out=odd, **kw)
    merged = qd.clone()
    c.Attend(0, merged, H, out=merged, **kw)
    assert torch.equal(got, odd) and torch.equal(got, merged)
    if H // KVH * nq <= 32:  # what the call without allocation takes
        c.AttendNoAlloc(0, qd, H, odd.zero_(), **kw)
        assert torch.equal(got, odd)
    res = got.double().cpu()
    kr, qr, off = 0, 0, 0
    for t, n in zip(lens, n_q):
        kk, vv = (x[kr:kr + t].double().repeat_interleave(H // KVH, 1).transpose(0, 1).contiguous() for x in (k, v))
        s = (q[qr:qr + n].double().transpose(0, 1) @ kk.transpose(1, 2).contiguous()) / math.sqrt(D)
        s.masked_fill_(torch.arange(t) > (t - n + torch.arange(n))[:, None], -math.inf)
        p = torch.softmax(s, -1)
        want, bound = p @ vv, p @ vv.abs()
        r = res.view(-1)[off:off + n * H * D]
        r = r.view(H, n, D) if layout == "HSD" else r.view(n, H, D).transpose(0, 1)
        # a probability and the output rounded to bf16; scores in float32 to 2^-12 of the sum
        assert ((r - want).abs() <= (2 * U + 2.0 ** -10) * bound + 1e-6).all()
        kr, qr, off = kr + t, qr + n, off + n * H * D


@pytest.mark.parametrize("lens,ranges", [
    ([200, 40, 130, 90, 65, 10, 190, 25] * 3, 24),  # a range each: 32 are there
    ([500], 1),
    ([750], 1),
    ([800], 13),                                    # cut: longer than 12 units
    ([750] * 31, 31),                               # an even share is a row
    ([60] * 40, 20),                                # more rows than ranges: even in rows
])
def test_ranges_of_short_rows(gpu, lens, ranges):
    """Rows share a work-group only where there are more rows than ranges (32
    at 8 kv heads on 256 CUs), and a row is cut where that is the faster form.
    The call's scratch request tells its ranges: a partial a row and a range."""
    from relux_amd import KVCache
    H, KVH, D, S = 32, 8, 128, len(lens)
    if torch.cuda.get_device_properties(gpu).multi_processor_count != 256:
        pytest.skip("the counts are of 256 CUs")
    c = KVCache(num_layers=1, max_len=max(lens), num_kv_heads=KVH, head_dim=D, max_seqs=S, device=gpu.index)
    k = torch.randn(sum(lens), KVH, D, device=gpu)
    c.Append(0, k, k, seq_ids=range(S), n_tok=lens, layout="SHD")
    c.Attend(0, torch.randn(S, H, D, device=gpu), H, seq_ids=range(S))
    parts = c.MemoryStats()["workspace_peak"] / (KVH * 16 * (D * 4 + 8))
    assert parts == S + ranges, parts
