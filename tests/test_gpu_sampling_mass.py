"""Sample without top-k over vocabulary chunks (past 12288 entries, without
top-p past 18432) against the whole-row path, which a handle whose workspace
may not grow takes; past 32768 entries that path searches the top-p cutoff by
bisection over f32 sums.

Bar: the same token ids on every row whose whole-row answer is unchanged with
the draw moved by +-1e-5 (the two paths sum in different orders)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DELTA = 1e-5


@pytest.fixture
def handles(gpu):
    from relux_amd import KVCache
    return [KVCache(num_layers=1, max_len=16, num_kv_heads=1, head_dim=64, device=gpu.index) for _ in range(2)]


def _compare(handles, monkeypatch, x, u, least, hist=None, **kw):
    from relux_amd import Sampler
    s = Sampler(**kw)
    n = torch.full((x.shape[0],), hist.shape[1], dtype=torch.int32, device=x.device) if hist is not None else None
    got = s.SampleAsync(x, hist, n, u, handles[0]).cpu().numpy()
    V, topp = x.shape[1], 0.0 < kw.get("top_p", 0.0) < 1.0
    # (from 12289 on the whole row ends with 6 or 7 entries a thread one by one)
    split = V > (12288 if topp or V // 512 % 8 >= 6 else 18432)
    if V <= 262144:
        assert (handles[0].MemoryStats()["workspace"] > 1 << 16) == split
    monkeypatch.setenv("RLX_WS_MAX_KB", "4")
    ref = [s.SampleAsync(x, hist, n, (u + d).clamp(0, 0.9999999), handles[1]).cpu().numpy()
           for d in (-DELTA, 0.0, DELTA)]
    assert handles[1].MemoryStats()["workspace"] <= 1 << 16  # the whole-row path ran
    monkeypatch.delenv("RLX_WS_MAX_KB")
    ok = (ref[0] == ref[1]) & (ref[1] == ref[2])
    np.testing.assert_array_equal(got[ok], ref[1][ok])
    assert ok.sum() >= least, int(ok.sum())


PARAMS = [dict(), dict(temperature=0.7, top_p=0.9), dict(top_p=0.3), dict(top_p=0.999999), dict(min_p=0.05),
          dict(temperature=0.8, top_p=0.95, min_p=0.02), dict(top_p=0.9, min_p=0.5), dict(min_p=1.5),
          dict(temperature=0.0, top_p=0.9), dict(temperature=25.0, top_p=0.9),
          dict(top_p=0.9, repeat_penalty=1.3, frequency_penalty=0.2, presence_penalty=0.3, repeat_window=100)]


# 12289: the smallest split; 15400, 18433: the smallest ones without top-p;
# 16387, 50257: rows off 16-byte alignment; 32768 /
# 32772: the last LDS row and the first memory row of the whole-row path;
# 262144: the largest split
@pytest.mark.parametrize("V", [12289, 15400, 16387, 18433, 32768, 32772, 50257, 262144])
@pytest.mark.parametrize("k", range(len(PARAMS)))
def test_split_equals_whole_row(gpu, handles, monkeypatch, V, k):
    g = torch.Generator(device=gpu).manual_seed(1000 * k + V)
    B = 12
    x = torch.randn(B, V, device=gpu, generator=g) * torch.linspace(0.5, 8.0, B, device=gpu)[:, None]
    u = torch.rand(B, device=gpu, generator=g)
    hist = torch.randint(0, V, (B, 128), device=gpu, generator=g, dtype=torch.int32)
    # (at temperature 25 the rows are nearly uniform: token boundaries are 1 / V
    # apart, within the draws' shift for most of them)
    _compare(handles, monkeypatch, x, u, 0 if PARAMS[k].get("temperature") == 25.0 else B // 3, hist=hist, **PARAMS[k])


@pytest.mark.parametrize("kw", [dict(top_p=0.9), dict(top_p=0.9, min_p=0.1), dict()])
@pytest.mark.parametrize("V", [20001, 40000])
def test_split_odd_rows(gpu, handles, monkeypatch, V, kw):
    """Rows that leave the buckets or their lists: constant and nearly
    constant rows, masks, infinities, NaN, a cutoff among tied weights."""
    g = torch.Generator(device=gpu).manual_seed(V)
    x = torch.randn(12, V, device=gpu, generator=g) * 3
    lowest = torch.finfo(torch.float32).min
    x[0] = 1.0                              # one weight: more entries than a list holds
    x[1] = 1.0 + 1e-3 * x[1]                # one bucket or two
    x[2] = float("-inf")
    x[3] = float("-inf")
    x[3, 7777] = 2.0
    x[4, ::2] = lowest
    x[5] = lowest
    x[6, 5] = float("inf")                  # every other weight 0
    x[7, ::3] = float("nan")
    x[8] = float("nan")
    x[9] = torch.round(x[9])                # thousands tied on every weight
    x[10] = -60.0                           # most of the mass below the buckets
    x[10, 100] = 0.0
    x[11] = -25.0 + 0.01 * x[11]            # half of it
    x[11, 100] = float(np.log(V)) - 25.0
    u = torch.rand(12, device=gpu, generator=g)
    u[2], u[3] = 0.5, 0.0
    _compare(handles, monkeypatch, x, u, 6, **kw)


def test_split_rows_past_the_scratch(gpu, handles, monkeypatch):
    """More rows than the scratch holds at a time."""
    g = torch.Generator(device=gpu).manual_seed(5)
    B, V = 90, 200001
    x = torch.randn(B, V, device=gpu, generator=g) * 4
    u = torch.rand(B, device=gpu, generator=g)
    hist = torch.randint(0, V, (B, 64), device=gpu, generator=g, dtype=torch.int32)
    _compare(handles, monkeypatch, x, u, B // 2, hist=hist, temperature=0.8, top_p=0.9, repeat_penalty=1.2)


@pytest.mark.parametrize("grown", [False, True])
def test_split_under_capture(gpu, grown):
    """A captured call allocates nothing and holds no scratch: the whole-row
    path, whether the split's workspace is there or not; replays follow their
    draws."""
    from relux_amd import KVCache, Sampler
    g = torch.Generator(device=gpu).manual_seed(9)
    B, V = 4, 40000
    x = torch.randn(B, V, device=gpu, generator=g) * 6
    u = torch.rand(B, device=gpu, generator=g)
    out = torch.zeros(B, dtype=torch.int32, device=gpu)
    s = Sampler(temperature=0.8, top_p=0.9)
    c = KVCache(num_layers=1, max_len=16, num_kv_heads=1, head_dim=64, device=gpu.index)
    if grown:
        s.SampleAsync(x, None, None, u, c, out=out)
    before = c.MemoryStats()["workspace"]
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    c.use_stream(stream)
    with torch.cuda.graph(graph, stream=stream):
        s.SampleAsync(x, None, None, u, c, out=out)
    assert c.MemoryStats()["workspace"] == before
    eager = KVCache(num_layers=1, max_len=16, num_kv_heads=1, head_dim=64, device=gpu.index)
    for _ in range(4):
        u.copy_(torch.rand(B, device=gpu, generator=g))
        want = s.SampleAsync(x, None, None, u, eager).cpu()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.cpu(), want)
