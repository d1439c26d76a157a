"""The workspace of a handle under graphs and reservations: scratch that a
captured call holds outlives every later growth, a captured call that can do
without scratch holds none, and a reserved handle does not grow for a call
that can do without."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SLACK = 8 << 20  # allocations of the runtime's own


def _used():
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


class _Sample:
    """A SampleAsync call whose scratch is 16 MiB and more."""

    def __init__(self, gpu, **kw):
        from relux_amd import Sampler
        g = torch.Generator(device=gpu).manual_seed(3)
        self.x = torch.randn(600, 65000, device=gpu, generator=g) * 4
        self.g, self.u = g, torch.rand(600, device=gpu, generator=g)
        self.out = torch.zeros(600, dtype=torch.int32, device=gpu)
        self.s = Sampler(**kw)

    def refresh(self):
        self.u.copy_(torch.rand(600, device=self.u.device, generator=self.g))

    def __call__(self, c, out=None):
        return self.s.SampleAsync(self.x, None, None, self.u, c, out=self.out if out is None else out)


def _handle(gpu, **kw):
    from relux_amd import KVCache
    return KVCache(**dict(dict(num_layers=1, max_len=16, num_kv_heads=1, head_dim=64, device=gpu.index), **kw))


def _grow(c, gpu):
    """An eager call that needs more scratch than any other here."""
    from relux_amd import Sampler
    x, u = torch.randn(3000, 65000, device=gpu), torch.rand(3000, device=gpu)
    out = torch.zeros(3000, dtype=torch.int32, device=gpu)
    before = _used()
    Sampler(top_k=256).SampleAsync(x, None, None, u, c, out=out)
    return _used() - before


# top-k: its chunk lists are scratch the call needs, so the graph holds them;
# top-p alone: the captured call runs the whole rows, whatever is there
@pytest.mark.parametrize("kw,holds", [(dict(top_k=256), True), (dict(top_p=0.9), False)])
def test_scratch_of_a_captured_call(gpu, kw, holds):
    call, c, other = _Sample(gpu, temperature=0.8, **kw), _handle(gpu), _handle(gpu)
    call(c)  # the workspace is there
    old = c.MemoryStats()["workspace"]
    assert old >= 2 * SLACK
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    c.use_stream(stream)
    with torch.cuda.graph(graph, stream=stream):
        call(c)
    stream.synchronize()
    got = _grow(c, gpu)
    new = c.MemoryStats()["workspace"]
    assert new >= 2 * old
    kept = got - (new - old)  # the outgrown buffer, if it is still there
    assert abs(kept - (old if holds else 0)) <= SLACK, (kept, old)
    for _ in range(3):
        call.refresh()
        want = call(other, out=torch.zeros_like(call.out)).cpu()
        torch.cuda.synchronize()
        graph.replay()
        _grow(c, gpu)
        torch.cuda.synchronize()
        same = (call.out.cpu() == want).sum().item()
        # (whole rows and their split sum in different orders: a draw within
        # rounding of a token's boundary may take its neighbour)
        assert same == 600 if holds else same >= 590, same
    del graph
    before = _used()
    c.close()
    assert before - _used() >= new - SLACK


def test_reserved_handle_does_not_grow_for_optional_scratch(gpu):
    """A trial run of the largest call gives the sizes to reserve, and no call
    of those sizes allocates after: a prefill that fills the chip takes no
    scratch, and a smaller one then takes none either."""
    g = torch.Generator(device=gpu).manual_seed(5)
    H, KVH, D, T = 32, 8, 128, 4096
    k, v = (torch.randn(T, KVH, D, device=gpu, generator=g).bfloat16() for _ in range(2))
    q = torch.randn(T, H, D, device=gpu, generator=g).bfloat16()

    def prefill(c, n):  # the last n of T tokens
        c.Append(0, k, v, seq_ids=[0], n_tok=[T], layout="SHD")
        o = c.Attend(0, q[:n].contiguous(), H, seq_ids=[0], n_q=[n])
        c.Rollback([0], [T])
        return o

    trial, served, free = (_handle(gpu, max_len=T, num_kv_heads=KVH, head_dim=D) for _ in range(3))
    prefill(trial, T)
    st = trial.MemoryStats()
    served.Reserve(st["workspace_peak"], st["staging_peak"], st["adapter_peak"])
    before = served.MemoryStats()
    got, want = prefill(served, 200), prefill(free, 200)
    prefill(served, T)
    assert free.MemoryStats()["workspace"] > 0, "the smaller call has no optional scratch: choose another"
    after = served.MemoryStats()
    assert after["workspace"] == before["workspace"] and after["staging"] == before["staging"]
    assert after["workspace_peak"] == free.MemoryStats()["workspace_peak"]  # what to reserve for it
    e = (got.double() - want.double()).abs()
    assert float(e.max()) <= 1e-2 and float(e.mean()) <= 1e-3
