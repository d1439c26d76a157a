"""The prefill-size projection GEMM (calls of more than 64 rows, of more than
80 with f32 activations, and from fewer whose features are more than one round
of the CUs: proj_use_gemm) against the decode-size kernels: the same rows
through calls of at most 32 rows.

Both take the same bf16 products (f32 activations as hi + lo pairs) and
differ in the order of the f32 sums: |difference| <= 2^-17 S per output, S =
sum |x||w| (the sums' bound is K 2^-24 S, K <= 512 here; RoPE adds two such
terms), and one bf16 step where the value is stored in bf16."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _weights(g, gpu, *shapes):
    return [(torch.randn(s, generator=g) * 0.02).to(torch.bfloat16).to(gpu) for s in shapes]


def _close(a, b, K, stored_bf16):
    a, b = a.float(), b.float()
    S = K * 4.0 * 0.08  # |x| < 4, |w| < 0.08 (4 sigma): an upper bound of S
    tol = 2.0 * S * 2.0 ** -17 + (b.abs() * 2.0 ** -7 if stored_bf16 else 0.0)
    assert bool(((a - b).abs() <= tol).all()), float((a - b).abs().max())


def _pieces(ntok, most=32):
    """ntok tokens of each sequence as calls of at most `most` rows: [(seq, first, n)]."""
    out = []
    for i, n in enumerate(ntok):
        out += [(i, j, min(most, n - j)) for j in range(0, n, most)]
    return out


# (d_model, H, KVH, D, cached, new, x dtype, q dtype): tile edges (64, 128
# rows and their neighbours), a last k-step of 32, heads narrower than a
# fragment (D 2, 4), padded heads (20, 36 features), head dims stored padded
# (80 in 96, 24 in 32), dims that are not a multiple of 4 (6, 50)
GQA = [
    (512, 8, 2, 64, [0, 40], [65, 0], torch.bfloat16, torch.bfloat16),
    (256, 8, 2, 128, [3, 0, 17], [100, 1, 28], torch.float32, torch.float32),
    (96, 4, 4, 32, [0], [127], torch.bfloat16, torch.float32),
    (512, 8, 4, 80, [5], [130], torch.float32, torch.bfloat16),
    (32, 8, 8, 2, [0, 9], [60, 70], torch.bfloat16, torch.float32),
    (64, 4, 4, 4, [1], [257], torch.float32, torch.float32),
    (96, 3, 1, 20, [0], [66], torch.bfloat16, torch.bfloat16),
    (160, 8, 8, 6, [2], [90], torch.bfloat16, torch.bfloat16),
    (64, 2, 2, 50, [11], [129], torch.float32, torch.bfloat16),
    (64, 6, 2, 24, [0, 0], [64, 64], torch.bfloat16, torch.bfloat16),
    # more 16-feature tiles than CUs: the GEMM from 37 rows
    (128, 259, 1, 16, [4], [33], torch.bfloat16, torch.bfloat16),
    (128, 259, 1, 16, [4], [37], torch.bfloat16, torch.bfloat16),
    # one round of tiles of a d_model of at most 1024 in bf16: the GEMM from 97 rows
    (512, 8, 2, 64, [0, 40], [97, 0], torch.bfloat16, torch.bfloat16),
    (96, 3, 1, 20, [0], [98], torch.bfloat16, torch.bfloat16),
    (160, 8, 8, 6, [2], [122], torch.bfloat16, torch.bfloat16),
]


@pytest.mark.parametrize("d_model,H,KVH,D,lens,ntok,x_dtype,q_dtype", GQA)
def test_gqa_gemm_equals_small_calls(gpu, d_model, H, KVH, D, lens, ntok, x_dtype, q_dtype):
    from relux_amd import KVCache, pack_qkv, rope_tables
    g = torch.Generator().manual_seed(d_model + D)
    wp = pack_qkv(*_weights(g, gpu, (d_model, H * D), (d_model, KVH * D), (d_model, KVH * D)), H, KVH, D)
    S, rope = len(lens), rope_tables(D, 10000.0, 512, gpu)
    x = torch.randn(sum(ntok), d_model, generator=g).clamp(-4, 4).to(gpu).to(x_dtype)
    caches = []
    for _ in range(2):
        c = KVCache(num_layers=1, max_len=512, num_kv_heads=KVH, head_dim=D, max_seqs=S, device=gpu.index)
        for i, n in enumerate(lens):
            if n:
                kv = torch.ones(n, KVH, D, device=gpu)
                c.Append(0, kv, kv, seq_ids=[i], n_tok=[n], layout="SHD")
        caches.append(c)
    q = caches[0].ProjectAppend(0, x, wp, H, rope=rope, seq_ids=list(range(S)), n_tok=ntok, q_dtype=q_dtype)
    at = np.concatenate([[0], np.cumsum(ntok)])
    for i, j, n in _pieces(ntok):
        r = int(at[i]) + j
        qp = caches[1].ProjectAppend(0, x[r:r + n].contiguous(), wp, H, rope=rope, seq_ids=[i], n_tok=[n],
                                     q_dtype=q_dtype)
        _close(q[r:r + n], qp, d_model, q_dtype == torch.bfloat16)
    for i in range(S):
        for a, b in zip(caches[0].View(0, i), caches[1].View(0, i)):
            assert (a is None) == (b is None)
            if a is not None:
                assert torch.equal(a[:, :, :lens[i]], b[:, :, :lens[i]])
                _close(a, b, d_model, True)


@pytest.mark.parametrize("d_model,H,D,dC,dR,lens,ntok,x_dtype", [
    (256, 16, 128, 512, 64, [0, 30], [64, 65], torch.bfloat16),
    (96, 2, 32, 130, 10, [7], [129], torch.float32),   # latent and rope widths not multiples of 4
    (64, 2, 4, 16, 2, [0], [70], torch.bfloat16),      # heads narrower than a fragment
    (64, 5, 6, 16, 8, [0], [70], torch.bfloat16),      # q_c heads packed padded, 6 dims stored
    (64, 2, 4, 16, 2, [0], [102], torch.bfloat16),     # the same in the GEMM
    (64, 5, 6, 16, 8, [0], [102], torch.bfloat16),
])
def test_mla_gemm_equals_small_calls(gpu, d_model, H, D, dC, dR, lens, ntok, x_dtype):
    from relux_amd import MLACache, pack_mla_proj, rope_tables
    g = torch.Generator().manual_seed(d_model + dC)
    wp = pack_mla_proj(*_weights(g, gpu, (d_model, H * D), (d_model, H * dR), (d_model, dC), (d_model, dR)), H, D)
    S, rope = len(lens), rope_tables(dR, 10000.0, 512, gpu)
    x = torch.randn(sum(ntok), d_model, generator=g).clamp(-4, 4).to(gpu).to(x_dtype)
    caches = []
    for _ in range(2):
        c = MLACache(num_layers=1, max_len=512, d_c=dC, d_r=dR, page_tokens=16, max_seqs=S, device=gpu.index)
        for i, n in enumerate(lens):
            if n:
                c.Append(0, torch.ones(n, dC, device=gpu), torch.ones(n, dR, device=gpu), seq_ids=[i], n_tok=[n])
        caches.append(c)
    qs = caches[0].ProjectAppend(0, x, wp, H, D, rope=rope, seq_ids=list(range(S)), n_tok=ntok)
    at = np.concatenate([[0], np.cumsum(ntok)])
    for i, j, n in _pieces(ntok):
        r = int(at[i]) + j
        qp = caches[1].ProjectAppend(0, x[r:r + n].contiguous(), wp, H, D, rope=rope, seq_ids=[i], n_tok=[n])
        for a, b in zip(qs, qp):
            _close(a[r:r + n], b, d_model, False)
    for i in range(S):
        for a, b in zip(caches[0].View(0, i), caches[1].View(0, i)):
            _close(a, b, d_model, True)


@pytest.mark.parametrize("rows,k_in,n_out,x_dtype,out_dtype,resid,off", [
    (65, 512, 256, torch.bfloat16, torch.bfloat16, True, 0),
    (129, 96, 100, torch.float32, torch.float32, True, 0),
    (200, 64, 37, torch.bfloat16, torch.float32, False, 0),  # rows not a multiple of 4 elements
    (70, 32, 64, torch.bfloat16, torch.bfloat16, True, 1),   # out and residual 2 bytes off alignment
    (33, 64, 4112, torch.float32, torch.bfloat16, False, 0),
    (49, 64, 4112, torch.float32, torch.bfloat16, False, 0),  # 257 tiles: the GEMM from 49 rows
])
def test_out_gemm_equals_small_calls(gpu, rows, k_in, n_out, x_dtype, out_dtype, resid, off):
    from relux_amd import KVCache, pack_out
    g = torch.Generator().manual_seed(rows + n_out)
    w, = _weights(g, gpu, (k_in, n_out))
    wp = pack_out(w)
    c = KVCache(num_layers=1, max_len=16, num_kv_heads=1, head_dim=64, device=gpu.index)
    x = torch.randn(rows, k_in, generator=g).clamp(-4, 4).to(gpu).to(x_dtype)

    def rows_at(t):  # a contiguous tensor that starts `off` elements past an allocation
        buf = torch.empty(t.numel() + off, dtype=out_dtype, device=gpu)
        v = buf[off:].view(t.shape)
        v.copy_(t)
        return v
    res = rows_at(torch.randn(rows, n_out, generator=g).to(gpu)) if resid else None
    out = rows_at(torch.zeros(rows, n_out, device=gpu))
    c.OutProject(x, wp, n_out, residual=res, out=out)
    for r in range(0, rows, 32):
        n = min(32, rows - r)
        part = c.OutProject(x[r:r + n].contiguous(), wp, n_out,
                            residual=res[r:r + n].contiguous() if resid else None, out_dtype=out_dtype)
        _close(out[r:r + n], part, k_in, out_dtype == torch.bfloat16)


@pytest.mark.parametrize("H,KVH,rows,x_dtype,gemm", [
    (32, 8, 36, torch.bfloat16, False), (32, 8, 37, torch.bfloat16, True),  # two rounds of the CUs
    (32, 8, 48, torch.float32, False), (32, 8, 49, torch.float32, True),
    (64, 8, 32, torch.bfloat16, False), (64, 8, 33, torch.float32, True),   # three
    (8, 2, 64, torch.bfloat16, False), (8, 2, 65, torch.bfloat16, True),    # one
    (8, 2, 80, torch.float32, False), (8, 2, 81, torch.float32, True),
])
def test_rows_from_which_the_gemm_is_taken(gpu, H, KVH, rows, x_dtype, gemm):
    """The GEMM only where it shortens the pass (sums in another order tell it
    from the decode-size kernels, which a stream under capture takes)."""
    from relux_amd import KVCache, pack_qkv, rope_tables
    if torch.cuda.get_device_properties(gpu).multi_processor_count != 256:
        pytest.skip("the bounds are of 256 CUs")
    D, dm = 128, 4096
    g = torch.Generator().manual_seed(H + rows)
    wp = pack_qkv(*_weights(g, gpu, (dm, H * D), (dm, KVH * D), (dm, KVH * D)), H, KVH, D)
    rope = rope_tables(D, 10000.0, 128, gpu)
    x = torch.randn(rows, dm, generator=g).to(gpu).to(x_dtype)

    def step(c):
        return c.ProjectAppend(0, x, wp, H, rope=rope, seq_ids=[0], n_tok=[rows], q_dtype=torch.float32)
    caches = [KVCache(num_layers=1, max_len=128, num_kv_heads=KVH, head_dim=D, device=gpu.index) for _ in range(2)]
    q = step(caches[0])
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    caches[1].use_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        small = step(caches[1])
    graph.replay()
    torch.cuda.synchronize()
    _close(q, small, dm, False)
    assert torch.equal(q, small) != gemm


@pytest.mark.parametrize("rows,k_in,n_out,x_dtype,gemm", [
    (72, 4096, 4096, torch.float32, False), (81, 4096, 4096, torch.float32, True),
    (72, 640, 4096, torch.float32, True), (65, 4096, 4096, torch.bfloat16, True),
])
def test_out_rows_from_which_the_gemm_is_taken(gpu, rows, k_in, n_out, x_dtype, gemm):
    from relux_amd import KVCache, pack_out
    if torch.cuda.get_device_properties(gpu).multi_processor_count != 256:
        pytest.skip("the bounds are of 256 CUs")
    g = torch.Generator().manual_seed(rows + n_out)
    w, = _weights(g, gpu, (k_in, n_out))
    wp = pack_out(w)
    c = KVCache(num_layers=1, max_len=16, num_kv_heads=1, head_dim=64, device=gpu.index)
    x = torch.randn(rows, k_in, generator=g).to(gpu).to(x_dtype)
    y = c.OutProject(x, wp, n_out, out_dtype=torch.float32)
    first = c.OutProject(x[:64].contiguous(), wp, n_out, out_dtype=torch.float32)
    assert torch.equal(y[:64], first) != gemm


# every tile shape the cost table may pick, at sizes past a turn of the unrolled
# loop (12 k-steps of 64) and of the register rings, with a last half k-step
# (800, 1568), chains of 4, 8 and 12 steps, and more than 16 row tiles whose
# last group is partial (2100 rows: 33 tiles of 64, 17 of 128)
@pytest.mark.parametrize("shape", [0, 1, 2])
@pytest.mark.parametrize("rows,k_in,n_out,x_dtype,out_dtype", [
    (200, 800, 300, torch.bfloat16, torch.float32),
    (131, 1568, 256, torch.float32, torch.float32),
    (2100, 4096, 520, torch.bfloat16, torch.bfloat16),
    (2100, 2048, 256, torch.float32, torch.float32),
])
def test_out_gemm_shapes(gpu, monkeypatch, shape, rows, k_in, n_out, x_dtype, out_dtype):
    """Against the 64-bit product: the f32 sums of exact products are within
    K 2^-24 S, S = sum |x||w| of the output itself, f32 activations lose
    2^-17 S to their bf16 pair, and a bf16 result one step."""
    from relux_amd import KVCache, pack_out
    monkeypatch.setenv("RLX_PROJ_GEMM", str(shape))
    g = torch.Generator().manual_seed(rows + k_in)
    w, = _weights(g, gpu, (k_in, n_out))
    x = torch.randn(rows, k_in, generator=g).to(gpu).to(x_dtype)
    res = torch.randn(rows, n_out, generator=g).to(gpu).to(out_dtype)
    c = KVCache(num_layers=1, max_len=16, num_kv_heads=1, head_dim=64, device=gpu.index)
    y = c.OutProject(x, pack_out(w), n_out, residual=res, out_dtype=out_dtype).double()
    want = torch.matmul(x.double(), w.double()) + res.double()
    S = torch.matmul(x.double().abs(), w.double().abs()) + res.double().abs()
    tol = S * (k_in * 2.0 ** -24 + (2.0 ** -17 if x_dtype == torch.float32 else 0.0))
    if out_dtype == torch.bfloat16:
        tol = tol + want.abs() * 2.0 ** -8
    assert bool(((y - want).abs() <= tol).all()), float(((y - want).abs() / tol).max())
    # (the bound would hide little: the sums' own error is a hundredth of it)
    if out_dtype == torch.float32:
        assert float((y - want).norm() / want.norm()) <= 1e-5


@pytest.mark.parametrize("shape", [0, 1, 2])
@pytest.mark.parametrize("H,KVH,D,dm,lens,ntok,x_dtype", [
    (8, 2, 128, 1568, [0, 7], [150, 61], torch.bfloat16),
    (4, 4, 80, 800, [3], [2100], torch.float32),
])
def test_gqa_gemm_shapes(gpu, monkeypatch, shape, H, KVH, D, dm, lens, ntok, x_dtype):
    """Q/K/V with RoPE and the append at every tile shape, against the 64-bit
    projection and rotation: bounds as above, twice for the rotation's two
    terms, and a bf16 step for the cached rows."""
    from relux_amd import KVCache, pack_qkv, rope_tables
    monkeypatch.setenv("RLX_PROJ_GEMM", str(shape))
    g = torch.Generator().manual_seed(dm)
    ws = _weights(g, gpu, (dm, H * D), (dm, KVH * D), (dm, KVH * D))
    S, rope = len(lens), rope_tables(D, 10000.0, 2200, gpu)
    x = torch.randn(sum(ntok), dm, generator=g).to(gpu).to(x_dtype)
    c = KVCache(num_layers=1, max_len=2200, num_kv_heads=KVH, head_dim=D, max_seqs=S, device=gpu.index)
    for i, n in enumerate(lens):
        if n:
            c.Append(0, torch.ones(n, KVH, D, device=gpu), torch.ones(n, KVH, D, device=gpu), seq_ids=[i], n_tok=[n],
                     layout="SHD")
    q = c.ProjectAppend(0, x, pack_qkv(*ws, H, KVH, D), H, rope=rope, seq_ids=list(range(S)), n_tok=ntok,
                        q_dtype=torch.float32)
    pos = torch.cat([torch.arange(a, a + b, device=gpu) for a, b in zip(lens, ntok)])
    co, si = (t.double()[pos][:, None, :] for t in rope)
    rel = dm * 2.0 ** -24 + 2.0 ** -20 + (2.0 ** -17 if x_dtype == torch.float32 else 0.0)

    def want(w, heads, turn):
        y = torch.matmul(x.double(), w.double()).view(-1, heads, D)
        s = torch.matmul(x.double().abs(), w.double().abs()).view(-1, heads, D)
        if turn:
            a, b, sa, sb = y[..., 0::2], y[..., 1::2], s[..., 0::2], s[..., 1::2]
            y = torch.stack([a * co - b * si, a * si + b * co], -1).flatten(-2)
            s = torch.stack([sa + sb, sa + sb], -1).flatten(-2)
        return y, s * rel
    y, tol = want(ws[0], H, True)
    assert bool(((q.double() - y).abs() <= tol).all())
    at = 0
    for i, n in enumerate(ntok):
        for (w, turn), got in zip(((ws[1], True), (ws[2], False)), c.View(0, i)):
            y, tol = want(w, KVH, turn)
            y, tol = (t[at:at + n].transpose(0, 1) for t in (y, tol))
            got = got[0].double()[:, lens[i]:]
            assert bool(((got - y).abs() <= tol + y.abs() * 2.0 ** -8 + 1e-9).all())
        at += n


@pytest.mark.parametrize("rows,dm,x_dtype,gemm", [
    (96, 640, torch.bfloat16, False), (97, 640, torch.bfloat16, True),
    (80, 640, torch.float32, False), (81, 640, torch.float32, True),
])
def test_rows_from_which_a_narrow_model_takes_the_gemm(gpu, rows, dm, x_dtype, gemm):
    from relux_amd import KVCache, pack_qkv
    if torch.cuda.get_device_properties(gpu).multi_processor_count != 256:
        pytest.skip("the bounds are of 256 CUs")
    H, KVH, D = 8, 2, 64
    g = torch.Generator().manual_seed(rows)
    wp = pack_qkv(*_weights(g, gpu, (dm, H * D), (dm, KVH * D), (dm, KVH * D)), H, KVH, D)
    x = torch.randn(rows, dm, generator=g).to(gpu).to(x_dtype)
    c = KVCache(num_layers=1, max_len=128, num_kv_heads=KVH, head_dim=D, max_seqs=2, device=gpu.index)
    q = c.ProjectAppend(0, x, wp, H, seq_ids=[0], n_tok=[rows], q_dtype=torch.float32)
    first = c.ProjectAppend(0, x[:64].contiguous(), wp, H, seq_ids=[1], n_tok=[64], q_dtype=torch.float32)
    assert torch.equal(q[:64], first) != gemm
