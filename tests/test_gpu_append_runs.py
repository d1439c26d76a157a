"""GQA appends of prompt size (whole runs of 8 slots turned in registers) and
of verify size: cache bytes against the rounded rows, bit for bit."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("KVH,D,P,before,n_tok", [
    (8, 128, 16, [0, 3, 8, 13], [2048, 5, 700, 1]),   # from every offset within an 8-slot group
    (8, 128, 48, [47, 0], [1201, 1300]),
    (16, 256, 16, [5], [600]),
    (8, 80, 64, [1, 2], [1500, 1300]),                # stored as 96 dims
    (12, 20, 16, [7], [9000]),                        # rows padded to 24, stored as 32
    (8, 128, 16, [0, 6, 15], [4, 4, 5]),              # verify sizes: runs cut at 8 slots
    (2, 128, 16, [9], [1]),
])
@pytest.mark.parametrize("layout", ["HSD", "SHD"])
@pytest.mark.parametrize("f32", [True, False])
def test_append_bytes(gpu, KVH, D, P, before, n_tok, layout, f32):
    from relux_amd import KVCache
    rng = np.random.default_rng(D + P + len(before))
    S = len(before)
    c = KVCache(num_layers=1, max_len=max(a + b for a, b in zip(before, n_tok)), num_kv_heads=KVH, head_dim=D,
                page_tokens=P, max_seqs=S, device=gpu.index)
    want = [[[], []] for _ in range(S)]
    for counts in (before, n_tok):
        seqs = [i for i in range(S) if counts[i]]
        src = []
        for which in range(2):
            rows = [rng.standard_normal((counts[i], KVH, D), dtype=np.float32) for i in seqs]
            if not f32:
                rows = [oracle.round_bf16(r) for r in rows]
            for i, r in zip(seqs, rows):
                want[i][which].append(oracle.bf16_from_f32(r))
            flat = np.concatenate([(r.transpose(1, 0, 2) if layout == "HSD" else r).reshape(-1) for r in rows])
            t = torch.from_numpy(flat).to(gpu).view(-1, KVH, D)
            src.append(t if f32 else t.to(torch.bfloat16))
        c.Append(0, *src, seq_ids=seqs, n_tok=[counts[i] for i in seqs], layout=layout)
    for i in range(S):
        for which, got in enumerate(c.View(0, i)):
            b = got.view(torch.int16).cpu().numpy().view(np.uint16)[0]  # [KVH, T, D]
            np.testing.assert_array_equal(b, np.concatenate(want[i][which]).transpose(1, 0, 2))
