"""The Attention node up to the last row of a contiguous cache (gpu).

A cache [Hkv][kv_stride][row] whose rows are no multiple of 16 ends inside the
last head's last tile, and nothing may be read behind it.  The walk takes that
tile earlier, so that it ends with the cache, and masks the rows that belong to
the tile before; caches of fewer than 16 rows are read row by row.  Each row
must count exactly once: against the oracle, for every position of the end
within a tile, whole segments and split pieces, with rows that are not numbers
where the sequence ends before the cache.  Tolerance as for every attention
output (test_decode_gpu)."""
import numpy as np
import pytest
import torch

import oracle
from test_decode_gpu import assert_close, to_dev

pytestmark = pytest.mark.gpu

KV = {"f32": oracle.KV_F32, "f16": oracle.KV_F16, "q4": oracle.KV_Q4}


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("kv", list(KV))
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 31, 33, 100, 1003])
def test_node_to_the_end_of_its_cache(gpu, rows, kv, head_dim):
    rng = np.random.default_rng(rows * head_dim)
    hq, hkv, dt = 6, 3, KV[kv]
    q = rng.standard_normal((hq, head_dim), dtype=np.float32)
    k, v = (rng.standard_normal((hkv, rows, head_dim), dtype=np.float32) for _ in "kv")
    if kv == "q4":
        k, v = oracle.q4_quantize_rows(k), oracle.q4_quantize_rows(v)
    elif kv == "f16":
        k, v = k.astype(np.float16), v.astype(np.float16)
    dq = to_dev(q)
    for seq_len in sorted({rows, max(1, rows - 1), max(1, rows - 14)}, reverse=True):
        for x in (k, v):  # past the sequence: a NaN in every format
            x[:, seq_len:] = 0xFF if kv == "q4" else np.nan
        wide = [x.astype(np.float32) if kv == "f16" else x for x in (k, v)]
        ref = oracle.attention(q.reshape(-1),
                               oracle.contiguous_layout(*wide, rows, head_dim,
                                                        oracle.KV_Q4 if kv == "q4" else oracle.KV_F32),
                               seq_len, seq_len - 1, hq, hkv, head_dim).reshape(hq, head_dim)
        dk, dv = to_dev(k), to_dev(v)
        for scores in (None, torch.empty(hq * seq_len, device="cuda")):
            out = torch.full_like(dq, float("nan"))
            gpu.attention_node(dq, dk, dv, out, hq, hkv, seq_len, head_dim, rows, kv_dtype=dt, scores=scores)
            torch.cuda.synchronize()
            assert_close(out.cpu().numpy(), ref, f"{kv}, {seq_len} of {rows} rows, scores {scores is not None}")
