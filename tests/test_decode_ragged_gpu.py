"""Full-context decode batches whose pieces follow the lengths (gpu).

In a batch of at most 64 sequences and 256 segments every segment is cut into
pieces in proportion to its tiles, or is one piece.  The batches: all lengths
equal (the cut is the host's), one long sequence among short and one-token
ones, 64 sequences (a whole wavefront of lengths), fewer pieces than
workgroups, the limits of the rule and one segment more, and partition sizes
from one tile per wavefront to whole segments.  Tolerance as for every attention
output (test_decode_gpu).
"""
import numpy as np
import pytest
import torch

import oracle
import workloads as W
from test_decode_gpu import assert_close, run_tracked
from test_q4_span_walks_gpu import decode, to_dev

pytestmark = pytest.mark.gpu

BATCHES = {
    "equal": ([777] * 4, 32, 4),
    "one long": ([3000, 1, 15, 16, 17, 33, 2], 32, 4),
    "two": ([31, 2049], 8, 2),
    "64 sequences": (list(range(1, 630, 10)) + [1500], 4, 1),
    "short": ([1, 2, 3, 4, 5, 6, 7, 8], 16, 8),
    "many": ([30 + 37 * i for i in range(24)], 16, 8),
    "many short": (list(range(1, 121, 3)), 8, 4),
    "256 segments": ([5 * i + 1 for i in range(64)], 4, 4),
    "257 segments": ([300 - i for i in range(257)], 1, 1),
}
KINDS = [(oracle.KV_F32, 64), (oracle.KV_F16, 64), (oracle.KV_Q4, 64), (oracle.KV_F32, 128),
         (oracle.KV_F16, 128), (oracle.KV_Q4, 128)]


@pytest.mark.parametrize("tokens", [0, 64, 1024])
@pytest.mark.parametrize("name", BATCHES)
@pytest.mark.parametrize("kv,d", KINDS)
def test_ragged_batches(gpu, kv, d, name, tokens):
    lens, hq, hkv = BATCHES[name]
    pb = W.paged_batch(lens, n_heads=hq, n_kv_heads=hkv, head_dim=d, block_tokens=16, seed=d + tokens,
                       kv_dtype=kv)
    q_pos = [max(0, x - 1 - 40 * (i % 3)) for i, x in enumerate(lens)]
    try:
        gpu.set_partition_tokens(tokens)
        out = decode(gpu, pb)
        out_q = decode(gpu, pb, q_pos=q_pos)
        tracked, imp = run_tracked(gpu, pb, q_pos=q_pos)
    finally:
        gpu.set_partition_tokens(0)
    assert_close(out, W.reference_decode(pb), name)
    ref = W.reference_decode(pb, q_pos=q_pos)
    assert_close(out_q, ref, f"{name}, q_pos")
    assert_close(tracked, ref, f"{name}, tracked")
    b = int(np.argmax(lens))
    _, ref_imp = oracle.attention(pb.q[b].reshape(-1), pb.layout(b), lens[b], q_pos[b], hq, hkv, d,
                                  importance=True)
    W.assert_importance(imp[b][:lens[b]], ref_imp, f"{name}, importance")


@pytest.mark.parametrize("kv,d", KINDS)
def test_ragged_batch_with_empty_sequences_and_loose_bound(gpu, kv, d):
    """Lengths of zero give zero rows, and a max_ctx far above the lengths
    changes the host's cut but not the result."""
    pb = W.paged_batch([40, 500, 16, 90], n_heads=8, n_kv_heads=2, head_dim=d, block_tokens=16, seed=d,
                       kv_dtype=kv)
    ref = W.reference_decode(pb)
    lens = pb.ctx_lens.copy()
    lens[0] = lens[3] = 0
    ref[0] = ref[3] = 0.0
    tables = np.full((4, 6250), -1, np.int32)  # room for the loose bound
    tables[:, :pb.tables.shape[1]] = pb.tables
    for bound in (500, 100000):
        out = torch.full(pb.q.shape, float("nan"), device="cuda")
        gpu.paged_decode(to_dev(pb.q), to_dev(pb.k_pool), to_dev(pb.v_pool), to_dev(tables), to_dev(lens),
                         out, 8, 2, d, 16, kv_dtype=kv, max_ctx=bound)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert not np.any(got[[0, 3]])
        assert_close(got, ref, f"bound {bound}")
