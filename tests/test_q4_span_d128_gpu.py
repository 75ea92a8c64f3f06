"""Q4-20B decode at head_dim 128 on contiguous walks against the oracle (gpu).

A tile's 16 K and 16 V rows (2560 bytes) are loaded as spans into the
wavefront's LDS slots, untracked in pairs from a ring of four, tracked one at
a time from a ring of two.  The partition size sweeps the tiles per wavefront
(test_q4_span_walks_gpu): none, one, odd, even, whole rings, partial last
tiles.  Tolerance as for every attention output (test_decode_gpu).
"""
import numpy as np
import pytest
import torch

import oracle
import workloads as W
from test_decode_gpu import assert_close, run_tracked
from test_q4_span_walks_gpu import CTX, Q_POS, decode, to_dev

pytestmark = pytest.mark.gpu


def batch(seed, hkv=8, **kw):
    return W.paged_batch(CTX, n_heads=32, n_kv_heads=hkv, head_dim=128, block_tokens=16, seed=seed,
                         kv_dtype=oracle.KV_Q4, **kw)


@pytest.mark.parametrize("tokens,hkv", [(64, 8), (128, 2), (256, 8), (512, 32), (1024, 1), (4096, 8)])
def test_q4_d128_walk_lengths(gpu, tokens, hkv):
    pb = batch(tokens, hkv)
    try:
        gpu.set_partition_tokens(tokens)
        full = decode(gpu, pb)
        qpos = decode(gpu, pb, q_pos=Q_POS)
        win = decode(gpu, pb, window=40, stride=0)
        glob = decode(gpu, pb, window=200, stride=16)
        tracked, imp = run_tracked(gpu, pb, q_pos=Q_POS)
    finally:
        gpu.set_partition_tokens(0)
    ref = W.reference_decode(pb, q_pos=Q_POS)
    assert_close(full, W.reference_decode(pb), f"{tokens} tokens: full")
    assert_close(qpos, ref, f"{tokens} tokens: q_pos")
    assert_close(win, W.reference_decode(pb, window=40), f"{tokens} tokens: window 40")
    assert_close(glob, W.reference_decode(pb, window=200, global_stride=16),
                 f"{tokens} tokens: window 200, globals every 16")
    assert_close(tracked, ref, f"{tokens} tokens: tracked out")
    for b in range(pb.batch):
        L = int(pb.ctx_lens[b])
        _, ref_imp = oracle.attention(pb.q[b].reshape(-1), pb.layout(b), L, Q_POS[b], pb.n_heads,
                                      pb.n_kv_heads, pb.head_dim, importance=True)
        W.assert_importance(imp[b][:L], ref_imp, f"{tokens} tokens: importance b={b}")


@pytest.mark.parametrize("tokens", [64, 512])
def test_q4_d128_absent_blocks_and_pool_alignment(gpu, tokens):
    """The same rows in blocks of 8 tokens take the gathered per-row walk: with
    table entries absent or out of range both skip the same positions, and
    pools that start 4 bytes past a 16-byte boundary read the same rows."""
    pb = batch(7)
    pb.tables[2, 0] = -1
    pb.tables[4, 5:9] = 1 << 20
    pb.tables[5, 83] = -1
    total, hkv = pb.k_pool.shape[:2]

    def halved(pool):
        p = pool.reshape(total, hkv, 2, 8, -1).transpose(0, 2, 1, 3, 4)
        return np.ascontiguousarray(p.reshape(2 * total, hkv, 8, -1))

    def shifted(pool):
        buf = torch.zeros(pool.size + 16, dtype=torch.uint8, device="cuda")
        view = buf[4:4 + pool.size].view(pool.shape)
        view.copy_(torch.from_numpy(pool))
        assert view.data_ptr() % 16 == 4
        return view

    t8 = np.stack([2 * pb.tables, 2 * pb.tables + 1], axis=-1).reshape(pb.batch, -1)
    t8[np.repeat(pb.tables < 0, 2, axis=1)] = -1

    def run(k, v, tables, bt, window):
        out = torch.full((pb.batch, 32, 128), float("nan"), device="cuda")
        gpu.paged_decode(to_dev(pb.q), k, v, to_dev(tables.astype(np.int32)), to_dev(pb.ctx_lens), out,
                         32, hkv, 128, bt, kv_dtype=pb.kv_dtype, window=window, global_stride=0,
                         max_ctx=int(pb.ctx_lens.max()))
        torch.cuda.synchronize()
        return out.cpu().numpy()

    try:
        gpu.set_partition_tokens(tokens)
        for window in (0, 300):
            gathered = run(to_dev(halved(pb.k_pool)), to_dev(halved(pb.v_pool)), t8, 8, window)
            spans = run(shifted(pb.k_pool), shifted(pb.v_pool), pb.tables, 16, window)
            assert_close(spans, gathered, f"window {window}")
    finally:
        gpu.set_partition_tokens(0)
