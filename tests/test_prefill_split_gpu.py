"""Prefill launches whose keys are split among groups of wavefronts (gpu):
few (head, row block) items against the oracle, at the edges of the groups'
tile ranges and of the rule that takes the split.

Inputs are bf16 on both sides and scores and sums are f32, so what is left is
the binary16 rounding of the weights: 2^-11 of each, so at most 2^-11 of the
largest |v| per output, and 1e-3 of the largest output holds it twice.
"""
import numpy as np
import pytest
import torch

import oracle
import workloads as W
from test_prefill_gpu import check, oracle_ctx_rows, oracle_rows, run_prefill, run_prefill_ctx

pytestmark = pytest.mark.gpu


# tiles of 64 keys over 4 groups (head_dim 64) or 2 (head_dim 128): fewer
# tiles than groups, one more than a multiple, one key past a tile, a last
# group without tiles; heads 1, 2 and 4 per group of wavefronts; the last
# shape that one workgroup per CU holds and the first beyond
CASES = [(0, 449, 4, 1, 64, True), (0, 513, 4, 4, 64, True), (0, 448, 4, 2, 64, True),
         (1, 1, 4, 2, 64, True), (64, 1, 2, 1, 64, False), (129, 33, 6, 2, 64, True),
         (300, 77, 12, 12, 64, True), (575, 65, 8, 1, 64, False), (70, 512, 32, 4, 64, True),
         (70, 513, 32, 4, 64, True), (0, 193, 8, 2, 128, True), (0, 192, 8, 8, 128, False),
         (0, 321, 8, 2, 128, True), (0, 385, 8, 8, 128, False),
         (1, 1, 4, 2, 128, True), (65, 31, 6, 3, 128, True), (190, 130, 8, 1, 128, False),
         (64, 257, 5, 5, 128, True), (100, 1024, 32, 8, 128, True), (100, 1025, 32, 8, 128, True)]


@pytest.mark.parametrize("n_hist,n,hq,hkv,d,causal", CASES)
def test_split_prefill_rows(gpu, n_hist, n, hq, hkv, d, causal):
    q, k, v = W.prefill_inputs(n_hist + n, hq, hkv, d, seed=n + n_hist)
    rows = np.unique(np.concatenate([np.arange(min(n, 40)), np.arange(max(0, n - 70), n)]))
    what = f"{n_hist}+{n} {hq}/{hkv} {d}"
    if n_hist == 0:
        check(run_prefill(gpu, q, k, v, causal), oracle_rows(q, k, v, rows, causal), rows, what)
        return
    args = (q[n_hist:], k[n_hist:], v[n_hist:], k[:n_hist], v[:n_hist])
    check(run_prefill_ctx(gpu, *args, causal), oracle_ctx_rows(*args, rows, causal), rows, what)
    assert gpu.take_status()[0] == 0


@pytest.mark.parametrize("d,step", [(64, 0.72), (64, -0.72), (128, 0.72), (128, -0.72)])
def test_split_prefill_groups_with_distant_maxima(gpu, d, step):
    """Scores that rise or fall by `step` per key: a group's maximum is
    hundreds away from the next one's, so all but one group's parts merge with
    a weight of zero."""
    n_hist, n, hq, hkv = 500, 100, 4, 2
    rng = np.random.default_rng(5)
    u = rng.standard_normal(d).astype(np.float32)
    u /= np.linalg.norm(u)
    t = np.arange(n_hist + n, dtype=np.float32)[:, None, None]
    q = np.tile(u * np.float32(np.sqrt(d)), (n, hq, 1)).astype(np.float32)
    k = np.repeat((step * t * u).astype(np.float32), hkv, axis=1)
    v = rng.standard_normal((n_hist + n, hkv, d)).astype(np.float32)
    args = (q, k[n_hist:], v[n_hist:], k[:n_hist], v[:n_hist])
    rows = np.arange(n)
    check(run_prefill_ctx(gpu, *args), oracle_ctx_rows(*args, rows), rows, f"step {step}")


@pytest.mark.parametrize("d,n,hq", [(64, 77, 8), (64, 1100, 32), (128, 77, 8), (128, 1100, 32)])
def test_prefill_q4_pool_rows(gpu, d, n, hq):
    """4-bit pools written by both kernels (split and not), from a position
    inside a block, byte for byte; the other rows keep their bytes."""
    hkv, bt, start, n_hist = 2, 16, 21, 30
    q, k, v = W.prefill_inputs(n_hist + n, hq, hkv, d, seed=d)
    nb = (start + n + bt - 1) // bt + 2
    table = np.random.default_rng(3).permutation(nb).astype(np.int32)
    kp = torch.full((nb, hkv, bt, oracle.q4_row_bytes(d)), 7, dtype=torch.uint8, device="cuda")
    vp = kp.clone()
    args = (q[n_hist:], k[n_hist:], v[n_hist:], k[:n_hist], v[:n_hist])
    run_prefill_ctx(gpu, *args, k_pool=kp, v_pool=vp, block_table=torch.from_numpy(table).cuda(),
                    block_tokens=bt, kv_dtype=oracle.KV_Q4, start_pos=start)
    t = np.arange(start, start + n)
    for pool, x in ((kp, k), (vp, v)):
        p = pool.cpu().numpy()
        assert np.array_equal(p[table[t // bt], :, t % bt],
                              oracle.q4_quantize_rows(W.bf16_round(x[n_hist:])))
        p[table[t // bt], :, t % bt] = 7
        assert np.all(p == 7)


@pytest.mark.parametrize("where", ["history", "chunk"])
@pytest.mark.parametrize("d,n,hq", [(64, 40, 4), (128, 40, 4), (64, 1100, 32), (128, 1100, 32)])
def test_prefill_v_beyond_binary16_is_reported(gpu, where, d, n, hq):
    """The largest bf16 below the binary16 overflow passes, the next one is
    reported, wherever it lies (the last kv head's last element)."""
    n_hist, hkv = 70, 2
    q, k, v = W.prefill_inputs(n_hist + n, hq, hkv, d, seed=1)
    at = n_hist - 1 if where == "history" else n_hist + n - 1
    for big, code in ((65280.0, 0), (-65536.0, gpu.ERR_RANGE)):
        v[at, hkv - 1, d - 1] = big
        run_prefill_ctx(gpu, q[n_hist:], k[n_hist:], v[n_hist:], k[:n_hist], v[:n_hist])
        assert gpu.take_status()[0] == code, big


# rows written by workgroups of their own, in one turn and in two (431), the
# last turn partly used; and at 449 and 321 rows the first that the split
# kernel's workgroups write
@pytest.mark.parametrize("n,hq,hkv,d", [(1, 4, 4, 64), (33, 12, 12, 64), (256, 12, 12, 64), (431, 12, 12, 64), (449, 12, 12, 64),
                                        (5, 8, 1, 64), (300, 32, 4, 64), (1, 2, 2, 128), (68, 32, 8, 128),
                                        (130, 8, 8, 128), (320, 8, 8, 128), (321, 8, 8, 128)])
def test_short_prefill_writes_and_checks_each_row_once(gpu, n, hq, hkv, d):
    """Every row of a chunk without history, byte for byte what the K/V write
    entry point stores, in each format; other rows keep their bytes.  Without
    pools the V of the same rows is checked."""
    bt, start = 16, 21
    q, k, v = W.prefill_inputs(n, hq, hkv, d, seed=n + d)
    nb = (start + n + bt - 1) // bt + 2
    table = torch.from_numpy(np.random.default_rng(3).permutation(nb).astype(np.int32)).cuda()
    rounded = [torch.from_numpy(W.bf16_round(x)).cuda() for x in (k, v)]
    rows = np.unique(np.concatenate([np.arange(min(n, 20)), np.arange(max(0, n - 20), n)]))
    ref = oracle_rows(q, k, v, rows)
    for kv, row in ((oracle.KV_F32, 4 * d), (oracle.KV_F16, 2 * d), (oracle.KV_Q4, oracle.q4_row_bytes(d))):
        got = [torch.full((nb, hkv, bt, row), 7, dtype=torch.uint8, device="cuda") for _ in "kv"]
        want = [x.clone() for x in got]
        gpu.kv_write(*want, table, bt, hkv, d, kv, start, *rounded)
        check(run_prefill(gpu, q, k, v, k_pool=got[0], v_pool=got[1], block_table=table, block_tokens=bt,
                          kv_dtype=kv, start_pos=start), ref, rows, f"{n} {hq}/{hkv} {d}")
        assert all(torch.equal(a, b) for a, b in zip(got, want)), kv
    for at, h, x in ((0, 0, 0), (n - 1, hkv - 1, d - 1)):
        big = v.copy()
        big[at, h, x] = 65280.0
        run_prefill(gpu, q, k, big)
        assert gpu.take_status()[0] == 0
        big[at, h, x] = -65536.0
        run_prefill(gpu, q, k, big)
        assert gpu.take_status()[0] == gpu.ERR_RANGE
