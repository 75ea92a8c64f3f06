"""Q4_K products at the edges of the kernels' tiles (gpu).

Row counts around the 8- and 16-row units and the smallest tiles, row lengths
of 1 to 208 blocks (fewer blocks than a step takes, blocks that do not divide
among the wavefronts or the four sums, rows whose converted inputs do not fit
the LDS) and input counts around 8, 16 and 32; then each of the tiles.  Outputs
are checked against the float64 dequantise-then-dot and must equal those of
single or eight-input calls bit for bit.

Tolerance: inputs are carried to within 2^-23 and products summed in f32, so
per output |error| <= c 2^-23 sum|w x| with a small c (the sums' roundings add
up like a random walk); c = 4 is taken, against sum_j of |d scale q x| +
|dmin min x|, the terms the formula adds.
"""
import numpy as np
import pytest
import torch

import workloads as W

pytestmark = pytest.mark.gpu

CASES = [
    (1, 256, 1), (15, 256, 3), (17, 512, 2), (33, 768, 4), (16, 1280, 5), (4080, 256, 1),
    (4081, 512, 1), (4097, 768, 2), (300, 2048, 8), (31, 2048, 9), (33, 1792, 16),
    (65, 2304, 17), (129, 512, 33), (383, 1280, 31), (385, 256, 100), (2050, 512, 200),
    (40, 5632, 6), (40, 5632, 13), (24, 14336, 1), (24, 14336, 3), (24, 14336, 7),
    (9, 53248, 2), (9, 53248, 1),
    # inputs converted by wavefronts that do not multiply: fewer pairs than
    # wavefronts, an odd number, more than one turn; the last row count and
    # length that take it, and the next
    (7, 256, 3), (40, 768, 2), (65, 1280, 4), (2048, 2048, 4), (2049, 2048, 3), (16, 2304, 4), (30, 1024, 7),
]


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def terms(w, n_rows, n_cols):
    """|d scale q| + |dmin min| of every weight, float64."""
    total = 0.0
    for field in (0, 2):  # without d, without dmin
        part = w.reshape(-1, 144).copy()
        part[:, field:field + 2] = 0
        total = total + np.abs(W.q4k_dequant_np(part, n_rows, n_cols).astype(np.float64))
    return total.reshape(n_rows, n_cols)


@pytest.mark.parametrize("n_rows,n_cols,batch", CASES)
def test_q4k_tile_edges(gpu, n_rows, n_cols, batch):
    w = W.q4k_random_weights(n_rows, n_cols, seed=n_rows + n_cols)
    x = np.random.default_rng(batch).standard_normal((batch, n_cols)).astype(np.float32)
    x[:, ::7] *= np.float32(1e-4)  # a spread of magnitudes within a block
    dw, dx = dev(w), dev(x)
    out = torch.full((batch, n_rows + 3), float("nan"), device="cuda")
    gpu.gemv_q4k_batched(dw, dx, out, n_rows, n_cols)
    single = torch.full((n_rows,), float("nan"), device="cuda")
    singles = []
    for b in sorted({0, batch // 2, batch - 1}):
        gpu.gemv_q4k(dw, dx[b].contiguous(), single, n_rows, n_cols)
        singles.append((b, single.clone()))
    torch.cuda.synchronize()
    for b, s in singles:
        assert torch.equal(out[b, :n_rows], s), b
    assert torch.isnan(out[:, n_rows:]).all()  # stride padding untouched
    deq = W.q4k_dequant_np(w, n_rows, n_cols).astype(np.float64).reshape(n_rows, n_cols)
    ref = x.astype(np.float64) @ deq.T
    bound = 4 * 2.0**-23 * (np.abs(x).astype(np.float64) @ terms(w, n_rows, n_cols).T)
    got = out[:, :n_rows].cpu().numpy().astype(np.float64)
    assert np.all(np.abs(got - ref) <= bound), np.max(np.abs(got - ref) / bound)


@pytest.mark.parametrize("n_cols,batch", [(512, 1), (512, 4), (512, 20), (14336, 5)])
def test_q4k_input_extremes(gpu, n_cols, batch):
    """Zeros, values at either end of f32 and a power-of-two ladder are scaled
    within their block, blocks and inputs apart from each other; an infinity or
    a NaN makes every output of its own input NaN and none of another's."""
    n_rows = 37
    w = W.q4k_random_weights(n_rows, n_cols, seed=5)
    rng = np.random.default_rng(6)
    x = rng.standard_normal((batch, n_cols)).astype(np.float32)
    x[0, :256] = 0
    x[-1, 256:512] = np.float32(1e-38)
    x[batch // 2, :256] = np.float32(2.0) ** rng.integers(-20, 20, 256)
    scale = {0: np.float32(1e30), batch - 1: np.float32(1e-30)}.get(batch // 2, np.float32(1))
    x[batch // 2] *= scale if batch > 2 else np.float32(1)
    out = torch.empty((batch, n_rows), device="cuda")
    gpu.gemv_q4k_batched(dev(w), dev(x), out, n_rows, n_cols)
    torch.cuda.synchronize()
    deq = W.q4k_dequant_np(w, n_rows, n_cols).astype(np.float64).reshape(n_rows, n_cols)
    ref = x.astype(np.float64) @ deq.T
    mag = np.abs(x).astype(np.float64) @ np.abs(deq).T
    got = out.cpu().numpy().astype(np.float64)
    assert np.all(np.isfinite(got))
    assert np.all(np.abs(got - ref) <= 64 * 2.0**-23 * mag + 1e-37)
    bad = x.copy()
    bad[0, 3] = np.inf
    bad[batch - 1, 300] = np.nan
    gpu.gemv_q4k_batched(dev(w), dev(bad), out, n_rows, n_cols)
    torch.cuda.synchronize()
    again = out.cpu().numpy()
    assert np.isnan(again[0]).all() and np.isnan(again[batch - 1]).all()
    for b in range(1, batch - 1):
        assert np.array_equal(again[b], got[b].astype(np.float32)), b


# (rows, inputs) for which the launch takes, on 256 CUs, the 32x16 and 64x16
# tiles with their blocks in four K groups, and the 64x16, 128x32, 256x32 and
# 384x32 tiles with one; remainders in both
TILES = [(100, 33), (1500, 129), (5633, 33), (5633, 129), (4097, 260), (4097, 509)]


@pytest.mark.parametrize("blocks", [1, 2, 3, 4, 5, 6, 7, 8, 11, 43])
@pytest.mark.parametrize("n_rows,batch", TILES)
def test_q4k_every_tile(gpu, n_rows, batch, blocks):
    """Every tile over row lengths of every remainder by the four sums, each sum
    of none, one or several blocks: all outputs equal those of calls with eight
    inputs (another kernel), and a sample of rows the float64 product."""
    n_cols = 256 * blocks
    w = W.q4k_random_weights(n_rows, n_cols, seed=blocks)
    x = np.random.default_rng(batch).standard_normal((batch, n_cols)).astype(np.float32)
    dw, dx = dev(w), dev(x)
    out = torch.full((batch, n_rows), float("nan"), device="cuda")
    few = torch.full((batch, n_rows), float("nan"), device="cuda")
    gpu.gemv_q4k_batched(dw, dx, out, n_rows, n_cols)
    for b in range(0, batch, 8):
        gpu.gemv_q4k_batched(dw, dx[b:b + 8], few[b:b + 8], n_rows, n_cols)
    torch.cuda.synchronize()
    assert torch.equal(out, few)
    rows = np.unique(np.linspace(0, n_rows - 1, 50).astype(int))
    deq = W.q4k_dequant_np(w[rows], len(rows), n_cols).astype(np.float64).reshape(len(rows), n_cols)
    ref = x.astype(np.float64) @ deq.T
    bound = 8 * 2.0**-23 * (np.abs(x).astype(np.float64) @ np.abs(deq).T)
    got = out[:, torch.from_numpy(rows).cuda()].cpu().numpy()
    assert np.all(np.abs(got - ref) <= bound), np.max(np.abs(got - ref) / bound)


@pytest.mark.parametrize("index", [3, 40, 131, 255])
@pytest.mark.parametrize("zero", ["scale and min", "min and nibble"])
@pytest.mark.parametrize("batch", [1, 3, 20])
def test_q4k_large_values_under_zero_weights(gpu, batch, zero, index):
    """One value of each block 2^6 to 2^28 times the others, where every weight
    is zero, through zero scale and min or zero min and nibble: the others keep
    their precision.

    The roundings of f32 sums are independent of each other and 2^-24 of terms
    or of sums of their size, so the errors' norm is c 2^-24 of the norm of the
    terms, for which |w x| stands; c = 6 (three roundings a term, twice)."""
    n_rows, n_cols = 300, 2048
    w = W.q4k_random_weights(n_rows, n_cols, seed=index)
    b = w.reshape(-1, 144)
    sub, i = index // 32, index % 32
    for field in (4,) if zero == "min and nibble" else (0, 4):  # the sub-block's scale, min
        if sub < 4:
            b[:, 4 + field + sub] &= 0xc0
        else:
            b[:, 8 + sub] &= 0xf0 if field == 0 else 0x0f
            b[:, field + sub] &= 0x3f
    if zero == "min and nibble":
        b[:, 16 + 32 * (sub // 2) + i] &= 0x0f if sub % 2 else 0xf0
    deq = W.q4k_dequant_np(w, n_rows, n_cols).astype(np.float64).reshape(n_rows, n_cols)
    assert not np.any(deq[:, index::256])
    rng = np.random.default_rng(batch)
    for bits in (6, 10, 16, 20, 24, 28):
        x = rng.standard_normal((batch, n_cols)).astype(np.float32)
        ref = x.astype(np.float64) @ deq.T
        norm = np.sqrt(np.sum(x.astype(np.float64)**2 @ (deq**2).T))
        x[:, index::256] = np.float32(1.37 * 2.0**bits)
        out = torch.full((batch, n_rows), float("nan"), device="cuda")
        gpu.gemv_q4k_batched(dev(w), dev(x), out, n_rows, n_cols)
        torch.cuda.synchronize()
        err = np.linalg.norm(out.cpu().numpy() - ref)
        assert err <= 6 * 2.0**-24 * norm, (bits, err / norm)
