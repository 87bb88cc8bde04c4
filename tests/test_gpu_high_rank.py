"""Ranks above 64: the kernels walk the rank 128 at a time (the tile-block shrinks 64 at a time in launches of few
workgroups).  Edges of those pieces (72, 128, 136, 256), ragged
widths, single rows to several tile blocks, adapters stored at their own rank; exact (dyadic) inputs against the
oracle, bit for bit."""
import numpy as np
import pytest
import torch

from test_gpu_parity import TDT, K, _ragged_segments, dev_t, dyadic, ptrs, to_np  # noqa: F401

pytestmark = pytest.mark.gpu

SHAPES = [
    # T, S, NA, h_in, h_out, r, ranks of the adapters (None: all r)
    (3, 2, 2, 64, 72, 128, None),
    (150, 7, 3, 264, 200, 72, None),
    (1100, 9, 3, 2048, 1160, 128, None),
    (511, 4, 2, 2048, 72, 128, None),       # single tiles forward, the row below tile blocks
    (512, 4, 2, 2048, 72, 128, None),
    (511, 5, 2, 4096, 72, 72, None),        # ... at ranks up to 96 and k of 4096
    (512, 5, 2, 4096, 72, 96, None),
    (512, 5, 2, 5504, 5504, 128, None),     # k slices of 576, 64 columns a workgroup: a last batch of half its k
    (1023, 5, 2, 264, 88, 72, None),        # ... and at shorter k
    (1024, 5, 2, 264, 88, 96, None),
    (1040, 5, 2, 136, 88, 136, None),
    (1030, 6, 2, 328, 264, 256, None),
    (1200, 9, 3, 256, 520, 128, [8, 72, 128]),
    (1200, 9, 3, 4096, 4096, 200, [200, 72, 136]),   # workgroups enough for shrinks 128 columns wide, both ways
]
IDS = ["3-rows", "rank72", "rank128", "511-rows", "512-rows", "511-rows-rank72", "512-rows-rank96", "slices-of-576", "1023-rows", "1024-rows", "rank136", "rank256", "packed", "wide-shrinks"]


def _inputs(case, dt, d, seed):
    T, S, NA, h_in, h_out, r, ranks = case
    rng = np.random.default_rng(seed)
    seg = _ragged_segments(rng, T, S)
    ids = [int(i) for i in rng.integers(0, NA, S)]
    ranks = ranks or [r] * NA
    A = [dyadic(rng, (q, h_in), 8, 64) for q in ranks]
    B = [dyadic(rng, (h_out, q), 8, 8) for q in ranks]
    rank_t = torch.tensor(ranks, dtype=torch.int32, device=d) if min(ranks) < r else None
    pad = lambda w, axis: np.pad(w, [(0, r - w.shape[i]) if i == axis else (0, 0) for i in range(2)])
    return (rng, seg, ids, A, B, [pad(a, 0) for a in A], [pad(b, 1) for b in B], [dev_t(a, dt, d) for a in A],
            [dev_t(b, dt, d) for b in B], rank_t)


@pytest.mark.parametrize("dt", ["fp16", "bf16"])
@pytest.mark.parametrize("case", SHAPES, ids=IDS)
def test_forward_dyadic_bit_exact(K, oracle, gpu_device, case, dt):
    T, S, NA, h_in, h_out, r, _ = case
    d = gpu_device
    rng, seg, ids, _, _, Ap, Bp, Ad, Bd, rank_t = _inputs(case, dt, d, 31)
    x, y0 = dyadic(rng, (T, h_in), 16, 8), dyadic(rng, (T, h_out), 16, 8)
    scale = (rng.integers(1, 5, S) / 2.0).astype(np.float32)
    plan = K.SegmentPlan(torch.tensor(seg, dtype=torch.int32, device=d),
                         torch.tensor(ids, dtype=torch.int32, device=d), T, defer=True)
    y, v = dev_t(y0, dt, d), torch.zeros(T, r, dtype=TDT[dt], device=d)
    K.smlm_lora_forward(y, dev_t(x, dt, d), ptrs(Ad, d), ptrs(Bd, d), plan, r, beta=1.0, v_out=v,
                        seg_scale=torch.from_numpy(scale).to(d), adapter_rank=rank_t, packed_ranks=rank_t is not None)
    yo, vo = oracle.lora_fused(y0, x, [Ap[i] for i in ids], [Bp[i] for i in ids], seg, scale.tolist(), 1.0, dt)
    covered = np.zeros(T, bool)
    covered[seg[0]:seg[-1]] = True
    assert np.array_equal(to_np(v)[covered], vo[covered]), "v"
    assert np.array_equal(to_np(y), yo), "y"


@pytest.mark.parametrize("dt", ["fp16", "bf16"])
@pytest.mark.parametrize("drop", [False, True], ids=["plain", "dropout"])
@pytest.mark.parametrize("case", SHAPES, ids=IDS)
def test_backward_dyadic_bit_exact(K, oracle, gpu_device, case, drop, dt):
    T, S, NA, h_in, h_out, r, _ = case
    d = gpu_device
    rng, seg, ids, A, B, Ap, Bp, Ad, Bd, rank_t = _inputs(case, dt, d, 32)
    tp = [c - seg[0] for c in seg]
    n = tp[-1]
    x, g = dyadic(rng, (n, h_in), 16, 8), dyadic(rng, (n, h_out), 16, 8)
    seg_p = np.array([0.5 if a % 2 == 0 else 0.0 for a in ids], np.float32)
    spec = K.DropoutSpec(torch.from_numpy(seg_p).to(d), n, 7, 11) if drop else None
    dA, dB = [torch.full_like(a, 9.0) for a in Ad], [torch.full_like(b, 9.0) for b in Bd]
    dx = torch.empty(n, h_in, dtype=TDT[dt], device=d)
    plan = K.SegmentPlan(torch.tensor(tp, dtype=torch.int32, device=d),
                         torch.tensor(ids, dtype=torch.int32, device=d), n, defer=True)
    xo = x
    if drop:
        rp = np.zeros(n, np.float32)
        for i in range(S):
            rp[tp[i]:tp[i + 1]] = seg_p[i]
        xo = oracle.dropout_rows(x, rp, 7, 11, dt)
    _, vo = oracle.add_lora_forward(xo, [Ap[i] for i in ids], [Bp[i] for i in ids], tp, h_out, dt)
    K.smlm_lora_backward(dx, ptrs(dA, d), ptrs(dB, d), dev_t(g, dt, d), dev_t(x, dt, d), dev_t(vo, dt, d), ptrs(Ad, d),
                         ptrs(Bd, d), plan, r, dropout=spec, adapter_rank=rank_t, packed_ranks=rank_t is not None)
    gx, ga, gb = oracle.add_lora_backward(g, xo, Ap, Bp, tp, ids, dt)
    if drop:
        gx = oracle.dropout_rows(gx, rp, 7, 11, dt)
    assert np.array_equal(to_np(dx), gx), "dX"
    for a in range(NA):
        assert np.array_equal(to_np(dA[a]), ga[a][:A[a].shape[0]]), f"dA[{a}]"
        assert np.array_equal(to_np(dB[a]), gb[a][:, :B[a].shape[1]]), f"dB[{a}]"


@pytest.mark.parametrize("dt", ["fp16", "bf16"])
@pytest.mark.parametrize("drop", [False, True], ids=["plain", "dropout"])
@pytest.mark.parametrize("packed", [False, True], ids=["padded", "packed"])
@pytest.mark.parametrize("k", [1024, 4096, 2560, 5504],
                         ids=["64-columns", "128-columns", "odd-split-falls-back", "slices-of-576"])
def test_plans_of_300_segments_built_in_the_shrinks(K, gpu_device, k, packed, drop, dt):
    """More segments than a four-wave workgroup has threads: the shrinks of both directions run two groups of waves a
    workgroup, 64 or 128 columns wide.  Everything they leave equals what plans built beforehand give, bit for bit."""
    d, tdt, r, NA, S = gpu_device, TDT[dt], 200, 9, 300
    T = 5 * S
    ranks = [(8, 72, 200)[a % 3] for a in range(NA)] if packed else [r] * NA
    gen = torch.Generator().manual_seed(7)
    rand = lambda *shape: torch.randn(*shape, generator=gen).to(tdt).to(d)
    A, B = [rand(q, k) / k ** 0.5 for q in ranks], [rand(k, q) / q ** 0.5 for q in ranks]
    x, y0, g = rand(T, k), rand(T, k), rand(T, k)
    int32 = lambda v: torch.tensor(v, dtype=torch.int32, device=d)
    seg, ids = int32(list(range(0, T + 1, 5))), int32([(i * 7) % NA for i in range(S)])
    rank = dict(adapter_rank=int32(ranks) if packed else None, packed_ranks=packed)
    scale = torch.full((S,), 1.5, device=d)
    seg_p = torch.tensor([0.5 if i % 7 else 0.0 for i in range(S)], device=d)
    nbytes = K.SegmentPlan.nbytes(T, S)

    def run(defer):
        plan, bplan = (K.SegmentPlan(seg, ids, T, buf=torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=d), defer=defer)
                       for _ in range(2))
        bits = torch.zeros(K.DropoutSpec.mask_nbytes(T, [k]), dtype=torch.uint8, device=d)
        spec = K.DropoutSpec(seg_p, T, 17, 3, bits) if drop else None
        y, v = y0.clone(), torch.zeros(T, r, dtype=tdt, device=d)
        K.smlm_lora_forward(y, x, ptrs(A, d), ptrs(B, d), plan, r, seg_scale=scale, beta=1.0, v_out=v, dropout=spec, **rank)
        dA, dB = [torch.full_like(a, 9.0) for a in A], [torch.full_like(b, 9.0) for b in B]
        dx = torch.full((T, k), 9.0, dtype=tdt, device=d)
        K.smlm_lora_backward(dx, ptrs(dA, d), ptrs(dB, d), g, x, v, ptrs(A, d), ptrs(B, d), bplan, r, scale, dropout=spec,
                             **rank)
        torch.cuda.synchronize()
        return [y, v, bits, plan.buf, bplan.buf, dx] + dA + dB

    for a, b in zip(run(False), run(True)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n", [1, 16, 63, 65, 200])
@pytest.mark.parametrize("r", [8, 40, 64, 72, 136])
def test_fold_of_dv_by_tile_slot(K, oracle, gpu_device, r, n):
    """The fold of dV takes four tiles and 64 columns at a time and leaves s dV and s v transposed: pieces of both, rows
    that end within a tile and within the four, an adapter without rows, scales; dyadic inputs, bit for bit."""
    d, dt, NA, h = gpu_device, "bf16", 4, 1024
    rng = np.random.default_rng(100 * r + n)
    seg, ids = [0, n // 3, n // 3, n // 2, n], [0, 3, 1, 0]
    A, B = [dyadic(rng, (r, h), 8, 64) for _ in range(NA)], [dyadic(rng, (h, r), 8, 8) for _ in range(NA)]
    x, g = dyadic(rng, (n, h), 16, 8), dyadic(rng, (n, h), 16, 8)
    Ad, Bd = [dev_t(a, dt, d) for a in A], [dev_t(b, dt, d) for b in B]
    dA, dB = [torch.full_like(a, 9.0) for a in Ad], [torch.full_like(b, 9.0) for b in Bd]
    dx = torch.empty(n, h, dtype=TDT[dt], device=d)
    int32 = lambda v: torch.tensor(v, dtype=torch.int32, device=d)
    _, v = oracle.add_lora_forward(x, [A[i] for i in ids], [B[i] for i in ids], seg, h, dt)
    K.smlm_lora_backward(dx, ptrs(dA, d), ptrs(dB, d), dev_t(g, dt, d), dev_t(x, dt, d), dev_t(v, dt, d), ptrs(Ad, d),
                         ptrs(Bd, d), K.SegmentPlan(int32(seg), int32(ids), n), r,
                         torch.full((len(ids),), 2.0, device=d))
    # a scale of two: every gradient is twice the unscaled one, bit for bit
    gx, ga, gb = oracle.add_lora_backward(g, x, A, B, seg, ids, dt)
    assert np.array_equal(to_np(dx), 2 * gx), "dX"
    for a in range(NA):
        assert np.array_equal(to_np(dA[a]), 2 * ga[a]), f"dA[{a}]"
        assert np.array_equal(to_np(dB[a]), 2 * gb[a]), f"dB[{a}]"
