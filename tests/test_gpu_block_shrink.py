"""Tile-block shrinks up to rank 64: pieces of 64 of k over four waves, slices of k, lists of chunk rows.  Edges of each
-- k short of a piece, of a round of the waves and of a slice, projections of different k in one launch, blocks of one to
four tiles, ranks short of the column block, adapters without weights -- with exact (dyadic) inputs against the oracle,
bit for bit; plans built beforehand and in the launch."""
import numpy as np
import pytest
import torch

from test_gpu_parity import TDT, K, _ragged_segments, dev_t, dyadic, ptrs, to_np  # noqa: F401

pytestmark = pytest.mark.gpu

CASES = {
    # T, S, NA, widths, r, ranks of the adapters (None: all r)
    "rank8": (2100, 9, 3, [(264, 72), (2048, 64), (72, 136)], 8, None),
    "rank16-ks": (2100, 300, 5, [(1000, 64), (4104, 72)], 16, None),
    "rank24": (3100, 9, 3, [(328, 64), (64, 72), (8, 64)], 24, None),
    "rank24-wide": (800, 9, 3, [(328, 64), (64, 72), (8, 64)], 24, None),  # (too few rows: the other tile-block shrink)
    "rank32-packed": (3100, 17, 4, [(1032, 72), (520, 264)], 32, [32, 8, 24, 16]),
    "rank40": (3100, 11, 3, [(2056, 64), (136, 72)], 40, None),
    "rank64": (3500, 400, 7, [(576, 64), (2048, 72)], 64, None),
    "rank64-packed": (3100, 40, 12, [(520, 72), (1096, 64)], 64, [8, 64, 40, 16, 24, 56, 32, 48, 8, 8, 64, 16]),
    "no-split": (8200, 6, 2, [(320, 64)], 32, None),
}


def _make(case, seed):
    T, S, NA, widths, r, ranks = case
    rng = np.random.default_rng(seed)
    ids = [int(i) for i in rng.integers(0, NA, S)]
    ranks = ranks or [r] * NA
    A = [[dyadic(rng, (q, h), 8, 64) for q in ranks] for h, _ in widths]
    B = [[dyadic(rng, (o, q), 8, 8) for q in ranks] for _, o in widths]
    return rng, _ragged_segments(rng, T, S), ids, ranks, A, B


@pytest.mark.parametrize("dt", ["fp16", "bf16"])
@pytest.mark.parametrize("name", CASES)
def test_forward_and_backward(K, oracle, gpu_device, name, dt):
    T, S, NA, widths, r, given = case = CASES[name]
    d, P = gpu_device, len(widths)
    rng, seg, ids, ranks, A, B = _make(case, 41)
    pad = lambda w, axis: np.pad(w, [(0, r - w.shape[i]) if i == axis else (0, 0) for i in range(2)])
    Ap, Bp = [[pad(a, 0) for a in w] for w in A], [[pad(b, 1) for b in w] for w in B]
    Ad, Bd = [[dev_t(a, dt, d) for a in w] for w in A], [[dev_t(b, dt, d) for b in w] for w in B]
    x, y0 = [dyadic(rng, (T, h), 16, 8) for h, _ in widths], [dyadic(rng, (T, o), 16, 8) for _, o in widths]
    int32 = lambda v: torch.tensor(v, dtype=torch.int32, device=d)
    rank = dict(adapter_rank=int32(ranks) if given else None, packed_ranks=bool(given))
    tabs = lambda ws: [ptrs(w, d) for w in ws]
    want = [oracle.lora_fused(y0[i], x[i], [Ap[i][a] for a in ids], [Bp[i][a] for a in ids], seg, None, 1.0, dt)
            for i in range(P)]
    tp, n = [c - seg[0] for c in seg], seg[-1] - seg[0]
    covered = slice(seg[0], seg[-1])
    g = [dyadic(rng, (n, o), 16, 8) for _, o in widths]
    xb = [a[covered] for a in x]
    vb = [v[covered] for _, v in want]
    grads = [oracle.add_lora_backward(g[i], xb[i], Ap[i], Bp[i], tp, ids, dt) for i in range(P)]
    for defer in (True, False):
        plan = K.SegmentPlan(int32(seg), int32(ids), T, defer=defer)
        y = [dev_t(a, dt, d) for a in y0]
        v = [torch.zeros(T, r, dtype=TDT[dt], device=d) for _ in widths]
        K.smlm_lora_forward_multi(y, [dev_t(a, dt, d) for a in x], tabs(Ad), tabs(Bd), plan, r, beta=1.0, v_out=v, **rank)
        for i in range(P):
            assert np.array_equal(to_np(v[i])[covered], vb[i]), f"v {i} defer {defer}"
            assert np.array_equal(to_np(y[i]), want[i][0]), f"y {i} defer {defer}"
        dA, dB = [[torch.full_like(a, 9.0) for a in w] for w in Ad], [[torch.full_like(b, 9.0) for b in w] for w in Bd]
        dx = [torch.empty(n, h, dtype=TDT[dt], device=d) for h, _ in widths]
        bplan = K.SegmentPlan(int32(tp), int32(ids), n, defer=defer)
        K.smlm_lora_backward_multi(dx, tabs(dA), tabs(dB), [dev_t(a, dt, d) for a in g], [dev_t(a, dt, d) for a in xb],
                                   [dev_t(a, dt, d) for a in vb], tabs(Ad), tabs(Bd), bplan, r, **rank)
        for i in range(P):
            gx, ga, gb = grads[i]
            assert np.array_equal(to_np(dx[i]), gx), f"dX {i} defer {defer}"
            for a in range(NA):
                assert np.array_equal(to_np(dA[i][a]), ga[a][:ranks[a]]), f"dA {i} {a}"
                assert np.array_equal(to_np(dB[i][a]), gb[a][:, :ranks[a]]), f"dB {i} {a}"


@pytest.mark.parametrize("r", [16, 64])
def test_inf_and_nan_stay_in_their_rows_and_columns(K, gpu_device, r):
    """Slots without a row multiply another row, columns past a rank other weights: neither must leak."""
    d, T, h = gpu_device, 3500, 1096
    x = torch.randn(T, h, device=d).half()
    x[0], x[64], x[3400] = float("inf"), float("nan"), float("-inf")
    A, B = [torch.randn(q, h, device=d).half() for q in (r, 8)], [torch.randn(72, q, device=d).half() for q in (r, 8)]
    A[1][3] = float("nan")
    int32 = lambda v: torch.tensor(v, dtype=torch.int32, device=d)
    v = torch.zeros(T, r, dtype=torch.float16, device=d)
    K.smlm_lora_forward_multi([torch.zeros(T, 72, dtype=torch.float16, device=d)], [x], [ptrs(A, d)], [ptrs(B, d)],
                              K.SegmentPlan(int32([0, 70, 3000, T]), int32([0, 1, 0]), T), r, v_out=[v],
                              adapter_rank=int32([r, 8]), packed_ranks=True)
    ok = torch.ones(T, dtype=torch.bool, device=d)
    ok[[0, 64, 3400]] = False
    mid = torch.zeros_like(ok)
    mid[70:3000] = True
    assert v[ok & ~mid].isfinite().all() and not v[~ok].isfinite().any()
    assert v[mid][:, 3].isnan().all() and v[mid][:, [0, 1, 2, 4, 5, 6, 7]].isfinite().all() and not v[mid][:, 8:].any()


@pytest.mark.parametrize("S", [9, 300])
@pytest.mark.parametrize("T,r,d_in", [(2100, 16, 520), (3100, 32, 72), (3100, 64, 520), (3100, 64, 2560)])
def test_scale_and_beta(K, gpu_device, T, r, d_in, S):
    """smlm_gemm: products of one slice store what they sum, scaled and added to beta y; the last one's slices are folded.
    With the plan built in the launch and beforehand; whole numbers, so both are exact."""
    from loquetier_amd import _lib as lib
    d, NA = gpu_device, 4
    g = torch.Generator().manual_seed(T + r)
    whole = lambda *s: torch.randint(-2, 3, s, generator=g).half()
    cut = [0] + sorted(int(c) for c in torch.randint(0, T - 5, (S - 1,), generator=g)) + [T - 5]
    x, y0, W = whole(T, d_in), whole(T, r), [whole(r, d_in) for _ in range(NA)]
    scale = torch.randint(1, 4, (S,), generator=g).float() / 2
    want = y0.clone()
    for i in range(S):
        q = slice(cut[i], cut[i + 1])
        want[q] = (0.5 * y0[q].double() + scale[i] * (x[q].double() @ W[i % NA].double().T)).half()
    xd, Wd, sd = x.to(d), [w.to(d) for w in W], scale.to(d)
    table, seg = ptrs([Wd[i % NA] for i in range(S)], d), torch.tensor(cut, dtype=torch.int32, device=d)
    need = lib.size_query("smlm_gemm_workspace_size", T, S, d_in, r)
    ws, got = torch.empty(need, dtype=torch.uint8, device=d), y0.to(d)
    rc = lib.load().smlm_gemm(got.data_ptr(), xd.data_ptr(), table.data_ptr(), seg.data_ptr(), ws.data_ptr(), need, T, S,
                              d_in, r, d_in, 0, lib.SMLM_DTYPE_F16, 0.5, sd.data_ptr(),
                              torch.cuda.current_stream(d).cuda_stream)
    assert rc == 0, lib.strerror(rc)
    planned = y0.to(d)
    K.smlm_gemm_planned(planned, xd, table, K.SegmentPlan(seg, None, T), seg_scale=sd, beta=0.5)
    assert torch.equal(got.cpu(), want) and torch.equal(planned.cpu(), want)


@pytest.mark.parametrize("S", [200, 300])
def test_weight_rows_out_of_the_block_kernels_reach(K, gpu_device, S):
    """Rows of 2 ** 25 elements and more go to the wide kernel: beyond 256 segments, with k in three, its two groups of
    waves a workgroup may not pair the slices up.  Whole numbers, so any order of the sums gives the same bits."""
    from loquetier_amd import _lib as lib
    d, T, d_in, d_out, ld = gpu_device, 2100, 1536, 16, 2 ** 25 + 8
    g = torch.Generator().manual_seed(1)
    whole = lambda *s: torch.randint(-3, 4, s, generator=g).half().to(d)
    seg = (torch.arange(S + 1) * T // S).to(torch.int32).to(d)
    x, w = whole(T, d_in), whole(d_out, d_in)
    far = torch.empty((d_out - 1) * ld + d_in, dtype=torch.float16, device=d)
    far.as_strided((d_out, d_in), (ld, 1)).copy_(w)
    need = lib.size_query("smlm_gemm_workspace_size", T, S, d_in, d_out)
    ws = torch.full((need + T * d_out * 4,), 0xA5, dtype=torch.uint8, device=d)
    y, table = torch.empty(T, d_out, dtype=torch.float16, device=d), ptrs([far] * S, d)
    rc = lib.load().smlm_gemm(y.data_ptr(), x.data_ptr(), table.data_ptr(), seg.data_ptr(), ws.data_ptr(), need,
                              T, S, d_in, d_out, ld, 0, lib.SMLM_DTYPE_F16, 0.0, None,
                              torch.cuda.current_stream(d).cuda_stream)
    assert rc == 0, lib.strerror(rc)
    assert torch.equal(y, (x.double() @ w.double().T).half()) and bool((ws[need:] == 0xA5).all())
