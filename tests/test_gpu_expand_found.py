"""Expanding products of smlm_gemm whose workgroups find their tiles without a plan: bit for bit what the same product
over a finished plan gives, at the edges of its range -- segments up to a thread each, empty and repeated ones, more items
than workgroups, k and columns short of a step and of a chunk, beta and scale, rows no segment covers."""
import numpy as np
import pytest
import torch

from test_gpu_parity import TDT, K, ptrs  # noqa: F401

pytestmark = pytest.mark.gpu

CASES = {
    # lengths of the segments, adapters, d_in, d_out, first row
    "one-row": ([1], 1, 8, 16, 0),
    "one-segment": ([700], 1, 16, 4104, 0),
    "ragged": ([0, 33, 1, 16, 0, 17, 90, 5, 64, 1], 3, 16, 11008, 3),
    "k-40": ([20, 7, 7, 100], 2, 40, 520, 1),
    "k-64": ([9] * 14, 5, 64, 512, 0),
    "k-72": ([3, 50, 31], 2, 72, 1000, 0),
    "k-128": ([1] * 100, 7, 128, 264, 5),
    "decode-256": ([1] * 256, 32, 16, 4096, 0),
    "rounds": ([1] * 256, 256, 16, 1032, 0),        # a tile a segment: several turns a workgroup
    "planned-257": ([2] * 257, 9, 16, 1032, 0),     # one segment too many: the plan's launch
    "equal-width": ([5, 6], 2, 8, 24, 0),
    "128-wide": ([1] * 128, 40, 16, 12296, 0),
    "129-wide": ([1] * 129, 40, 16, 12296, 0),
    "256-13-chunks": ([1] * 256, 40, 16, 6152, 0),
    "70-chunks": ([40] * 30, 30, 16, 35336, 2),         # more column chunks than lists are priced
}


@pytest.mark.parametrize("dt", ["fp16", "bf16"])
@pytest.mark.parametrize("name", CASES)
def test_equals_the_planned_product(K, gpu_device, name, dt):
    from loquetier_amd import _lib as lib
    lens, NA, d_in, d_out, first = CASES[name]
    d, S = gpu_device, len(lens)
    g = torch.Generator().manual_seed(5)
    seg = torch.tensor([0] + lens).cumsum(0) + first
    T = int(seg[-1]) + 4
    seg = seg.to(torch.int32).to(d)
    randn = lambda *s: torch.randn(*s, generator=g).to(TDT[dt]).to(d)
    x, y0, W = randn(T, d_in), randn(T, d_out), [randn(d_out, d_in) for _ in range(NA)]
    table = ptrs([W[(7 * i) % NA] for i in range(S)], d)
    scale = (torch.rand(S, generator=g) + 0.5).to(d)
    plan = K.SegmentPlan(seg, None, T)
    stream = torch.cuda.current_stream(d).cuda_stream
    code = lib.SMLM_DTYPE_F16 if dt == "fp16" else lib.SMLM_DTYPE_BF16
    need = lib.size_query("smlm_gemm_workspace_size", T, S, d_in, d_out)
    ws = torch.empty(need, dtype=torch.uint8, device=d)
    for beta, sc in ((0.0, None), (0.75, scale)):
        want, got = y0.clone(), y0.clone()
        K.smlm_gemm_planned(want, x, table, plan, seg_scale=sc, beta=beta)
        rc = lib.load().smlm_gemm(got.data_ptr(), x.data_ptr(), table.data_ptr(), seg.data_ptr(), ws.data_ptr(), need, T, S,
                                  d_in, d_out, d_in, 0, code, beta, None if sc is None else sc.data_ptr(), stream)
        assert rc == 0, lib.strerror(rc)
        assert torch.equal(got, want)
        outside = list(range(first)) + list(range(int(seg[-1]), T))
        assert torch.equal(got[outside], y0[outside])


def _colliding(base, n, slots, per):
    """Addresses in `n` sixteenths of bytes from `base` of which `per` share both hash slots of first_equal_pair."""
    at = (np.uint64(base >> 4) + np.arange(n, dtype=np.uint64))
    with np.errstate(over="ignore"):
        h = (at * np.uint64(0x9E3779B97F4A7C15)) ^ (at * np.uint64(0xC2B2AE3D27D4EB4F))
    both = (h >> np.uint64(40)) % np.uint64(slots) * np.uint64(slots) + (h >> np.uint64(24)) % np.uint64(slots)
    order = np.argsort(both, kind="stable")
    run = np.flatnonzero(both[order[:-per + 1]] == both[order[per - 1:]])
    first = run[np.concatenate([[True], np.diff(run) >= per])]
    return [int(at[order[i + j]]) << 4 for i in first[:250 // per] for j in range(per)]


def test_addresses_that_collide_twice(K, gpu_device):
    """Segments whose address loses its slot in both rounds of the numbering: three of every four here, each address
    twice.  The product equals the one over a plan, which sorts the addresses."""
    from loquetier_amd import _lib as lib
    d, d_in, d_out = gpu_device, 16, 64
    g = torch.Generator().manual_seed(3)
    pool = torch.randn(1 << 25, generator=g).half().to(d)  # the weights overlap in it
    some = _colliding(pool.data_ptr(), pool.numel() // 8 - d_in * d_out, 1024, 4)[:128]
    assert len(some) == 128
    table = torch.tensor(some + some[::-1], dtype=torch.int64, device=d)
    S = 256
    seg = torch.arange(S + 1, dtype=torch.int32, device=d)
    x, want, got = torch.randn(S, d_in, generator=g).half().to(d), *torch.zeros(2, S, d_out, dtype=torch.float16, device=d)
    K.smlm_gemm_planned(want, x, table, K.SegmentPlan(seg, None, S))
    need = lib.size_query("smlm_gemm_workspace_size", S, S, d_in, d_out)
    ws = torch.empty(need, dtype=torch.uint8, device=d)
    rc = lib.load().smlm_gemm(got.data_ptr(), x.data_ptr(), table.data_ptr(), seg.data_ptr(), ws.data_ptr(), need, S, S, d_in,
                              d_out, d_in, 0, lib.SMLM_DTYPE_F16, 0.0, None, torch.cuda.current_stream(d).cuda_stream)
    assert rc == 0, lib.strerror(rc)
    assert torch.equal(got, want)


def test_many_addresses_take_no_longer_than_the_planned_product(K, gpu_device):
    """256 one-row segments on as many addresses: several items a workgroup, and as many addresses
    as can be to tell apart.  The planned product does the same work plus the plan's launch, so its time is the bound;
    half as much again for what two timings differ by (140 us against 20 with the search done again for every tile)."""
    from loquetier_amd import _lib as lib
    d, S, d_in, d_out, n = gpu_device, 256, 16, 6144, 20
    x, W = torch.randn(S, d_in, device=d).half(), torch.randn(S, d_out, d_in, device=d).half()
    seg, table = torch.arange(S + 1, dtype=torch.int32, device=d), ptrs(list(W), d)
    y = torch.empty(S, d_out, dtype=torch.float16, device=d)
    need = lib.size_query("smlm_gemm_workspace_size", S, S, d_in, d_out)
    ws = torch.empty(need, dtype=torch.uint8, device=d)
    code, stream, lib_ = lib.SMLM_DTYPE_F16, torch.cuda.current_stream(d).cuda_stream, lib.load()
    plan = torch.empty(K.SegmentPlan.nbytes(S, S), dtype=torch.uint8, device=d)

    def found():
        return lib_.smlm_gemm(y.data_ptr(), x.data_ptr(), table.data_ptr(), seg.data_ptr(), ws.data_ptr(), need, S, S, d_in,
                              d_out, d_in, 0, code, 0.0, None, stream)

    def planned():
        return lib_.smlm_plan_build(plan.data_ptr(), plan.numel(), seg.data_ptr(), table.data_ptr(), lib.SMLM_KEY_PTR, S, S,
                                    stream) or \
            lib_.smlm_gemm_planned(y.data_ptr(), x.data_ptr(), table.data_ptr(), S, plan.data_ptr(), ws.data_ptr(), need, S,
                                   S, d_in, d_out, d_in, 0, code, 0.0, None, stream)

    def time(call):
        best = []
        for _ in range(7):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(n):
                assert call() == 0
            b.record()
            b.synchronize()
            best.append(a.elapsed_time(b))
        return sorted(best)[1]
    time(found), time(planned)
    assert time(found) <= 1.5 * time(planned)
