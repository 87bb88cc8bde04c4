"""Expanding products of smlm_gemm whose workgroups find their tiles without a plan: bit for bit what the same product
over a finished plan gives, at the edges of its range -- segments up to a thread each, empty and repeated ones, more tiles
than rows of workgroups, k and columns short of a step and of a chunk, beta and scale, rows no segment covers."""
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
    "rounds": ([1] * 256, 256, 16, 1032, 0),        # a tile a segment: more than the launch has rows of workgroups
    "planned-257": ([2] * 257, 9, 16, 1032, 0),     # one segment too many: the plan's launch
    "equal-width": ([5, 6], 2, 8, 24, 0),
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
