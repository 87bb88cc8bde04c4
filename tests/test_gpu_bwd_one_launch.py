"""dX and the weight gradients in one launch (bwd_tail_kernel) against the stages issued one by one, which launch each for
itself: the same bits, at every kernel the launch is made of, and rows past the plan cleared either way.  Which of the two a
call takes is read off its graph: the launches it records."""
import ctypes

import pytest
import torch

from test_gpu_parity import K, dev_t, ptrs  # noqa: F401

pytestmark = pytest.mark.gpu


def launches(call):
    """Kernels that call() launches (recorded, not run)."""
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    n = ctypes.c_size_t(0)
    assert ctypes.CDLL("libamdhip64.so.7").hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("drop", [0.0, 0.25], ids=["plain", "dropout"])
@pytest.mark.parametrize("r", [8, 24, 40, 64, 72, 128, 136])
@pytest.mark.parametrize("lens,NA,dims,joint", [
    ([5], 1, [(64, 1032)], True), ([40, 33, 9], 4, [(264, 1160), (72, 2056)], True), ([300, 250], 2, [(512, 1032)], True),
    ([400], 1, [(200, 1288)], True), ([16] * 70, 40, [(192, 1024), (64, 1096)], True),
    ([70, 9], 2, [(264, 520), (72, 136)], False)],   # (dV is not folded: dX's launch leaves what the gradients read)
    ids=["tiny", "one-wave", "four-waves", "four-waves-one-adapter", "many", "not-folded"])
def test_one_launch_equals_stages(K, gpu_device, lens, NA, dims, joint, r, drop):  # noqa: F811
    d, dt = gpu_device, torch.bfloat16
    g = torch.Generator(d).manual_seed(r + len(lens))
    rand = lambda *s: torch.randn(*s, generator=g, device=d).to(dt)
    n, extra = sum(lens), 7
    bounds = [0]
    for l in lens:
        bounds.append(bounds[-1] + l)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=d)
    plan = K.SegmentPlan(i32(bounds), i32([i % NA for i in range(len(lens))]), n)
    x, gy = [rand(n, h) for h, _ in dims], [rand(n, o) for _, o in dims]
    v = [rand(n, r) for _ in dims]
    A, B = [[rand(r, h) for _ in range(NA)] for h, _ in dims], [[rand(o, r) for _ in range(NA)] for _, o in dims]
    ta, tb = [ptrs(a, d) for a in A], [ptrs(b, d) for b in B]
    scale = torch.rand(len(lens), generator=g, device=d)
    spec = None
    if drop:
        bits = torch.randint(0, 256, (K.DropoutSpec.mask_nbytes(n, [h for h, _ in dims]),), generator=g, device=d,
                             dtype=torch.uint8)
        p = torch.full((len(lens),), drop, device=d)
        p[::3] = 0.0
        spec = K.DropoutSpec(p, n, 3, 5, bits)
    results, counts = [], []
    for stages in ((0,), (1, 2, 4), (1, 6)):
        dx = [torch.full((n + extra, h), 7.0, dtype=dt, device=d) for h, _ in dims]
        dA, dB = [[torch.full_like(a, 7.0) for a in w] for w in A], [[torch.full_like(b, 7.0) for b in w] for w in B]
        da, db = [ptrs(a, d) for a in dA], [ptrs(b, d) for b in dB]
        ws = K.Workspace(d)

        def call():
            for st in stages:
                K.smlm_lora_backward_multi(dx, da, db, gy, x, v, ta, tb, plan, r, scale, dropout=spec, workspace=ws,
                                           stages=st, zero_dx_tail=True)
        call()
        counts.append(launches(call))
        results.append([*dx, *[t for w in dA + dB for t in w]])
    assert counts[1] - counts[0] == (1 if joint else 0) and counts[2] == counts[0]
    for other in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))
    assert not any(t[n:].any() for t in results[0][:len(dims)])
    assert all(torch.isfinite(t.float()).all() for t in results[0])
