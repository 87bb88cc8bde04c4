"""Backward of RMSNorm at the edges of its launch: rows of one wave's pieces and of 1024 threads', the change to two
pieces a thread (8200 columns), row counts around the workgroups' turns, the fold's 16, 32 and 64 columns a
workgroup.  Exact inputs (unit-magnitude rows, dyadic w and g, power-of-two widths: every term is exact in float) equal
the oracle; other widths within the bars of the RMSNorm parity tests."""
import numpy as np
import pytest
import torch

from test_gpu_rms_norm import K, ULP, dev_t, run_fwd, to_np, within_ulps  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["fp16", "bf16"])
@pytest.mark.parametrize("rows,cols", [(1, 8), (2, 64), (513, 64), (1025, 512), (5, 8192), (515, 16384), (6, 8200), (515, 72), (40, 2048),
                                       (40, 2056), (40, 4096), (40, 4104), (1300, 12288),
                                       (511, 8192), (512, 8192), (1023, 4096), (1025, 3072), (257, 8208)])
def test_backward(K, oracle, gpu_device, dt, rows, cols):
    exact = cols & (cols - 1) == 0
    rng = np.random.default_rng(rows * 31 + cols)
    if exact:
        x = np.where(rng.random((rows, cols)) < 0.5, -1.0, 1.0).astype(np.float32)
        w = (rng.integers(-8, 9, cols) / 4.0).astype(np.float32)
        g = (rng.integers(-8, 9, (rows, cols)) / 8.0).astype(np.float32)
    else:
        x = oracle.round_to(rng.standard_normal((rows, cols)), dt)
        w = oracle.round_to(1.0 + 0.2 * rng.standard_normal(cols), dt)
        g = oracle.round_to(rng.standard_normal((rows, cols)), dt)
    _, rms, (xd, wd, m) = run_fwd(K, x, w, 0.0, dt, gpu_device)
    dx, dw = torch.empty_like(xd), torch.empty_like(wd)
    K.rms_norm_backward(dx, dw, dev_t(g, dt, gpu_device), xd, wd, m)
    want_dx, want_dw = oracle.rms_norm_bwd(g, x, w, rms, dt)
    if exact:
        assert np.array_equal(to_np(dx), want_dx) and np.array_equal(to_np(dw), want_dw)
    else:
        assert within_ulps(to_np(dx), want_dx, dt, 2)
        # dw sums `rows` terms in float in another order than the oracle's double
        assert np.all(np.abs(to_np(dw) - want_dw) <= 1.5 * ULP[dt] * np.maximum(np.abs(want_dw), np.sqrt(rows) * 2.0 ** -6))


@pytest.mark.parametrize("cols", [72, 512, 3000, 8200])
def test_backward_infinite_gradient(K, gpu_device, cols):
    # an infinite g in the first column makes every dx of its row infinite, with the sign the formula gives it, and its
    # own NaN; threads beyond the row's last column add nothing to the dot
    x = torch.ones(3, cols)
    g = torch.full((3, cols), 0.5)
    g[1, 0] = float("inf")
    xd, gd = (t.to(torch.bfloat16).to(gpu_device) for t in (x, g))
    w, rms = torch.ones(cols, dtype=torch.bfloat16, device=gpu_device), torch.ones(3, device=gpu_device)
    dx, dw = torch.empty_like(xd), torch.empty_like(w)
    K.rms_norm_backward(dx, dw, gd, xd, w, rms)
    got = dx.float().cpu()
    assert torch.isnan(got[1, 0]) and (got[1, 1:] == float("-inf")).all()
    assert (got[[0, 2]].abs() < 2.0 ** -20).all()  # g - x * mean(g * x), 1 / cols rounded to float
    assert dw[0].item() == float("inf") and (dw[1:].float() == 1.5).all()
