"""Keep bits in the order dX and the weight gradients read them, two slots of a tile to a load: partly filled tiles whose
pairs of slots lack one row or both, rows of the mask of an odd number of bytes, a mask at an odd address, rows that are not
dropped beside dropped ones, one-wave and four-wave weight gradients, one and two blocks of 64 ranks.  p = 1/2 doubles what
is kept and dyadic inputs stay exact, so all results must equal the oracle's bit for bit, with the caller's bits and with
bits made anew."""
import numpy as np
import pytest
import torch

from test_gpu_dropout import K, dev_t, dyadic, row_probs, run_backward  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0, 1, None], ids=["aligned", "odd-address", "made-anew"])
@pytest.mark.parametrize("h_in", [8, 192, 200, 584])   # mask rows of 1, 24, 25 and 73 bytes
@pytest.mark.parametrize("r", [16, 64, 72])
@pytest.mark.parametrize("tp", [[0, 1, 6, 19, 42, 97], [0, 3, 300, 305, 318, 640]], ids=["one-wave", "four-waves"])
# (1032 columns of dY are summed in two: the fold of dV then turns the bits, and dX shares the gradients' launch)
@pytest.mark.parametrize("h_out", [72, 1032], ids=["turned-alone", "turned-in-fold"])
def test_backward_keep_bits(K, oracle, gpu_device, h_out, tp, r, h_in, shift):  # noqa: F811
    d, dt, n_rows = gpu_device, "bf16", tp[-1]
    part_ad, ad_p = [2, 0, 1, 2, 0], [0.5, 0.5, 0.0]
    rows = n_rows - 5   # the last five keep everything
    rng = np.random.default_rng(n_rows + h_in)
    x, g = dyadic(rng, (n_rows, h_in), 4, 4), dyadic(rng, (n_rows, h_out), 4, 4)
    A = [dyadic(rng, (r, h_in), 2, 16) for _ in ad_p]
    B = [dyadic(rng, (h_out, r), 2, 4) for _ in ad_p]
    seg_p = np.array([ad_p[a] for a in part_ad], np.float32)
    rp = row_probs(tp, seg_p, n_rows, rows)
    mask = None
    if shift is not None:
        keep = np.packbits(oracle.dropout_mask(rows, h_in, rp[:rows], 21, 6), axis=1, bitorder="little")
        buf = torch.full((n_rows * (h_in // 8) + 4,), 0xAA, dtype=torch.uint8, device=d)
        mask = buf[shift: shift + n_rows * (h_in // 8)]
        mask[: keep.size].copy_(torch.from_numpy(keep.reshape(-1)))

    class Spec(K.DropoutSpec):  # (the Python call wants every row covered, the C call does not)
        def struct(self, plan, widths):
            c = super().struct(plan, widths)
            c.rows = rows
            return c

    spec = Spec(torch.from_numpy(seg_p).to(d), n_rows, 21, 6, mask_bits=mask)
    xdrop = oracle.dropout_rows(x, rp, 21, 6, dt)
    _, vo = oracle.add_lora_forward(xdrop, [A[a] for a in part_ad], [B[a] for a in part_ad], tp, h_out, dt)
    dx, dA, dB = run_backward(K, d, dt, x, A, B, g, tp, part_ad, r, spec, dev_t(vo, dt, d))
    gx, ga, gb = oracle.add_lora_backward(g, xdrop, A, B, tp, part_ad, dt)
    assert np.array_equal(dx[:n_rows], oracle.dropout_rows(gx, rp, 21, 6, dt))
    for a in range(3):
        assert np.array_equal(dA[a], ga[a]) and np.array_equal(dB[a], gb[a])
