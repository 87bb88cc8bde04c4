"""Keep bits the shrinks leave behind under dropout, and the x they multiply: rows of the mask that cannot be stored two
or four bytes at a time (odd and even widths of the mask, a mask at an odd address), p of 0, 1/2 and 1, rows that are not
dropped in the same tile, on every shrink kernel that drops, with the plan built beforehand and in the launch.  p = 1/2
doubles what is kept, so dyadic inputs stay exact and v must equal the oracle bit for bit."""
import numpy as np
import pytest
import torch

from test_gpu_dropout import TDT, dev_t, dyadic, ptrs, row_probs, to_np

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from loquetier_amd import _lib
    from loquetier_amd.ops import _kernels
    _lib.load()
    return _kernels


@pytest.mark.parametrize("defer", [False, True], ids=["planned", "self-planned"])
@pytest.mark.parametrize("shift", [0, 1, 2], ids=["aligned", "odd-address", "even-address"])
@pytest.mark.parametrize("h_in", [2056, 2064, 2080, 2176])   # mask rows of 257, 258, 260 and 272 bytes
@pytest.mark.parametrize("T,r", [(70, 16), (70, 64), (150, 64), (800, 32), (1600, 128)],
                         ids=["single", "single-64", "blocks-64", "blocks-32", "blocks-128"])
def test_keep_bits(K, oracle, gpu_device, T, r, h_in, shift, defer):
    d, dt = gpu_device, "bf16"
    rng = np.random.default_rng(T + h_in)
    train = T - 20
    seg = [0, train // 3, train // 2, train, T - 3, T]
    ids, ad_p = [0, 1, 2, 0, 3], [0.5, 0.0, 1.0, 0.5]
    x = dyadic(rng, (T, h_in), 4, 4)
    A = [dyadic(rng, (r, h_in), 2, 64) for _ in range(4)]
    xd, Ad = dev_t(x, dt, d), [dev_t(a, dt, d) for a in A]
    B = dev_t(np.zeros((64, r), np.float32), dt, d)
    seg_p = np.array([ad_p[i] for i in ids], np.float32)
    rp = row_probs(seg, seg_p, T, train)
    n_bits = K.DropoutSpec.mask_nbytes(train, h_in)
    buf = torch.full((n_bits + 4,), 0xAA, dtype=torch.uint8, device=d)
    spec = K.DropoutSpec(torch.from_numpy(seg_p).to(d), train, 99, 7, mask_bits=buf[shift: shift + n_bits])
    plan = K.SegmentPlan(torch.tensor(seg, dtype=torch.int32, device=d),
                         torch.tensor(ids, dtype=torch.int32, device=d), T, defer=defer)
    y, v = torch.zeros(T, 64, dtype=TDT[dt], device=d), torch.zeros(T, r, dtype=TDT[dt], device=d)
    K.smlm_lora_forward(y, xd, ptrs(Ad, d), ptrs([B] * 4, d), plan, r, v_out=v, dropout=spec)
    got = buf.cpu().numpy()
    keep = np.packbits(oracle.dropout_mask(train, h_in, rp[:train], 99, 7), axis=1, bitorder="little")
    bits = got[shift: shift + n_bits].reshape(train, h_in // 8)
    on = rp[:train] > 0
    assert np.array_equal(bits[on], keep[on]) and np.all(bits[~on] == 0xAA)
    assert np.all(got[:shift] == 0xAA) and np.all(got[shift + n_bits:] == 0xAA)
    xdrop = oracle.dropout_rows(x, rp, 99, 7, dt)
    _, vo = oracle.lora_fused(np.zeros((T, 64), np.float32), xdrop, [A[j] for j in ids],
                              [np.zeros((64, r), np.float32)] * 5, seg, None, 1.0, dt)
    assert np.array_equal(to_np(v), vo)
