"""The scales of segments and train partitions in one launch (smlm_segment_scales) against the tensor expressions."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from loquetier_amd import _lib
    from loquetier_amd.ops import _kernels
    _lib.load()
    return _kernels


@pytest.mark.parametrize("S,P", [(1, 0), (1, 1), (2, 5), (255, 3), (256, 256), (257, 700), (1000, 4)])
def test_against_tensor_expressions(K, gpu_device, S, P):
    g = torch.Generator().manual_seed(S + P)
    n = 13
    table = torch.randn(n, generator=g).to(gpu_device)
    ids = torch.randint(-n, n, (S,), generator=g, dtype=torch.int32)   # (negative: from the end)
    lens = torch.randint(0, 4, (S,), generator=g)                      # (empty segments too)
    segment = torch.cat([torch.zeros(1, dtype=torch.int64), lens.cumsum(0)]).to(torch.int32)
    starts = torch.randint(0, int(segment[-1]) + 2, (P,), generator=g, dtype=torch.int32).sort()[0]
    ids, segment, starts = ids.to(gpu_device), segment.to(gpu_device), starts.to(gpu_device)
    want_seg = (torch.searchsorted(segment, starts, right=True) - 1).clamp_(0, S - 1)
    want = table[ids.long()]
    scale, part_seg, part = K.segment_scales(ids, table, segment, starts)
    assert torch.equal(scale, want) and torch.equal(part_seg, want_seg) and torch.equal(part, want[want_seg])
    assert part_seg.dtype == torch.int64
    assert torch.equal(K.segment_scales(ids, segment=segment, starts=starts)[1], want_seg)
    again = K.segment_scales(ids, table, part_seg=want_seg)
    assert torch.equal(again[0], want) and torch.equal(again[2], want[want_seg])
    alone = K.segment_scales(ids, table)
    assert torch.equal(alone[0], want) and alone[1] is None and alone[2] is None


def test_ids_past_the_table(K, gpu_device):
    ids = torch.tensor([0, 2, 3, -4, 1 << 30], dtype=torch.int32, device=gpu_device)
    table = torch.tensor([2.0, 3.0, 4.0], device=gpu_device)
    assert K.segment_scales(ids, table)[0].tolist() == [2.0, 4.0, 1.0, 1.0, 1.0]
    with pytest.raises(RuntimeError):
        K.segment_scales(ids, table.double())
    with pytest.raises(RuntimeError):
        K.segment_scales(ids, table, segment=ids, starts=ids)
