"""Host tables put on the device by launches (smlm_put_words): the edges of a launch's words, tables that are copied
instead, replays of a captured call, refused arguments."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(gpu_device):
    from loquetier_amd import _lib
    from loquetier_amd.ops import _kernels
    _lib.load()
    return _kernels


@pytest.mark.parametrize("n64,n32", [(0, 0), (0, 1), (1, 0), (64, 0), (63, 2), (64, 1), (448, 0), (448, 1), (900, 7),
                                     (1792, 0), (1792, 1), (3000, 11)])
def test_words_arrive(K, gpu_device, n64, n32):
    big = [(i * 0x9E3779B97F4A7C15) % (1 << 63) for i in range(n64)]
    small = [i * 7919 - (1 << 30) for i in range(n32)]
    a, b = K.put_ints(gpu_device, big, small)
    assert a.dtype == torch.int64 and b.dtype == torch.int32 and a.is_contiguous() and b.is_contiguous()
    assert a.tolist() == big and b.tolist() == small


def test_replays_write_the_captured_words(K, gpu_device):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        a, b = K.put_ints(gpu_device, [1 << 40, 3], [5, 6, 7])
        c = a + 1
    for _ in range(3):
        a.zero_(), b.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert a.tolist() == [1 << 40, 3] and b.tolist() == [5, 6, 7] and c.tolist() == [(1 << 40) + 1, 4]


def test_bad_arguments(K, gpu_device):
    from loquetier_amd import _lib
    buf = torch.zeros(16, dtype=torch.uint8, device=gpu_device)
    put, data = _lib.load().smlm_put_words, bytes(16)
    assert put(buf.data_ptr(), data, 6, None) == -3 and put(buf.data_ptr() + 2, data, 4, None) == -3
    assert put(None, data, 4, None) == -1 and put(buf.data_ptr(), None, 4, None) == -1
    assert put(None, None, 0, None) == 0
