"""Saved tensors that come back from a program's own hooks in another form than they were saved in: torch hands on whatever
the hook returns, and the kernels read rows end to end, so both host paths must refuse the same forms in the same words."""
import pytest
import torch

from test_gpu_host_path import _layer, general, host, table  # noqa: F401

pytestmark = pytest.mark.gpu

# (strided: elements apart in memory; wider: more bytes than the kernels would read; elsewhere: on the host)
FORMS = {"strided": lambda t: t.t().contiguous().t() if t.dim() == 2 and min(t.shape) > 1 else torch.stack([t, t], -1)[..., 0],
         "wider": lambda t: t.double(), "elsewhere": lambda t: t.cpu()}


def hooks(which, change):
    count = iter(range(1 << 30))
    return torch.autograd.graph.saved_tensors_hooks(
        lambda t: (next(count), t), lambda p: change(p[1]) if p[0] == which else p[1])


def refusals(host, run, which, change):  # noqa: F811
    """What the backward of run() raises natively and through the general path."""
    texts = []
    for path in (None, general(host)):
        if path:
            path.__enter__()
        try:
            with hooks(which, change):
                out = run()
            with pytest.raises(RuntimeError) as e:
                out.backward(torch.ones_like(out))
            texts.append(str(e.value))
        finally:
            if path:
                path.__exit__(None, None, None)
    return texts


def rms_case(d):
    from loquetier_amd.kernel_utils import rms_norm
    x, w = (torch.randn(*s, device=d).to(torch.bfloat16).requires_grad_(True) for s in ((24, 64), (64,)))
    return lambda: rms_norm.apply(x, w, 1e-5)


def add_case(d):
    from loquetier_amd.kernel_utils import add_lora
    A, B, x = (torch.randn(*s, device=d).to(torch.bfloat16).requires_grad_(True) for s in ((16, 64), (72, 16), (40, 64)))
    s = torch.tensor([0, 30, 40], dtype=torch.int32, device=d)
    wa, wb = table([A, A], d), table([B, B], d)
    return lambda: add_lora.apply((40, 72), x, wa, wb, s, 16, 30, [0, 30], A, B)


def layer_case(d):
    from loquetier_amd.kernel_utils import BatchLenInfo
    ctx, layer = _layer(d, "bf16", [16, 16], 16, 64, 72, 3)
    layer.set_trainable([0])
    blen = BatchLenInfo([(1, 30)], [], 10, [], d)
    segment = torch.tensor([0, 30] + list(range(31, 41)), dtype=torch.int32, device=d)
    x = torch.randn(40, 64, device=d).to(torch.bfloat16).requires_grad_(True)

    def run():
        ctx.update(blen=blen, lora_ids=[0] + [1] * 10, lora_len=None, segment=segment, train_idx=[0])
        return layer(x)
    return run


# saved tensor, form, words of the refusal.  (rms_norm's dx takes the strides of x, dw those of w; the layer's base linear
# saves its weight first.)
CASES = [(rms_case, 0, "strided", "must be contiguous"), (rms_case, 0, "wider", "must share one dtype"),
         (rms_case, 1, "wider", "must share one dtype"), (rms_case, 2, "wider", "float32 with one entry per row"),
         (rms_case, 2, "elsewhere", "rms must be a CUDA tensor"),
         (add_case, 0, "strided", "x must be contiguous"), (add_case, 0, "wider", "must share one dtype"),
         (add_case, 1, "strided", "v must be a contiguous"), (add_case, 1, "wider", "must share one dtype"),
         *[(add_case, w, form, "the weights must share dy's dtype and device") for w in (2, 3) for form in ("wider", "elsewhere")],
         *[(add_case, w, "strided", "laid out as they were saved") for w in (2, 3)],
         (add_case, 0, "elsewhere", "must be a CUDA tensor"), (add_case, 1, "elsewhere", "must share one device"),
         (layer_case, 1, "strided", "x must be contiguous"), (layer_case, 1, "wider", "must share one dtype"),
         (layer_case, 2, "strided", "v must be a contiguous"), (layer_case, 2, "wider", "must share one dtype"),
         (layer_case, 2, "elsewhere", "must share one device")]


@pytest.mark.parametrize("case,which,form,text", CASES, ids=[f"{c[0].__name__}-{c[1]}-{c[2]}" for c in CASES])
def test_refused_alike(host, gpu_device, case, which, form, text):  # noqa: F811
    native, python = refusals(host, case(gpu_device), which, FORMS[form])
    assert native == python and text in native
