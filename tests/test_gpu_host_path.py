"""The native host path against the Python functions it stands before: the same bits, the same refusals, and the forms of
a call it must leave to them (hooks on saved tensors, functorch transforms, forward-mode tangents, tracing, subclasses)."""
import concurrent.futures
import contextlib

import pytest
import torch

from loquetier_amd import _lib

pytestmark = pytest.mark.gpu
DT = {"fp16": torch.float16, "bf16": torch.bfloat16}


@pytest.fixture(scope="module")
def host(gpu_device):
    from loquetier_amd.ops import _kernels
    _lib.load()
    return _kernels._host()


@contextlib.contextmanager
def general(host):
    """Every native function declines: the Python functions take the calls."""
    kept = {n: getattr(host, n) for n in ("rms_norm", "add_lora", "fused_add_lora", "forward")}
    try:
        for n in kept:
            setattr(host, n, (lambda *a: False) if n == "forward" else (lambda *a: None))
        yield
    finally:
        for n, f in kept.items():
            setattr(host, n, f)


def same(a, b):
    assert len(a) == len(b)
    for p, q in zip(a, b):
        assert (p is None) == (q is None)
        if p is not None:
            assert p.dtype == q.dtype and p.shape == q.shape and torch.equal(p, q)


@contextlib.contextmanager
def taken(host, by):
    """The native function `by` takes every call it is given within the block, and is given one."""
    native, answers = getattr(host, by), []

    def watched(*args):
        answers.append(native(*args))
        return answers[-1]
    setattr(host, by, watched)
    try:
        yield
    finally:
        setattr(host, by, native)
    assert answers and not any(a is None or a is False for a in answers)


def both(host, run, by):
    """run() natively, where the function `by` must take its calls, and through the general path."""
    with taken(host, by):
        native = run()
    with general(host):
        same(native, run())
    return native


def table(ts, d):
    return torch.tensor([t.data_ptr() for t in ts], dtype=torch.int64, device=d)


@pytest.mark.parametrize("dt", list(DT))
@pytest.mark.parametrize("rows,cols", [(1, 8), (37, 264), (300, 4096), (5, 20480)])
@pytest.mark.parametrize("need", ["both", "x", "w"])
def test_rms_norm(host, gpu_device, dt, rows, cols, need):
    from loquetier_amd.kernel_utils import rms_norm
    g = torch.Generator(gpu_device).manual_seed(rows)
    rand = lambda *s: torch.randn(*s, generator=g, device=gpu_device).to(DT[dt])
    x, w, up = rand(rows, cols).requires_grad_(need != "w"), rand(cols).requires_grad_(need != "x"), rand(rows, 2 * cols)

    def run():
        x.grad = w.grad = None
        o = rms_norm.apply(x, w, 1e-5)
        o.backward(up[:, ::2])       # (a gradient that is not contiguous)
        return o.detach(), x.grad, w.grad
    want = both(host, run, "rms_norm")
    for mode in (torch.no_grad, torch.inference_mode):
        with mode():
            same([rms_norm.apply(x, w, 1e-5)], want[:1])
    same([rms_norm.apply(x, w)], [rms_norm.apply(x, w, 1e-6)])


def test_rms_norm_forms_left_to_the_general_path(host, gpu_device):
    from loquetier_amd.kernel_utils import rms_norm
    x = torch.randn(6, 64, device=gpu_device, dtype=torch.bfloat16, requires_grad=True)
    w = torch.randn(64, device=gpu_device, dtype=torch.bfloat16, requires_grad=True)
    one = torch.ones_like(x)

    class mine(rms_norm):
        @staticmethod
        def forward(ctx, x, w, eps=1e-6):
            return rms_norm.forward(ctx, x, w, eps) * 0
    assert not mine.apply(x, w, 1e-5).any()
    packed, unpacked = [], []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.clone(),
                                                  lambda t: unpacked.append(t.shape) or t):
        o = rms_norm.apply(x, w, 1e-5)
    want = torch.autograd.grad(rms_norm.apply(x, w, 1e-5), (x, w), one)
    same(torch.autograd.grad(o, (x, w), one), want)
    assert len(packed) == len(unpacked) == 3
    o = rms_norm.apply(x, w, 1e-5)
    same(torch.autograd.grad(o, (x, w), one, retain_graph=True), want)
    torch.autograd.grad(o, (x, w), one)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(o, (x, w), one)
    z = x.detach().clone().requires_grad_(True)
    h = z * 1
    o = rms_norm.apply(h, w, 1e-5)
    h.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        o.backward(one)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda t: rms_norm.apply(t, w, 1e-5))(torch.stack([x.detach()] * 2))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: rms_norm.apply(t, w, 1e-5).float().sum())(x.detach())
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x.detach(), one)
        with pytest.raises((RuntimeError, NotImplementedError)):
            rms_norm.apply(dual, w.detach(), 1e-5)
    for bad, text in (((x.t(), w), "contiguous"), ((x.float(), w.float()), "No suitable kernel"),
                      ((x.cpu(), w), "CUDA tensor"), ((x, w[:32]), "column"), ((x[0], w), "2D")):
        with pytest.raises(RuntimeError, match=text):
            rms_norm.apply(*bad, 1e-5)


@pytest.mark.parametrize("dt", list(DT))
@pytest.mark.parametrize("tp,ids,tail", [([0, 40, 64], [0, 1], 8), ([0, 20, 20, 90], [1, 1, 0], 0), ([0, 700], [0], 100),
                                         ([0] + [5 * i for i in range(1, 301)], [i % 7 for i in range(300)], 3)],
                         ids=["two", "shared-and-empty", "one-long", "three-hundred"])
def test_add_lora(host, gpu_device, dt, tp, ids, tail):
    from loquetier_amd.kernel_utils import add_lora
    d, r, h_in, h_out = gpu_device, 16, 256, 320
    g = torch.Generator(d).manual_seed(tp[-1])
    rand = lambda *s: torch.randn(*s, generator=g, device=d).to(DT[dt])
    T, NA = tp[-1] + tail, max(ids) + 1
    A, B = [rand(r, h_in).requires_grad_(True) for _ in range(NA)], [rand(h_out, r).requires_grad_(True) for _ in range(NA)]
    x, up = rand(T, h_in).requires_grad_(True), rand(T, h_out)
    seg = tp + ([T] if tail else [])
    all_ids = ids + ([0] if tail else [])
    s = torch.tensor(seg, dtype=torch.int32, device=d)
    wa, wb = table([A[i] for i in all_ids], d), table([B[i] for i in all_ids], d)
    weights = [w for i in ids for w in (A[i], B[i])]

    def run():
        y = add_lora.apply((T, h_out), x, wa, wb, s, r, tp[-1], tp, *weights)
        grads = torch.autograd.grad(y, [x] + [w for i in sorted(set(ids)) for w in (A[i], B[i])], up)
        return [y.detach(), *grads]
    want = both(host, run, "add_lora")
    with torch.no_grad():
        same([add_lora.apply((T, h_out), x, wa, wb, s, r, tp[-1], tp, *weights)], want[:1])
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.clone(), lambda t: t):
        y = add_lora.apply((T, h_out), x, wa, wb, s, r, tp[-1], tp, *weights)
    assert len(packed) == 2 + len(weights)
    if len(set(ids)) == len(ids):  # (clones of a shared adapter are two adapters: their gradients are summed by autograd)
        same([torch.autograd.grad(y, x, up)[0]], want[1:2])
    with pytest.raises(RuntimeError):
        add_lora.apply((T, h_out), x[:-1], wa, wb, s, r, tp[-1], tp, *weights)


def _layer(d, dt, ranks, r, h_in, h_out, seed):
    from loquetier_amd.mixed_lora import MixedLoraContext, MixedLoraLinear, NamedLoraLayer, prepare_weight
    torch.manual_seed(seed)
    base = torch.nn.Linear(h_in, h_out, bias=False, device=d, dtype=DT[dt])
    base.weight.requires_grad_(False)
    pack = min(ranks) < r
    named = [NamedLoraLayer(f"a{i}", prepare_weight(torch.randn(q, h_in, device=d), r, DT[dt], d, 0, pack=pack),
                            prepare_weight(torch.randn(h_out, q, device=d), r, DT[dt], d, 1, pack=pack),
                            torch.nn.Identity(), 0.5 * (i + 1), q) for i, q in enumerate(ranks)]
    ctx = MixedLoraContext()
    return ctx, MixedLoraLinear(ctx, base, named, r, DT[dt], is_scaled=False, fused=True)


@pytest.mark.parametrize("dt", list(DT))
@pytest.mark.parametrize("ranks", [[16, 16, 16], [8, 16, 8]], ids=["one-rank", "packed"])
@pytest.mark.parametrize("lens,train,tail", [([40, 24], [1, 0], 7), ([30, 30, 12], [1, 1, 2], 0), ([600], [2], 40)])
def test_layers(host, gpu_device, dt, ranks, lens, train, tail):
    from loquetier_amd.kernel_utils import BatchLenInfo
    d, h_in, h_out = gpu_device, 512, 384
    ctx, layer = _layer(d, dt, ranks, 16, h_in, h_out, 3)
    layer.set_trainable(sorted(set(train)))
    T = sum(lens) + tail
    blen = BatchLenInfo([(1, l) for l in lens], [], tail, [], d)
    bounds = [0]
    for l in lens + [1] * tail:
        bounds.append(bounds[-1] + l)
    ids = train + [i % 3 for i in range(tail)]
    segment = torch.tensor(bounds, dtype=torch.int32, device=d)
    lens_t = torch.tensor(lens + [1] * tail, dtype=torch.int32, device=d)
    x = torch.randn(T, h_in, device=d).to(DT[dt]).requires_grad_(True)
    up = torch.randn(T, h_out, device=d).to(DT[dt])
    params = [p for p in layer.parameters() if p.requires_grad]

    def run(hooks=None):
        for p in params + [x]:
            p.grad = None
        ctx.update(blen=blen, lora_ids=ids, lora_len=lens_t, segment=segment, train_idx=train)
        with hooks or contextlib.nullcontext():
            y = layer(x)
        y.backward(up)
        return [y.detach().clone(), x.grad, *[p.grad for p in params]]
    # (gradients of two shapes are Python's; the forward below it is not)
    want = both(host, run, "fused_add_lora" if len({ranks[i] for i in train}) == 1 else "forward")
    assert all(g is not None for g in want)
    for _ in range(3):   # the tables of the gradients' addresses are kept: other blocks, the same values
        same(run(), want)
    packed = []
    same(run(torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t, lambda t: t)), want)
    assert packed
    with torch.no_grad():
        ctx.update(blen=blen, lora_ids=ids, lora_len=lens_t, segment=segment, train_idx=train)
        same([layer(x)], want[:1])


def test_streams_and_threads_at_once(host, gpu_device):
    """Four threads, a stream each, against the same calls one after the other."""
    from loquetier_amd.kernel_utils import add_lora, rms_norm
    d, r, T = gpu_device, 16, 300
    s = torch.tensor([0, 180, T], dtype=torch.int32, device=d)

    def inputs(seed):
        g = torch.Generator(d).manual_seed(seed)
        rand = lambda *n: torch.randn(*n, generator=g, device=d).to(torch.bfloat16)
        A, B = [rand(r, 1024).requires_grad_(True) for _ in range(2)], [rand(512, r).requires_grad_(True) for _ in range(2)]
        return rand(T, 1024).requires_grad_(True), rand(1024).requires_grad_(True), A, B, table(A, d), table(B, d), rand(T, 512)
    cases = [inputs(i) for i in range(4)]

    def run(case):
        x, w, A, B, wa, wb, up = case
        y = add_lora.apply((T, 512), rms_norm.apply(x, w, 1e-5), wa, wb, s, r, T, [0, 180, T], A[0], B[0], A[1], B[1])
        return [y.detach(), *torch.autograd.grad(y, [x, w, *A, *B], up)]
    want = [run(c) for c in cases]
    torch.cuda.synchronize()

    def work(case):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            outs = [run(case) for _ in range(8)]
        stream.synchronize()
        return outs
    with taken(host, "add_lora"), taken(host, "rms_norm"), concurrent.futures.ThreadPoolExecutor(4) as pool:
        for outs, ref in zip(pool.map(work, cases), want):
            for o in outs:
                same(o, ref)


def test_what_is_refused_stays_refused(host, gpu_device):
    from loquetier_amd.ops import _kernels as K
    d, dt = gpu_device, torch.bfloat16
    x, y = torch.randn(20, 64, device=d).to(dt), torch.zeros(20, 128, device=d, dtype=dt)
    A, B = torch.randn(8, 64, device=d).to(dt), torch.randn(128, 8, device=d).to(dt)
    plan = K.SegmentPlan(torch.tensor([0, 20], dtype=torch.int32, device=d), torch.zeros(1, dtype=torch.int32, device=d), 20)
    ta, tb, ok = table([A], d), table([B], d), {}
    calls = [((y, x[:10], ta, tb, plan, 8), ok), ((y.float(), x, ta, tb, plan, 8), ok), ((y, x.t(), ta, tb, plan, 8), ok),
             ((y, x, ta.int(), tb, plan, 8), ok), ((y, x.cpu(), ta, tb, plan, 8), ok), ((y, x, ta, tb, plan, 12), ok),
             ((y, x, ta, tb, plan, 8), dict(seg_scale=torch.ones(3, device=d))),
             ((y, x, ta, tb, plan, 8), dict(v_out=torch.zeros(20, 16, device=d, dtype=dt))),
             ((y, x, ta, tb, plan, 8), dict(packed_ranks=True)),
             ((y, x, ta, tb, plan, 8), dict(adapter_rank=torch.zeros(1, device=d)))]
    for args, kw in calls:
        with pytest.raises(RuntimeError) as native:
            K.smlm_lora_forward(*args, **kw)
        with general(host), pytest.raises(RuntimeError) as python:
            K.smlm_lora_forward(*args, **kw)
        assert str(native.value) == str(python.value)


@pytest.mark.parametrize("ranks", [[16, 16], [8, 16]], ids=["one-shape", "two-shapes"])
@pytest.mark.parametrize("path", ["native", "general"])
def test_recorded_layer_steps_share_a_pool(host, gpu_device, path, ranks):
    """Two graphs of one memory pool: the second is recorded over the first one's freed gradients and replayed first, so it
    must make the tables of their addresses for itself."""
    from loquetier_amd.kernel_utils import BatchLenInfo
    d = gpu_device
    ctx, layer = _layer(d, "bf16", ranks, 16, 512, 384, 5)
    layer.set_trainable([0, 1])
    blen = BatchLenInfo([(1, 40), (1, 24)], [], 0, [], d)
    segment = torch.tensor([0, 40, 64], dtype=torch.int32, device=d)
    x = torch.randn(64, 512, device=d).to(torch.bfloat16).requires_grad_(True)
    up = torch.randn(64, 384, device=d).to(torch.bfloat16)
    params = [p for p in layer.parameters() if p.requires_grad]
    step = lambda: torch.autograd.grad(layer(x), [x, *params], up)
    with general(host) if path == "general" else contextlib.nullcontext():
        ctx.update(blen=blen, lora_ids=[0, 1], lora_len=None, segment=segment, train_idx=[0, 1])
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            layer.base_layer(x)
            side.synchronize()
            with pytest.raises(RuntimeError, match="run the step once before"):
                with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=side):
                    layer(x)
            for _ in range(2):
                want = [t.clone() for t in step()]
            side.synchronize()
            kept = {k: dict(t["grad_tabs"]) for k, t in layer._train_tabs.items()}
            first, second = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
            with torch.cuda.graph(first, stream=side):
                outs = step()
            del outs
            with torch.cuda.graph(second, pool=first.pool(), stream=side):
                outs = step()
    assert kept and all(t["grad_tabs"].keys() == kept[k].keys() for k, t in layer._train_tabs.items())
    for _ in range(3):
        for graph in (second, first, second):
            for t in outs:
                t.fill_(7.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            if graph is second:
                same(outs, want)
        same(step(), want)
