"""What the time of this framework is measured on: the work a serving or fine-tuning program has it do, through the
public entry points, with the sizes such programs use.

`listed()` names the cases, `draw(rng)` makes further ones of the same ranges.  A case is a dict of plain values:

  kind      which entry points a pass goes through
              "layers"     MixedLoraContext / MixedLoraLinear, the layers of one or more decoder blocks
              "operator"   smlm_lora_forward_multi / smlm_lora_backward_multi over plans the pass makes
              "reference"  add_lora.apply with per-segment pointer tables (the reference's own call), and its backward
              "gemm"       two smlm_forward_cutlass calls, the reference's lowest entry point
              "rmsnorm"    rms_norm.apply and its backward
  dtype     "fp16" or "bf16"
  train     segments of training rows, first in the batch (forward and backward), as "LENGTHxCOUNT,..."
  serve     segments of serving rows (forward only), likewise; "~8x700": 700 lengths of a geometric law of mean 8
  adapters  resident adapters; segment i uses adapter i modulo their number (rotated by the seed); the training
            segments of a mixed batch use the first train_adapters of them, the serving segments the others
  ranks     "16": every adapter has that rank; "8,16,32,64": adapter a has rank a modulo the list, stored at its own rank
  widths    the projections, as "H_INxH_OUT,..."
  blocks    how often the projections are repeated (decoder blocks of one pass)
  dropout   dropout probability of the training adapters
  graph     the pass is recorded once as a HIP graph and replayed, as a serving loop does with its decode step
"""
from __future__ import annotations

import math
import random

import torch

from loquetier_amd.kernel_utils import BatchLenInfo, add_lora, rms_norm
from loquetier_amd.mixed_lora import MixedLoraContext, MixedLoraLinear, NamedLoraLayer, prepare_weight
from loquetier_amd.ops import _kernels as K
from loquetier_amd.segments import build_segments_device

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
LLAMA2_7B = "4096x4096,4096x4096,4096x4096,4096x4096,4096x11008,4096x11008,11008x4096"
SCALE = 2.0  # lora_alpha / r


def _case(kind, dtype, widths, train="", serve="", adapters=1, train_adapters=0, ranks="16", blocks=1, dropout=0.0,
          graph=False):
    return dict(kind=kind, dtype=dtype, widths=widths, train=train, serve=serve, adapters=adapters,
                train_adapters=train_adapters, ranks=ranks, blocks=blocks, dropout=dropout, graph=graph)


def listed():
    cases = {
        # a handful of users: eight requests decode one token each, every linear of one decoder block called from
        # Python, routing built on the device: launches and host time are all there is
        "decode_few": _case("layers", "fp16", LLAMA2_7B, serve="1x8", adapters=4),
        # a busy server's decode step (256 requests over 32 adapters) through the layers of two decoder blocks,
        # replayed from a graph
        "decode_layers": _case("layers", "fp16", LLAMA2_7B, serve="1x256", adapters=32, blocks=2, graph=True),
        # the same batch where the program issues q/k/v/o of a block in one call: six blocks, one plan
        "decode_qkvo": _case("operator", "fp16", "4096x4096,4096x4096,4096x4096,4096x4096", serve="1x256", adapters=32,
                             blocks=6, graph=True),
        # prompts join a decoding batch: four of 512 tokens and 64 single tokens, the MLP's projections
        "prefill_mixed": _case("operator", "fp16", "4096x11008,4096x11008,11008x4096", serve="512x4,1x64", adapters=16,
                               ranks="32"),
        # long prompts at a high rank, the wider MLP: the largest forward
        "prefill_long": _case("operator", "bf16", "4096x14336,4096x14336,14336x4096", serve="2048x3,1531x1",
                              adapters=8, ranks="64"),
        # fine-tuning beside serving: four sequences of 1024 tokens and 128 decoding requests, the attention
        # projections through autograd
        "finetune_layers": _case("layers", "bf16", "4096x4096,4096x4096,4096x4096,4096x4096", train="1024x4",
                                 serve="1x128", adapters=36, train_adapters=4),
        # many small requests over 64 adapters of four ranks, a quarter of them training, all wide projections of a
        # block in one call each way: the largest pass
        "finetune_many_ranks": _case("operator", "bf16", "4096x4096,4096x1024,4096x1024,4096x14336,4096x14336,14336x4096",
                                     train="~8x268", serve="~8x807", adapters=64, ranks="8,16,32,64"),
        # the usual fine-tuning recipe: dropout on the adapters' input, ragged sequences, query and value
        "finetune_dropout": _case("operator", "bf16", "4096x4096,4096x1024", train="700x2,1021x1,333x1", serve="1x32",
                                  adapters=6, train_adapters=2, ranks="32", dropout=0.05),
        # high-rank adapters on the attention projections
        "finetune_rank128": _case("operator", "bf16", "4096x4096,4096x4096", train="512x4", serve="1x16", adapters=6,
                                  train_adapters=2, ranks="128"),
        # a program written against the reference: its own operator, pointer tables per segment, a small training
        # batch beside decoding requests
        "reference_train": _case("reference", "bf16", "4096x4096", train="200x3", serve="1x40", adapters=8,
                                 train_adapters=3),
        # ... and its lowest entry point, on a ragged prefill batch
        "reference_gemm": _case("gemm", "fp16", "4096x11008", serve="~90x24", adapters=10),
        # the other operator of the model: RMSNorm over the fine-tune + serve batch, forward and backward
        "rmsnorm_train": _case("rmsnorm", "bf16", "4096x4096", train="1024x4", serve="1x128"),
    }
    return [dict(c, name=name) for name, c in cases.items()]


def draw(rng: random.Random):
    """A case of the ranges the listed ones stand for: any of their entry points; batches of 1 to 8192 rows, hidden
    sizes of 512 to 14336 (multiples of eight), ranks of 8 to 128, 1 to 64 adapters."""
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    width = lambda lo, hi: rng.choice([8 * log(lo // 8, hi // 8), 4096])
    dtype = rng.choice(["fp16", "bf16"])
    rank = str(rng.choice([8, 16, 16, 24, 32, 48, 64, 128]))
    adapters = log(1, 64)
    family = rng.choice(["decode", "decode", "prefill", "prefill", "finetune", "finetune", "many_ranks", "reference",
                         "gemm", "rmsnorm"])
    while True:
        if family == "decode":
            kind = rng.choice(["layers", "operator"])
            h, m = width(1024, 8192), width(2048, 14336)
            widths = f"{h}x{h},{h}x{h},{h}x{m},{m}x{h}" if rng.random() < 0.5 else f"{h}x{h},{h}x{h},{h}x{h}"
            graph = rng.random() < 0.7
            case = _case(kind, dtype, widths, serve=f"1x{log(1, 512)}", adapters=adapters,
                         ranks=rng.choice([rank, "16", "8,16,32"]), blocks=2 if graph else 1, graph=graph)
        elif family == "prefill":
            h, m = width(1024, 8192), width(2048, 14336)
            serve = f"{log(16, 2048)}x{rng.randint(1, 4)}" + (f",1x{log(1, 128)}" if rng.random() < 0.7 else "")
            case = _case(rng.choice(["operator", "operator", "layers"]), dtype, f"{h}x{m},{m}x{h}", serve=serve,
                         adapters=adapters, ranks=rank)
        elif family == "finetune":
            h, o = width(1024, 8192), width(512, 8192)
            n_train = rng.randint(1, 4)
            case = _case(rng.choice(["operator", "layers"]), "bf16", f"{h}x{h},{h}x{o}", train=f"{log(32, 1024)}x{n_train}",
                         serve=rng.choice(["", f"1x{log(1, 128)}"]), adapters=n_train + log(1, 32), train_adapters=n_train,
                         ranks=rank)
            if case["kind"] == "operator" and rng.random() < 0.4:
                case["dropout"] = rng.choice([0.05, 0.1])
        elif family == "many_ranks":
            h, m = width(1024, 4096), width(1024, 14336)
            case = _case("operator", "bf16", f"{h}x{h},{h}x{m},{m}x{h}", train=f"~{rng.randint(4, 12)}x{log(20, 268)}",
                         serve=f"~{rng.randint(4, 12)}x{log(20, 800)}", adapters=rng.choice([16, 32, 48, 64]),
                         ranks=rng.choice(["8,16,32,64", "16,32"]))
        elif family == "reference":
            h, o = width(1024, 8192), width(1024, 8192)
            n_train = rng.randint(0, 4)
            case = _case("reference", "bf16" if n_train else dtype, f"{h}x{o}",
                         train=f"{log(16, 600)}x{n_train}" if n_train else "", serve=f"1x{log(4, 256)}",
                         adapters=n_train + log(1, 32), train_adapters=n_train, ranks=rank)
        elif family == "gemm":
            case = _case("gemm", dtype, f"{width(1024, 8192)}x{width(1024, 14336)}", serve=f"~{log(1, 128)}x{log(4, 64)}",
                         adapters=adapters, ranks=rank)
        else:
            h = width(1024, 8192)
            case = _case("rmsnorm", dtype, f"{h}x{h}", train=f"{log(16, 8192)}x1", serve=rng.choice(["", f"1x{log(1, 256)}"]))
        # no dearer than the largest listed case
        if sum(_lengths(case)[0]) + sum(_lengths(case)[1]) <= 8192 and work(case)["bytes"] <= 2e9:
            return case


# ------------------------------------------------------------------------------------------------ sizes of a case
def _parse(text, rng):
    out = []
    for piece in filter(None, text.split(",")):
        n, count = piece.split("x")
        if n.startswith("~"):
            p = 1.0 / float(n[1:])
            out += [max(1, min(2048, int(math.log(1.0 - rng.random()) / math.log1p(-p)) + 1)) if p < 1 else 1
                    for _ in range(int(count))]
        else:
            out += [int(n)] * int(count)
    return out


def _lengths(case):
    rng = random.Random(f"{case['train']}|{case['serve']}")  # the lengths belong to the case, not to the seed
    return _parse(case["train"], rng), _parse(case["serve"], rng)


def _widths(case):
    return [tuple(int(v) for v in w.split("x")) for w in case["widths"].split(",")]


def _ranks(case):
    listed_ranks = [int(r) for r in case["ranks"].split(",")]
    return [listed_ranks[a % len(listed_ranks)] for a in range(case["adapters"])]


def _routing(case, seed=0):
    """Adapter of every segment.  Training segments use adapters of their own where the case says so."""
    train, serve = _lengths(case)
    NA, TA = case["adapters"], case["train_adapters"]
    turn = seed * len(case["ranks"].split(","))
    if not TA:
        return [(i + turn) % NA for i in range(len(train) + len(serve))]
    rest = max(1, NA - TA)
    return [(i + turn) % TA for i in range(len(train))] + [(TA + (i + turn) % rest) % NA for i in range(len(serve))]


def work(case):
    """Bytes and multiply-adds a pass cannot do without: x, the gradients and the weights of every adapter in use read
    once, results written once (the forward's y also read where it is added to), v and dV once at their own width."""
    train, serve = _lengths(case)
    n, T = sum(train), sum(train) + sum(serve)
    if case["kind"] == "rmsnorm":
        h = _widths(case)[0][0]
        rows = T if n else 0  # the backward covers the whole batch
        return {"bytes": 4 * T * h + 6 * rows * h + 6 * h + 8 * T, "flops": 4 * T * h + 10 * rows * h}
    ids, ranks = _routing(case), _ranks(case)
    lens = train + serve
    rank_sum = sum(ranks[a] for a in set(ids))
    train_sum = sum(ranks[a] for a in set(ids[:len(train)]))
    row_ranks = sum(l * ranks[a] for l, a in zip(lens, ids))
    train_row_ranks = sum(l * ranks[a] for l, a in zip(train, ids))
    adds = case["kind"] in ("layers", "operator")
    nbytes = flops = 0
    for h_in, h_out in _widths(case):
        nbytes += 2 * (T * h_in + T * h_out * (2 if adds else 1) + rank_sum * (h_in + h_out) + 2 * row_ranks)
        flops += 2 * row_ranks * (h_in + h_out)
        if n:
            nbytes += 2 * (n * (h_out + 2 * h_in) + 2 * train_sum * (h_in + h_out) + 3 * train_row_ranks)
            flops += 4 * train_row_ranks * (h_in + h_out)
    return {"bytes": nbytes * case["blocks"], "flops": flops * case["blocks"]}


def tolerance(case):
    """Four times what a pass differs by from the same path in float64 (16-bit inputs, v and dV rounded to 16 bits as the
    operator's contract says, sums in float64): measured 1.7e-3 in bf16 and 2.1e-4 in fp16 over all outputs, the
    rounding of the results; the largest single differences 1.2e-2 and 1.4e-3."""
    return {"rel": 7e-3, "max": 0.05} if case["dtype"] == "bf16" else {"rel": 9e-4, "max": 6e-3}


# -------------------------------------------------------------------------------------------------- inputs of a case
class _Base(torch.nn.Module):
    """Stands in for a frozen base projection, whose GEMM is not this framework's: returns its output, to which the
    layer adds the adapters' terms."""

    def __init__(self, out):
        super().__init__()
        self.weight = torch.nn.Parameter(torch.empty(1, device=out.device), requires_grad=False)
        self.out = out

    def forward(self, x):
        return self.out.detach()


def _table(tensors, dev):
    return torch.tensor([t.data_ptr() for t in tensors], dtype=torch.int64, device=dev)


def prepare(case, seed):
    dev = torch.device("cuda:0")
    dt = DTYPES[case["dtype"]]
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    randn = lambda *shape, std=1.0: (torch.randn(*shape, generator=gen, device=dev) * std).to(dt)
    train, serve = _lengths(case)
    lens = train + serve
    T, n, P = sum(lens), sum(train), len(train)
    s = dict(case=case, T=T, n=n, P=P)
    if case["kind"] == "rmsnorm":
        h = _widths(case)[0][0]
        s.update(x=randn(T, h), w=1 + 0.1 * randn(h), g=randn(T, h))
        s["x"].requires_grad_(n > 0), s["w"].requires_grad_(n > 0)
        return s
    ids, ranks, NA, r = _routing(case, int(seed)), _ranks(case), case["adapters"], max(_ranks(case))
    bounds = [0]
    for l in lens:
        bounds.append(bounds[-1] + l)
    int32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    ids_t, lens_t, seg_t = int32(ids), int32(lens), int32(bounds)
    packed = min(ranks) < r
    s.update(ids=ids, ids_t=ids_t, lens_t=lens_t, seg_t=seg_t, r=r, packed=packed)

    def adapters(h_in, h_out):
        A = [randn(q, h_in, std=h_in ** -0.5) for q in ranks]
        B = [randn(h_out, q, std=q ** -0.5) for q in ranks]
        return [prepare_weight(a, r, dt, dev, 0, pack=packed) for a in A], [prepare_weight(b, r, dt, dev, 1, pack=packed) for b in B]

    order = list(dict.fromkeys(ids[:P]))  # the training adapters, by first appearance
    s["projs"] = []
    for _ in range(case["blocks"]):
        for h_in, h_out in _widths(case):
            A, B = adapters(h_in, h_out)
            p = dict(A=A, B=B, x=randn(T, h_in), y=randn(T, h_out))
            if n:
                p["g"] = randn(T, h_out)
            s["projs"].append(p)

    if case["kind"] == "layers":
        ctx = s["ctx"] = MixedLoraContext()
        s["blen"] = BatchLenInfo([(1, l) for l in train], [], T - n, [], dev)
        for p in s["projs"]:
            named = [NamedLoraLayer(f"a{a}", p["A"][a], p["B"][a], torch.nn.Identity(), SCALE, ranks[a]) for a in range(NA)]
            p["layer"] = MixedLoraLinear(ctx, _Base(p["y"]), named, r, dt, is_scaled=False, fused=True)
            if n:
                p["layer"].set_trainable(order)
                p["x"].requires_grad_(True)
        s["params"] = [q for p in s["projs"] for q in p["layer"].parameters() if q.requires_grad]
        s["pass"] = _train_layers if n else _serve_layers
    elif case["kind"] == "operator":
        s["scale"] = torch.full((len(lens),), SCALE, device=dev)
        s["rank_t"] = int32(ranks) if packed else None
        s["workspace"] = K.Workspace(dev)
        for p in s["projs"]:
            p["a_tab"], p["b_tab"] = _table(p["A"], dev), _table(p["B"], dev)
            if n:
                p.update(v=torch.empty(T, r, dtype=dt, device=dev), dx=torch.empty(n, p["x"].size(1), dtype=dt, device=dev),
                         ta=_table([p["A"][a] for a in order], dev), tb=_table([p["B"][a] for a in order], dev))
                p["g"] = p["g"][:n].contiguous()
                for w, grads, table in (("A", "dA", "da"), ("B", "dB", "db")):  # all adapters' gradients in one buffer
                    sizes = [p[w][a].numel() for a in order]
                    p[grads] = torch.empty(sum(sizes), dtype=dt, device=dev)
                    p[table] = _table(p[grads].split(sizes), dev)
        if n:
            s["parts"], s["part_ad"] = int32(bounds[:P + 1]), int32([order.index(a) for a in ids[:P]])
            s["part_scale"] = torch.full((P,), SCALE, device=dev)
            s["rank_b"] = int32([ranks[a] for a in order]) if packed else None
        if case["dropout"]:
            seg_p = torch.zeros(len(lens), device=dev)
            seg_p[:P] = case["dropout"]
            bits = torch.empty(K.DropoutSpec.mask_nbytes(n, [h for h, _ in _widths(case)]), dtype=torch.uint8, device=dev)
            s["drop"] = K.DropoutSpec(seg_p, n, 17, int(seed), bits)
            s["drop_b"] = K.DropoutSpec(seg_p[:P].contiguous(), n, 17, int(seed), bits)
        s["pass"] = _operator
    else:
        p = s["projs"][0]
        s["wa_ptr"], s["wb_ptr"] = (_table([p[w][a] for a in ids], dev) for w in ("A", "B"))
        if case["kind"] == "gemm":
            s.update(v=torch.empty(T, r, dtype=dt, device=dev),
                     tmp=torch.empty(K.smlm_forward_cutlass_tmp_size(len(lens)), dtype=torch.uint8, device=dev))
        elif n:
            p["x"].requires_grad_(True)
            for w in ("A", "B"):
                p[w] = [t.requires_grad_(a in order) for a, t in enumerate(p[w])]
            s["weights"] = [p[w][a] for a in ids[:P] for w in ("A", "B")]
            s["partition"] = bounds[:P + 1]
            s["leaves"] = [p["x"]] + [p[w][a] for a in order for w in ("A", "B")]
        s["pass"] = _gemm if case["kind"] == "gemm" else _reference

    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        keep = [p["y"].clone() for p in s["projs"]]
        with torch.cuda.stream(side):  # once outside the recording: sizes the scratch memory
            s["pass"](s)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            s["out"] = s["pass"](s)
        for p, y in zip(s["projs"], keep):
            p["y"].copy_(y)
        s["graph"] = graph
    return s


# ---------------------------------------------------------------------------------------------------------- one pass
def run(state):
    if state["case"]["kind"] == "rmsnorm":
        return _rmsnorm(state)
    if state["case"]["graph"]:
        state["graph"].replay()
        return state["out"]
    return state["pass"](state)


def _serve_layers(s):
    with torch.no_grad():
        # the step's routing, from the requests' adapters and lengths, on the device
        ids, lens, segment, _ = build_segments_device(s["ids_t"], s["lens_t"])
        s["ctx"].update(blen=s["blen"], lora_ids=ids, lora_len=lens, segment=segment)
        return [p["layer"](p["x"]) for p in s["projs"]]


def _train_layers(s):
    for q in s["params"]:
        q.grad = None
    for p in s["projs"]:
        p["x"].grad = None
    s["ctx"].update(blen=s["blen"], lora_ids=s["ids_t"], lora_len=s["lens_t"], segment=s["seg_t"], train_idx=s["ids"][:s["P"]])
    outs = [p["layer"](p["x"]) for p in s["projs"]]
    torch.autograd.backward(outs, [p["g"] for p in s["projs"]])
    return [o.detach() for o in outs], [p["x"].grad for p in s["projs"]], [q.grad for q in s["params"]]


def _operator(s):
    case, n, r = s["case"], s["n"], s["r"]
    plan = K.SegmentPlan(s["seg_t"], s["ids_t"], s["T"], defer=True)
    bplan = K.SegmentPlan(s["parts"], s["part_ad"], n, defer=True) if n else None
    per_block = len(s["projs"]) // case["blocks"]
    for b in range(case["blocks"]):
        ps = s["projs"][b * per_block:(b + 1) * per_block]
        col = lambda key: [p[key] for p in ps]
        K.smlm_lora_forward_multi(col("y"), col("x"), col("a_tab"), col("b_tab"), plan, r, seg_scale=s["scale"],
                                  beta=1.0, v_out=col("v") if n else None, dropout=s.get("drop"),
                                  adapter_rank=s["rank_t"], workspace=s["workspace"], packed_ranks=s["packed"])
        if n:
            K.smlm_lora_backward_multi(col("dx"), col("da"), col("db"), col("g"), col("x"), col("v"), col("ta"), col("tb"),
                                       bplan, r, s["part_scale"], dropout=s.get("drop_b"), adapter_rank=s["rank_b"],
                                       workspace=s["workspace"], packed_ranks=s["packed"])
    keys = ("y", "dx", "dA", "dB") if n else ("y",)
    return [p[k] for p in s["projs"] for k in keys]


def _reference(s):
    p, r = s["projs"][0], s["r"]
    shape = (s["T"], p["B"][0].size(0))
    if not s["n"]:
        with torch.no_grad():
            return add_lora.apply(shape, p["x"], s["wa_ptr"], s["wb_ptr"], s["seg_t"], r, 0, [])
    y = add_lora.apply(shape, p["x"], s["wa_ptr"], s["wb_ptr"], s["seg_t"], r, s["n"], s["partition"], *s["weights"])
    return y.detach(), torch.autograd.grad(y, s["leaves"], p["g"])


def _gemm(s):
    p = s["projs"][0]
    y = torch.empty((s["T"], p["B"][0].size(0)), dtype=p["x"].dtype, device=p["x"].device)
    K.smlm_forward_cutlass(s["v"], p["x"], s["wa_ptr"], s["seg_t"], s["tmp"], False)
    K.smlm_forward_cutlass(y, s["v"], s["wb_ptr"], s["seg_t"], s["tmp"], False)
    return s["v"], y


def _rmsnorm(s):
    o = rms_norm.apply(s["x"], s["w"], 1e-5)
    if not s["n"]:
        return o
    return o.detach(), torch.autograd.grad(o, (s["x"], s["w"]), s["g"])
