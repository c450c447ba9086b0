"""Workloads that stand for this package's use: optimizer steps and state quantisation.

A step is what a training loop calls once per iteration on all of a model's tensors, with the gradients a
backward pass has left; parameters and gradients lie in two flat buffers, as data-parallel wrappers lay
them out.  `prepare` builds the model's tensors and an optimizer whose states exist, `run` is one
`optimizer.step()` (or one quantise / dequantise round trip of a state tensor).
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "low-bit-optimizers_amd"))
import lpmm  # noqa: E402
import lpmm.functional as F  # noqa: E402

CONFIGS = os.path.join(os.path.dirname(lpmm.config.__file__), "configs")
MOST_OUTPUTS = 60


# ---- cases -------------------------------------------------------------------------------------
def _adamw(name=None, *, model, layers, width, ffn=0, vocab=0, config="", fused=False, factored=False, half=False):
    case = dict(path="adamw", model=model, layers=layers, width=width, ffn=ffn, vocab=vocab, config=config,
                fused=fused, factored=factored, half=half)
    return dict(case, name=name) if name else case


def _sgd(name=None, *, model, layers, width, ffn=0, vocab=0):
    case = dict(path="sgd", model=model, layers=layers, width=width, ffn=ffn, vocab=vocab)
    return dict(case, name=name) if name else case


def _quantise(name=None, *, rows, cols=0, kernel=0, bits=4, gp_sz=128):
    case = dict(path="quantise", rows=rows, cols=cols, kernel=kernel, bits=bits, gp_sz=gp_sz)
    return dict(case, name=name) if name else case


def listed():
    gpt2xl = dict(model="plain", layers=48, width=1600, ffn=6400, vocab=50257)
    decoder = dict(model="gated", layers=4, width=4096, ffn=11008)
    return [
        # full fine-tuning of a LLaMA-7B-shaped model with the fused step: the package's headline use
        _adamw("fused_llama7b", model="gated", layers=32, width=4096, ffn=11008, vocab=32000, fused=True),
        # a GPT-2-XL-shaped model, fused: half of its 580 tensors are short vectors with fp32 states
        _adamw("fused_gpt2xl", fused=True, **gpt2xl),
        # the smallest models one trains: fifty tensors of a few thousand to a million values, where host
        # work and launches are what a step costs
        _adamw("fused_small_model", model="plain", layers=4, width=256, ffn=1024, vocab=8192, fused=True),
        # the configuration the package recommends (4-bit m by blocks, rank-1 v) without the fused flag, on a
        # pipeline stage of decoder layers
        _adamw("default_decoder_layers", config="default.yml", **decoder),
        # the same configuration on the model with odd sizes: 1600 columns, a 50257-row embedding, bias vectors
        _adamw("default_gpt2xl", config="default.yml", **gpt2xl),
        # image models: 203 convolution weights of a ResNet-152 at twice the width, 1x1 and 3x3
        _adamw("default_conv", model="conv", layers=50, width=512, config="default.yml"),
        # Adafactor-style second moment, on the matrices of LLaMA's MLP and attention and their biases
        _adamw("factored_mlp", model="mlp", layers=8, width=4096, ffn=11008, fused=True, factored=True),
        # first moment kept in fp32, second in 4 bits
        _adamw("second_moment_only", config="2nd_moment_only_default.yml", **decoder),
        # 8-bit states for runs where 4 bits lose accuracy
        _adamw("eight_bit_layers", config="default_8b.yml", **decoder),
        # float16 parameters and gradients
        _adamw("half_decoder_layers", config="default.yml", half=True, **decoder),
        # SGD with a 4-bit momentum buffer on the image model
        _sgd("sgd_conv", model="conv", layers=50, width=512),
        # one state tensor through the quantisers and back (checkpoint conversion, other optimizers): a first
        # moment by blocks and a second moment by rank-1 scales, on an embedding's odd number of rows
        _quantise("quantise_embedding", rows=50257, cols=1600),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _near(rng, value, steps):
    step = rng.choice(steps)
    return max(step, value // step * step)


def draw(rng):
    path = rng.choice(["fused", "fused", "default", "default", "conv", "factored", "config", "half", "sgd", "quantise",
                       "quantise"])
    if path == "quantise":
        n = _log_int(rng, 1 << 12, 1 << 26)
        form = rng.choice(["vector", "matrix", "matrix", "conv"])
        bits, gp_sz = rng.choice([4, 4, 4, 5, 8]), rng.choice([128, 128, 128, 256, 1024])
        if form == "vector":
            return _quantise(rows=n, bits=bits, gp_sz=gp_sz)
        kernel = 3 if form == "conv" and n > 9 * 256 else 0
        cols = _near(rng, _log_int(rng, 16, max(17, min(16384, n // 16))), [1, 8, 64, 128])
        return _quantise(rows=max(1, n // cols // (kernel * kernel or 1)), cols=cols, kernel=kernel, bits=bits, gp_sz=gp_sz)
    if path == "conv" or (path == "sgd" and rng.random() < 0.5):
        model = dict(model="conv", layers=rng.randint(2, 50), width=_near(rng, _log_int(rng, 64, 512), [32, 64]))
        return _sgd(**model) if path == "sgd" else _adamw(config="default.yml", **model)
    total = _log_int(rng, 1 << 20, 1 << 29)
    # odd and unaligned widths as often as the usual multiples
    width = _near(rng, _log_int(rng, 64, min(8192, max(65, int((total / 12) ** 0.5)))), [2, 8, 64, 64, 128, 128])
    ffn = _near(rng, int(width * rng.uniform(2.0, 4.0)), [2, 8, 64, 128])
    model = rng.choice(["gated", "plain"])
    per_layer = 4 * width * width + (3 if model == "gated" else 2) * width * ffn
    most = 48 if width % 64 == 0 and ffn % 64 == 0 else 3
    layers = max(1, min(most, total // per_layer))
    vocab = _log_int(rng, 256, 65536) // 2 * 2 if rng.random() < 0.5 and width <= 4096 else 0
    sizes = dict(model=model, layers=layers, width=width, ffn=ffn, vocab=vocab)
    if path == "fused":
        return _adamw(config=rng.choice(["", "2nd_moment_group_128.yml"]), fused=rng.random() < 0.75, **sizes)
    if path == "sgd":
        return _sgd(**sizes)
    if path == "factored":
        return _adamw(fused=True, factored=True, **dict(sizes, model="mlp", vocab=0))
    if path == "config":
        config = rng.choice(["2nd_moment_only_default.yml", "2nd_moment_only_group_128.yml", "1st_moment_group_256.yml",
                             "1st_moment_group_1024.yml", "default_5b.yml", "default_8b.yml"])
        return _adamw(config=config, **sizes)
    if path == "half":
        config = rng.choice(["default.yml", "2nd_moment_group_128.yml"])
        sizes["layers"] = min(layers, 12)
        return _adamw(config=config, half=True, **sizes)
    return _adamw(config="default.yml", **sizes)


# ---- tensors -----------------------------------------------------------------------------------
def _shapes(case):
    """(shape, is an embedding) of every tensor of the case's model."""
    d, f, vocab = case["width"], case["ffn"], case["vocab"]
    out = []
    if case["model"] == "gated":
        if vocab:
            out.append(((vocab, d), True))
        for _ in range(case["layers"]):
            out += [(s, False) for s in [(d, d)] * 4 + [(f, d)] * 2 + [(d, f)] + [(d,)] * 2]
        if vocab:
            out += [((d,), False), ((vocab, d), False)]
    elif case["model"] == "plain":
        if vocab:
            out += [((vocab, d), True), ((1024, d), False)]
        for _ in range(case["layers"]):
            out += [(s, False) for s in [(d,), (d,), (d, 3 * d), (3 * d,), (d, d), (d,), (d,), (d,), (d, f), (f,), (f, d), (d,)]]
        if vocab:
            out += [((d,), False)] * 2
    elif case["model"] == "mlp":
        for _ in range(case["layers"]):
            out += [(s, False) for s in [(d, f), (f, d), (d, d), (f,), (d,)]]
    else:  # bottleneck blocks in four stages (50 blocks: 3, 8, 36, 3) between a stem and a classifier
        n, w = case["layers"], d
        out.append(((w // 4, 3, 7, 7), False))
        for k in range(n):
            s = w << (0 if k < 0.06 * n else 1 if k < 0.22 * n else 2 if k < 0.94 * n else 3)
            out += [((s // 4, s, 1, 1), False), ((s // 4, s // 4, 3, 3), False), ((s, s // 4, 1, 1), False), ((s,), False)]
        out += [((1000, 8 * w), False), ((1000,), False)]
    return out


class _Flat:
    """Tensors laid out one after another, at the alignment the caching allocator would give each."""

    def __init__(self, sizes, dtype):
        item = torch.empty((), dtype=dtype).element_size()
        self.at, end = [], 0
        for n in sizes:
            align = ((2 << 20) if n * item >= (1 << 20) else 512) // item
            self.at.append(-(-end // align) * align)
            end = self.at[-1] + n
        self.sizes = sizes
        self.data = torch.zeros(end, dtype=dtype, device="cuda")

    def view(self, k, shape):
        return self.data[self.at[k]: self.at[k] + self.sizes[k]].view(shape)


def _fill_gradients(grads, views, gen, size):
    """Normal values whose scale differs from row to row; an embedding gets none in the rows of tokens the
    batch does not hold."""
    grads.data.normal_(generator=gen)
    for g, embedding in views:
        if g.dim() == 1:
            g.mul_(size)
            continue
        scale = torch.randn(g.shape[0], device="cuda", generator=gen).mul_(0.5).exp_().mul_(size)
        if embedding:
            scale.mul_(torch.rand(g.shape[0], device="cuda", generator=gen).lt_(0.5))
        g.mul_(scale.to(g.dtype).view([-1] + [1] * (g.dim() - 1)))


def _state_slots(opt, params):
    """Where to find every tensor on the GPU in the parameters' states, the quantisation maps aside:
    (dict, key, index where the dict holds a list of tensors)."""
    slots = []
    for p in params:
        state = opt.state[p]
        for key in sorted(state):
            if key.endswith("_qstate"):
                overhead = state[key]["overhead"]
                if overhead.get("max1") is not None:
                    slots.append((overhead, "max1", None))
                slots += [(overhead, "max_dims", i) for i in range(len(overhead.get("max_dims") or ()))]
            elif state[key].is_cuda and state[key].numel() > 1:
                slots.append((state, key, None))
    return slots


def _tensor(slot):
    holder, key, index = slot
    return holder[key] if index is None else holder[key][index]


def _gather_states(slots):
    """Moves states into one flat buffer per data type."""
    flats = {}
    for dtype in (torch.int8, torch.float32, torch.float16):
        kind = [s for s in slots if _tensor(s).dtype is dtype]
        if not kind:
            continue
        flat = _Flat([_tensor(s).numel() for s in kind], dtype)
        for k, (holder, key, index) in enumerate(kind):
            view = flat.view(k, _tensor((holder, key, index)).shape)
            view.copy_(_tensor((holder, key, index)))
            if index is None:
                holder[key] = view
            else:
                holder[key][index] = view
        flats[str(dtype)[6:]] = flat.data
    return flats


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["path"] == "quantise":
        shape = [case["rows"]] + [case["cols"]] * (case["cols"] > 0) + [case["kernel"]] * 2 * (case["kernel"] > 0)
        x = torch.randn(shape, device="cuda", generator=gen)
        scale = torch.randn(shape[0], device="cuda", generator=gen).exp_().view([-1] + [1] * (len(shape) - 1))
        x.mul_(scale)
        jobs = []
        for data, kind, signed, scaling in ((x * 1e-3, "nonlinear", True, "group"), (x.square_().mul_(1e-6), "power-1", False, "rank1")):
            jobs.append((data, dict(qmap=F.create_general_qmap(kind, case["bits"], signed).cuda(), b=case["bits"], scale_type=scaling,
                                    quant_type=kind, round_type="real-nearest", gp_sz=case["gp_sz"], signed=signed, shape=data.shape)))
        return {"jobs": jobs}

    half = case["path"] == "adamw" and case["half"]
    shapes = _shapes(case)
    sizes = [math.prod(s) for s, _ in shapes]
    weights, grads = (_Flat(sizes, torch.float16 if half else torch.float32) for _ in range(2))
    weights.data.normal_(0, 0.02, generator=gen)
    params, views = [], []
    for k, (shape, embedding) in enumerate(shapes):
        p = torch.nn.Parameter(weights.view(k, shape))
        p.grad = grads.view(k, shape)
        params.append(p)
        views.append((p.grad, embedding))
    if case["path"] == "sgd":
        opt = lpmm.optim.SGD(params, lr=1e-3, momentum=0.9, weight_decay=1e-4)
    else:
        # float16 keeps neither 1e-8 nor the squares of small gradients: a loss-scaled run's sizes
        opt = lpmm.optim.AdamW(params, lr=1e-4, betas=(0.9, 0.999), eps=1e-3 if half else 1e-8, weight_decay=0.01,
                               factor_second_moment=case["factored"], fused=case["fused"],
                               qconfig=os.path.join(CONFIGS, case["config"]) if case["config"] else None)
    size = 0.1 if half else 1e-3
    _fill_gradients(grads, views, gen, size)
    opt.step()
    slots = _state_slots(opt, params)
    before = [_tensor(s) for s in slots]
    _fill_gradients(grads, views, gen, size)
    opt.step()
    # states that a step replaces by other tensors instead of writing them in place are returned one by one,
    # where they are few enough; where they are not (the row and column maxima of a whole model), the codes that
    # decode with them are all there
    moved = [s for s, t in zip(slots, before) if _tensor(s).data_ptr() != t.data_ptr()]
    flats = _gather_states([s for s, t in zip(slots, before) if _tensor(s).data_ptr() == t.data_ptr()])
    return {"opt": opt, "grads": grads, "outputs": dict(flats, weights=weights.data),
            "moved": moved if len(moved) <= MOST_OUTPUTS - len(flats) else []}


def run(state):
    if "jobs" in state:
        out = []
        for x, kw in state["jobs"]:
            codes, made = F.vectorwise_quant(x, **kw)
            back = F.vectorwise_dequant(codes, **made, **kw)
            out.append([codes, made["max_dims"] if made["max1"] is None else made["max1"], back])
        return out
    state["opt"].step()
    return [state["outputs"], [_tensor(s) for s in state["moved"]]]


def work(case):
    """Bytes: parameters and gradients read, parameters written, every state and its scales read and written.
    Flops: about 30 operations a value for a step, 10 for a round trip."""
    if case["path"] == "quantise":
        rows, cols, taps = case["rows"], case["cols"] or 1, (case["kernel"] or 1) ** 2
        n = rows * cols * taps
        codes = 0.5 if case["bits"] == 4 else 1.0
        scales = 4 * n / case["gp_sz"] + 4 * (rows + cols + 2 * case["kernel"] if case["cols"] else n / 128)
        return {"bytes": 4 * (4 + codes) * n + 2 * scales, "flops": 20 * n}
    real = 2 if case["path"] == "adamw" and case["half"] else 4
    total = values = 0
    for shape, _ in _shapes(case):
        n = math.prod(shape)
        values += n
        total += 3 * real * n
        if n <= 4096:
            total += (2 if case["path"] == "adamw" else 1) * 2 * real * n
            continue
        if case["path"] == "sgd":
            total += 2 * (0.5 + 4 / 128) * n
            continue
        config = case["config"]
        bits = 1.0 if config in ("default_5b.yml", "default_6b.yml", "default_7b.yml", "default_8b.yml") else 0.5
        group = int(config.split("_")[-1][:-4]) if config.startswith("1st_moment_group_") else 128
        total += 8 * n if config.startswith("2nd_moment_only") else 2 * (bits + real / group) * n
        if case["factored"] and len(shape) > 1:
            total += 2 * 4 * (shape[-2] + shape[-1])
        elif "group_128" in config or config == "" or len(shape) == 1 or case["fused"]:
            total += 2 * (bits + real / 128) * n
        else:
            total += 2 * (bits * n + real * sum(shape))
    return {"bytes": total, "flops": 30 * values}


def tolerance(case):
    """Codes, and the scales they decode with, are fixed to the bit, as is a decoded value (one product).  The
    parameter update is free to round otherwise.  Against the same update in 64 bits the weights are off by 4e-8 in
    float32 and by 2e-4 (at most 6e-4 in one value) in float16; the fused step's float32 update folds its constants,
    which one value shows by up to 1e-6."""
    if case["path"] == "quantise":
        return "exact"
    if case["path"] == "adamw" and case["half"]:
        return {"rel": 8e-4, "max": 2.5e-3, "differ": 0.0}
    return {"rel": 2e-7, "max": 4e-6, "differ": 0.0}
