"""Performance cases: the work that programs built on this package have it do.

Two entry points are exercised. "stack" cases go through `sru_amd.SRU`, the layer stack that
training and serving programs construct; "scan" cases go through `sru_amd.ElementwiseRecurrence`
under autograd, the boundary at which a program that keeps its own layer code calls the kernels.
`draw` gives further cases of the ranges that the listed ones stand for.
"""
import math

import torch

import sru_amd

DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
DEVICE = "cuda"

# Limits of the drawn cases, so that none costs more than the largest listed one.
MAX_TRAIN_FLOPS = {"float32": 2.0e11, "bfloat16": 4.0e12}
MAX_SCAN_CELLS = 256 * 64 * 2048
MAX_INFER_CELLS = 4096 * 256 * 512


def _stack(name, **kw):
    case = dict(name=name, path="stack", mode="train", length=0, batch=0, input=0, hidden=0, layers=2,
                bidirectional=False, projection=0, layer_norm=False, rescale=False, highway_bias=0.0,
                weights="float32", autocast="", padded=False, state=False, input_grad=False)
    case.update(kw)
    return case


def _scan(name, **kw):
    case = dict(name=name, path="scan", length=0, batch=0, hidden=0, bidirectional=False, k=3, dtype="float32",
                x_float32=False, tanh=False, padded=False, dropout=False, state=False, last_grad=False)
    case.update(kw)
    return case


def listed():
    return [
        # The smallest forward call: the README's two-layer example as a program evaluates it.
        _stack("readme_forward", mode="infer", length=20, batch=32, input=128, hidden=128, highway_bias=-2.0),
        # Generation: one token at a time through the language-model stack in 16-bit weights, the
        # state of every layer carried by the caller.
        _stack("decode_step", mode="infer", length=1, batch=16, input=2048, hidden=2048, layers=10, projection=512,
               weights="bfloat16", state=True),
        # The same stack reading one prompt before generation starts.
        _stack("prompt_prefill", mode="infer", length=512, batch=1, input=2048, hidden=2048, layers=10,
               projection=512, weights="bfloat16"),
        # A small training step (the layer size of the reference's speed chart, L=32, d=256, batch 32).
        _stack("train_small", length=32, batch=32, input=256, hidden=256),
        # Classification-scale training step under bf16 autocast: bidirectional, layer norm, rescale.
        _stack("train_classifier", length=256, batch=64, input=1024, hidden=1024, layers=4, bidirectional=True,
               layer_norm=True, rescale=True, autocast="bfloat16"),
        # Language-model-scale training step under bf16 autocast; the input is a batch of float32
        # embedding rows whose gradient goes back to the table. (Without the layers' random dropout
        # masks, so that a step can be repeated; "scan" cases have one.)
        _stack("train_language_model", length=512, batch=16, input=2048, hidden=2048, layers=10, projection=512,
               autocast="bfloat16", input_grad=True),
        # Long-sequence inference in 16-bit weights: right-padded batches with a given initial state.
        _stack("long_sequences", mode="infer", length=4096, batch=256, input=256, hidden=256, bidirectional=True,
               weights="float16", padded=True, state=True),
        # The recurrence alone, forward + backward, at the size the package is quoted on, in both
        # stream types that are trained with.
        _scan("scan_headline_f32", length=256, batch=64, hidden=1024, bidirectional=True),
        _scan("scan_headline_bf16", length=256, batch=64, hidden=1024, bidirectional=True, dtype="bfloat16"),
        # Right-padded mini-batches of medium length in float32.
        _scan("scan_padded_f32", length=128, batch=32, hidden=512, bidirectional=True, padded=True),
        # A language-model layer with its variational dropout mask in bf16: few columns, long walk.
        _scan("scan_language_model_bf16", length=512, batch=16, hidden=2048, dtype="bfloat16", dropout=True),
        # Ragged sizes: a width that is no multiple of a wavefront, an odd length and batch, four
        # streams, fp16, padding, an initial state and a loss on the last state.
        _scan("scan_ragged_f16", length=201, batch=77, hidden=304, bidirectional=True, k=4, dtype="float16",
              padded=True, state=True, last_grad=True),
    ]


# ---------------------------------------------------------------------------------- drawn cases
def _log_int(rng, lo, hi, multiple=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi, max(lo, round(v / multiple) * multiple, multiple)))


def _width(rng, lo, hi):
    """A hidden size: mostly multiples of 64 or 8, sometimes any number."""
    return _log_int(rng, lo, hi, rng.choice([64, 64, 8, 8, 2, 1]))


def _gemm_flops(case):
    rows = case["length"] * case["batch"]
    out = case["hidden"] * (2 if case["bidirectional"] else 1)
    total, width = 0, case["input"]
    for _ in range(case["layers"]):
        streams = out * (3 if width == out else 4)
        n_proj = case["projection"]
        if 0 < n_proj < min(width, out):
            total += 2 * rows * (width * n_proj + n_proj * streams)
        else:
            total += 2 * rows * width * streams
        width = out
    return total


def draw(rng):
    family = rng.choice(["forward", "decode", "prefill", "train", "train", "long", "scan", "scan", "scan"])
    bi = rng.random() < 0.5
    if family == "forward":
        d = _width(rng, 64, 512)
        return _drawn(_stack("", mode="infer", length=_log_int(rng, 4, 64), batch=_log_int(rng, 1, 64), input=d,
                             hidden=d, layers=rng.randint(1, 4), bidirectional=bi, highway_bias=-2.0,
                             layer_norm=rng.random() < 0.25))
    if family in ("decode", "prefill"):
        d = _log_int(rng, 256, 2048, 64)
        length, batch = (1, _log_int(rng, 1, 64)) if family == "decode" else \
            (_log_int(rng, 128, 1024), _log_int(rng, 1, 4))
        return _drawn(_stack("", mode="infer", length=length, batch=batch, input=d, hidden=d,
                             layers=rng.randint(2, 10), projection=rng.choice([0, d // 4]),
                             weights=rng.choice(["bfloat16", "bfloat16", "float16", "float32"]),
                             state=family == "decode" or rng.random() < 0.5))
    if family == "train":
        amp = rng.choice(["", "bfloat16", "bfloat16"])
        d = _log_int(rng, 128, 1024, rng.choice([64, 64, 16, 2]))
        case = _stack("", length=_log_int(rng, 16, 512), batch=_log_int(rng, 8, 64), input=d,
                      hidden=d if rng.random() < 0.7 else _log_int(rng, 128, 1024, 16), layers=rng.randint(2, 6),
                      bidirectional=bi, layer_norm=rng.random() < 0.5, rescale=rng.random() < 0.5,
                      projection=rng.choice([0, 0, d // 4]), autocast=amp, padded=rng.random() < 0.5,
                      input_grad=rng.random() < 0.5)
        limit = MAX_TRAIN_FLOPS[amp or "float32"] / 3
        while _gemm_flops(case) > limit:
            if case["length"] > 16:
                case["length"] = max(16, case["length"] * 2 // 3)
            elif case["batch"] > 8:
                case["batch"] = max(8, case["batch"] * 2 // 3)
            else:
                case["layers"] -= 1
        return _drawn(case)
    if family == "long":
        d = _log_int(rng, 64, 256, rng.choice([64, 8]))
        length = _log_int(rng, 1024, 4096)
        dirs = 2 if bi else 1
        batch = min(_log_int(rng, 16, 256), MAX_INFER_CELLS // (length * d * dirs))
        return _drawn(_stack("", mode="infer", length=length, batch=batch, input=d, hidden=d, bidirectional=bi,
                             weights=rng.choice(["float16", "bfloat16"]), padded=rng.random() < 0.75,
                             state=rng.random() < 0.5))
    d, length = _width(rng, 32, 2048), _log_int(rng, 16, 1024)
    dirs = 2 if bi else 1
    batch = min(_log_int(rng, 4, 128), max(1, MAX_SCAN_CELLS // (length * d * dirs)))
    dtype = rng.choice(["float32", "bfloat16", "bfloat16", "float16"])
    k = rng.choice([3, 3, 3, 4])
    return _drawn(_scan("", length=length, batch=batch, hidden=d, bidirectional=bi, k=k, dtype=dtype,
                        x_float32=dtype != "float32" and k == 3 and rng.random() < 0.25, tanh=rng.random() < 0.1,
                        padded=rng.random() < 0.5, dropout=rng.random() < 0.5, state=rng.random() < 0.5,
                        last_grad=rng.random() < 0.5))


def _drawn(case):
    del case["name"]
    return case


# ---------------------------------------------------------------------------------- a user's state
def _right_padding(gen, length, batch):
    """Mask of a right-padded batch, lengths uniform in [length / 4, length]."""
    lens = torch.randint(max(1, length // 4), length + 1, (batch,), generator=gen, device=DEVICE)
    return torch.arange(length, device=DEVICE)[:, None] >= lens[None, :]


def _prepare_stack(case, seed):
    torch.manual_seed(seed)
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    weights = DTYPES[case["weights"]]
    with torch.device(DEVICE):
        model = sru_amd.SRU(case["input"], case["hidden"], num_layers=case["layers"],
                            bidirectional=case["bidirectional"], projection_size=case["projection"],
                            layer_norm=case["layer_norm"], rescale=case["rescale"],
                            highway_bias=case["highway_bias"])
    model = model.to(weights)
    L, B, out = case["length"], case["batch"], model.output_size
    randn = lambda *size: torch.randn(*size, generator=gen, device=DEVICE)
    state = dict(case=case, model=model, x=randn(L, B, case["input"]).to(weights), c0=None, mask=None, probe=None)
    if case["state"]:
        state["c0"] = randn(case["layers"], B, out).to(weights)
    if case["padded"]:
        state["mask"] = _right_padding(gen, L, B)
    if case["mode"] == "infer":
        model.eval()
    else:
        model.train()
        state["x"].requires_grad_(case["input_grad"])
        state["probe"] = randn(L, B, out).to(DTYPES[case["autocast"] or case["weights"]])
    return state


def _prepare_scan(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    L, B = case["length"], case["batch"]
    dirs = 2 if case["bidirectional"] else 1
    D = case["hidden"] * dirs
    dtype = DTYPES[case["dtype"]]
    randn = lambda *size: torch.randn(*size, generator=gen, device=DEVICE)
    state = dict(case=case, c0=None, mask=None, mask_c=None, scale=None, grad_last=None)
    state["u"] = randn(L, B, D * case["k"]).to(dtype).requires_grad_()
    state["x"] = randn(L, B, D).to(torch.float32 if case["x_float32"] else dtype).requires_grad_(case["k"] == 3)
    state["weight_c"] = ((2 * torch.rand(2 * D, generator=gen, device=DEVICE) - 1) * 1.5 ** 0.5).requires_grad_()
    state["bias"] = (0.5 * randn(2 * D)).requires_grad_()
    if case["state"]:
        state["c0"] = randn(B, D).requires_grad_()
    if case["k"] == 3:
        state["scale"] = torch.full((1,), 3 ** 0.5, device=DEVICE)
    if case["dropout"]:
        state["mask_c"] = (torch.rand(B, D, generator=gen, device=DEVICE) < 0.9).float() / 0.9
    if case["padded"]:
        state["mask"] = _right_padding(gen, L, B)
    state["grad_h"] = randn(L, B, D).to(dtype)
    if case["last_grad"]:
        state["grad_last"] = randn(B, D).to(dtype)
    return state


def prepare(case, seed):
    return _prepare_stack(case, seed) if case["path"] == "stack" else _prepare_scan(case, seed)


# ---------------------------------------------------------------------------------- one pass
def _run_stack(s):
    model, case = s["model"], s["case"]
    if case["mode"] == "infer":
        with torch.no_grad():
            h, c = model(s["x"], s["c0"], mask_pad=s["mask"])
        return {"h": h, "c": c}
    model.zero_grad(set_to_none=True)
    s["x"].grad = None
    if case["autocast"]:
        with torch.autocast("cuda", dtype=DTYPES[case["autocast"]]):
            h, c = model(s["x"], s["c0"], mask_pad=s["mask"])
    else:
        h, c = model(s["x"], s["c0"], mask_pad=s["mask"])
    h.backward(s["probe"])
    out = {"h": h.detach(), "c": c.detach()}
    for name, p in model.named_parameters():
        out["grad_" + name] = p.grad
    if s["x"].grad is not None:
        out["grad_x"] = s["x"].grad
    return out


def _run_scan(s):
    case = s["case"]
    h, last = sru_amd.ElementwiseRecurrence.apply(
        s["u"], s["x"], s["weight_c"], s["bias"], s["c0"], 1 if case["tanh"] else 0, case["hidden"],
        case["bidirectional"], True, s["scale"], s["mask_c"], s["mask"])
    inputs = {n: s[n] for n in ("u", "x", "weight_c", "bias", "c0") if s[n] is not None and s[n].requires_grad}
    outputs, seeds = [h], [s["grad_h"]]
    if s["grad_last"] is not None:
        outputs.append(last)
        seeds.append(s["grad_last"])
    grads = torch.autograd.grad(outputs, list(inputs.values()), seeds)
    out = {"h": h.detach(), "last": last.detach()}
    out.update(("grad_" + n, g) for n, g in zip(inputs, grads))
    return out


def run(state):
    return _run_stack(state) if state["case"]["path"] == "stack" else _run_scan(state)


# ---------------------------------------------------------------------------------- the same in 64 bits
def _scan64(u, x, weight_c, bias, c0, hidden, dirs, k, tanh, scale, mask_c, pad):
    """The recurrence written out step by step: u (L, B, D * k), x (L, B, D) or None -> h, last state."""
    L, B = u.shape[:2]
    D = hidden * dirs
    u = u.view(L, B, D, k)
    w1, w2, b1, b2 = weight_c[:D], weight_c[D:], bias[:D], bias[D:]
    skip = u[..., 3] if k == 4 else x.view(L, B, D) * scale
    c0 = u.new_zeros(B, D) if c0 is None else c0
    hs, lasts = [], []
    for i in range(dirs):
        cols = slice(i * hidden, (i + 1) * hidden)
        reverse = (lambda t: t.flip(0)) if i else (lambda t: t)
        uu, ss = reverse(u[:, :, cols]), reverse(skip[:, :, cols])
        keep = None if pad is None else reverse(pad)[..., None]
        c, prev, cur = c0[:, cols], [], []
        u0, u1 = uu[..., 0].unbind(0), (uu[..., 1] + b1[cols]).unbind(0)
        for t in range(L):
            prev.append(c)
            new = torch.lerp(u0[t], c, torch.sigmoid(torch.addcmul(u1[t], w1[cols], c)))
            c = new if keep is None else torch.where(keep[t], c, new)
            cur.append(c)
        prev, cur = torch.stack(prev), torch.stack(cur)
        out = torch.sigmoid(uu[..., 2] + w2[cols] * prev + b2[cols])
        if mask_c is not None:
            out = out * mask_c[:, cols]
        h = ss + ((torch.tanh(cur) if tanh else cur) - ss) * out
        hs.append(reverse(h if keep is None else h.masked_fill(keep, 0.0)))
        lasts.append(c)
    return torch.cat(hs, -1), torch.cat(lasts, -1)


def _stack64(case, named, x, c0, pad):
    dirs = 2 if case["bidirectional"] else 1
    L, B, D = case["length"], case["batch"], case["hidden"] * dirs
    finals = []
    for i in range(case["layers"]):
        get = lambda n: named.get(f"rnn_lst.{i}.{n}")
        k = get("weight").size(1) // D
        y = x
        if get("layer_norm.weight") is not None:
            y = torch.nn.functional.layer_norm(x, x.shape[-1:], get("layer_norm.weight"), get("layer_norm.bias"), 1e-5)
        y = y.reshape(L * B, -1)
        if get("weight_proj") is not None:
            y = y @ get("weight_proj")
        scale = get("scale_x") if case["rescale"] else 1.0
        x, last = _scan64((y @ get("weight")).view(L, B, -1), x, get("weight_c"), get("bias"),
                          None if c0 is None else c0[i], case["hidden"], dirs, k, False, scale, None, pad)
        finals.append(last)
    return x, torch.stack(finals)


def exact(case, seed):
    s = prepare(case, seed)
    wide = lambda t: None if t is None else t.detach().double().requires_grad_(t.requires_grad)
    if case["path"] == "scan":
        t = {n: wide(s[n]) for n in ("u", "x", "weight_c", "bias", "c0", "scale", "mask_c")}
        h, last = _scan64(t["u"], t["x"], t["weight_c"], t["bias"], t["c0"], case["hidden"],
                          2 if case["bidirectional"] else 1, case["k"], case["tanh"],
                          1.0 if t["scale"] is None else t["scale"], t["mask_c"], s["mask"])
        inputs = {n: t[n] for n in ("u", "x", "weight_c", "bias", "c0") if t[n] is not None and t[n].requires_grad}
        outputs, seeds = [h], [s["grad_h"].double()]
        if s["grad_last"] is not None:
            outputs.append(last)
            seeds.append(s["grad_last"].double())
        grads = torch.autograd.grad(outputs, list(inputs.values()), seeds)
        out = {"h": h.detach(), "last": last.detach()}
        out.update(("grad_" + n, g) for n, g in zip(inputs, grads))
        return out
    params = {n: wide(p) for n, p in s["model"].named_parameters()}
    named = dict(params, **{n: b.double() for n, b in s["model"].named_buffers()})
    x, c0 = wide(s["x"]), wide(s["c0"])
    if case["mode"] == "infer":
        with torch.no_grad():
            h, c = _stack64(case, named, x, c0, s["mask"])
        return {"h": h, "c": c}
    h, c = _stack64(case, named, x, c0, s["mask"])
    wanted = dict(params, x=x) if x.requires_grad else params
    grads = torch.autograd.grad([h], list(wanted.values()), [s["probe"].double()])
    out = {"h": h.detach(), "c": c.detach()}
    out.update(("grad_" + n, g) for n, g in zip(wanted, grads))
    return out


# ---------------------------------------------------------------------------------- what a pass needs
def _bytes(name):
    return DTYPES[name].itemsize


def _work_stack(case):
    L, B = case["length"], case["batch"]
    out = case["hidden"] * (2 if case["bidirectional"] else 1)
    rows, size = L * B, _bytes(case["weights"])
    gemm = _gemm_flops(case)
    cells = rows * out * case["layers"]
    weights = gemm // (2 * rows) * size
    states = case["layers"] * B * out * size * (2 if case["state"] else 1)
    moved = rows * case["input"] * size + weights + states + (rows if case["padded"] else 0)
    h_size = _bytes(case["autocast"] or case["weights"])
    if case["mode"] == "infer":
        return {"bytes": moved + rows * out * h_size, "flops": gemm + 20 * cells}
    # h written, its gradient read, every weight gradient and, where asked for, the input's written
    moved += 2 * rows * out * h_size + weights + (rows * case["input"] * size if case["input_grad"] else 0)
    first = 0
    if not case["input_grad"] and not case["layer_norm"]:
        one = dict(case, layers=1)
        first = _gemm_flops(one)    # the first layer's product with the weights' transpose is not needed
        if 0 < case["projection"] < min(case["input"], out):
            first = 2 * rows * case["input"] * case["projection"]
    return {"bytes": moved, "flops": 3 * gemm - first + 60 * cells}


def _work_scan(case):
    D = case["hidden"] * (2 if case["bidirectional"] else 1)
    cells = case["length"] * case["batch"] * D
    size = _bytes(case["dtype"])
    x_size = 0 if case["k"] == 4 else 4 if case["x_float32"] else size
    # U, x and the gradient of h in; h and the gradients of U and x out
    moved = cells * (2 * case["k"] * size + 2 * x_size + 2 * size)
    small = case["batch"] * D * 4
    moved += small * (1 + 2 * case["state"] + case["dropout"] + case["last_grad"]) + 4 * 8 * D
    moved += case["length"] * case["batch"] if case["padded"] else 0
    return {"bytes": moved, "flops": 60 * cells}


def work(case):
    return _work_stack(case) if case["path"] == "stack" else _work_scan(case)


def tolerance(case):
    # About four times what the path differs by from itself in float64 (scan), with its products'
    # sums in double (float32 stacks) or in float32 throughout (16-bit stacks), on the listed cases;
    # a 16-bit stack's error grows with its depth, 16-bit scans show the rounding of their results.
    if case["path"] == "scan":
        return {"float32": {"rel": 2e-6, "max": 6e-5}, "bfloat16": {"rel": 7e-3, "max": 2e-2},
                "float16": {"rel": 9e-4, "max": 2e-3}}[case["dtype"]]
    if case["autocast"]:
        return {"rel": 3e-2, "max": 3e-1}
    return {"float32": {"rel": 5e-6, "max": 5e-5}, "bfloat16": {"rel": 2e-2, "max": 1e-1},
            "float16": {"rel": 3e-3, "max": 5e-2}}[case["weights"]]
