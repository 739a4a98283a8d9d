"""The optimizer steps that a training program has this package do, for timing and comparison.

A case is one model's parameter list with the options it is trained with; a pass is one
``ApexW.step()`` (or the hybrid Muon step) in the middle of a run.  Parameters, grads and
optimizer state lie in flat buffers, one per state key and dtype, and the optimizer holds views
of them, as programs that shard, offload or checkpoint flat buffers keep them; a pass returns
the flat buffers it updated.

The parameter lists: an MLP (the smallest calls, where launches and host time count), a
convolutional network (many small 4-D weights), GPT-2-like and Llama-like transformers at sizes
from one narrow layer to Llama-3-8B, and thousands of ragged tensors.
"""

import math

import torch

import apexw_amd

LR, WD, EPS = 1e-3, 0.1, 1e-8
AMP_SCALE = 65536.0        # GradScaler's initial scale
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32, "fp16": torch.float16}
STEPS_BEFORE = 3           # steps that a prepared state has behind it
ALIGN = 256                # bytes: every tensor of a flat buffer starts on such a boundary


def _case(model, precision, dtype="bf16", **kw):
    c = dict(model=model, precision=precision, dtype=dtype, sr=True, clip=0.0, gc=False, factored=False, amp=False,
             muon=False, layers=0, width=0, kv=0, ffn=0, vocab=0, context=0, count=0, shapes=0)
    c.update(kw)
    return c


def listed():
    gpt2 = dict(layers=12, width=768, ffn=3072, vocab=50257, context=1024)
    llama = dict(width=4096, kv=1024, ffn=14336)
    return [
        # a small regression MLP in fp32: six tensors, 0.1 M parameters; launch and host latency
        dict(_case("mlp", "compact", "fp32", layers=3, width=256, ffn=100), name="mlp_compact"),
        # GPT-2-small pretrained in bf16 with the default precision
        dict(_case("gpt", "compact", **gpt2), name="gpt2_compact"),
        # the same model in fp32 with full-precision moments under autocast and GradScaler, clipped
        dict(_case("gpt", "full", "fp32", clip=1.0, amp=True, **gpt2), name="gpt2_full_amp"),
        # 20,000 tensors of 64 to 2^20 elements with the global-norm clip
        dict(_case("ragged", "compact", clip=1.0, count=20000, shapes=2), name="ragged_clip"),
        # Llama-3-8B, 8-bit: the headline configuration
        dict(_case("llama", "8bit", layers=32, vocab=128256, **llama), name="llama_8b_8bit"),
        # fine-tuning of the upper layers with INT8 m and a dense v
        dict(_case("llama", "ultra", layers=4, **llama), name="layers_ultra"),
        # 8-bit with grad centralization and the clip
        dict(_case("llama", "8bit", layers=4, clip=1.0, gc=True, **llama), name="layers_8bit_gc"),
        # 8-bit with a factored second moment
        dict(_case("llama", "8bit", layers=4, factored=True, **llama), name="layers_factored"),
        # an image classifier: 3 x 3 and 1 x 1 convolutions, norms, a head of 1000 classes (INT8 m)
        dict(_case("conv", "8bit", layers=16, width=64, vocab=1000), name="conv_8bit"),
        # hybrid Muon on a small MLP with odd widths
        dict(_case("mlp", "compact", "fp32", muon=True, layers=4, width=500, ffn=384), name="mlp_muon"),
        # hybrid Muon on GPT-2-small, every block matrix sent to Muon by its group's tag
        dict(_case("gpt", "compact", muon=True, **gpt2), name="gpt2_muon"),
        # hybrid Muon on one Llama-3-8B layer
        dict(_case("llama", "compact", muon=True, layers=1, **llama), name="layer_muon"),
    ]


def draw(rng):
    def logint(lo, hi, step=1):
        return max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi)))) // step * step)

    kind = rng.choice(["mlp", "gpt", "gpt_full", "ragged", "llama_8bit", "llama_ultra", "llama_gc", "llama_factored",
                       "conv", "mlp_muon", "gpt_muon", "llama_muon"])
    step = rng.choice([1, 2, 8, 64])
    if kind == "mlp":
        return _case("mlp", rng.choice(["compact", "auto", "full", "8bit"]), rng.choice(["bf16", "fp32", "fp16"]),
                     layers=rng.randint(2, 3), width=logint(24, 1500, step), ffn=logint(10, 1000),
                     sr=rng.random() < 0.7, clip=rng.choice([0.0, 1.0]))
    if kind in ("gpt", "gpt_full", "gpt_muon"):
        w = logint(96, 1280, rng.choice([8, 32, 64]))
        sizes = dict(layers=rng.randint(1, 12), width=w, ffn=4 * w, vocab=logint(1000, 50257), context=logint(64, 2048))
        if kind == "gpt":
            return _case("gpt", rng.choice(["compact", "compact", "auto"]), rng.choice(["bf16", "bf16", "fp32"]),
                         sr=rng.random() < 0.7, clip=rng.choice([0.0, 1.0]), gc=rng.random() < 0.2, **sizes)
        if kind == "gpt_full":
            return _case("gpt", "full", rng.choice(["fp32", "bf16"]), clip=rng.choice([0.0, 1.0]),
                         amp=rng.random() < 0.5, **sizes)
        return _case("gpt", "compact", rng.choice(["bf16", "fp32"]), muon=True, **sizes)
    if kind == "ragged":
        return _case("ragged", rng.choice(["compact", "8bit"]), count=logint(100, 8000), shapes=rng.randint(3, 1000),
                     clip=rng.choice([0.0, 1.0]))
    if kind == "conv":
        return _case("conv", rng.choice(["8bit", "compact", "ultra"]), layers=rng.randint(4, 24),
                     width=logint(16, 160, step), vocab=logint(10, 2000), sr=rng.random() < 0.7)
    if kind == "mlp_muon":
        return _case("mlp", "compact", rng.choice(["bf16", "fp32"]), muon=True, layers=rng.randint(2, 6),
                     width=logint(64, 2000, step), ffn=logint(40, 1500, step))
    w = logint(256, 4096, rng.choice([8, 64, 128]))
    sizes = dict(width=w, kv=max(w // rng.choice([1, 4, 8]), 32), ffn=logint(2 * w, 4 * w, rng.choice([1, 8, 64])))
    if kind == "llama_muon":
        return _case("llama", "compact", muon=True, layers=rng.randint(1, max(1, min(4, (4096 // w) ** 2 // 2))), **sizes)
    # at most a quarter of the largest listed case's parameters
    layers = rng.randint(1, max(1, min(16, 2 ** 31 // (4 * w * w + 3 * w * sizes["ffn"]) - 1)))
    if kind == "llama_8bit":
        return _case("llama", "8bit", layers=layers, vocab=logint(1000, 32000), sr=rng.random() < 0.7, **sizes)
    if kind == "llama_ultra":
        return _case("llama", "ultra", layers=layers, sr=rng.random() < 0.7, **sizes)
    if kind == "llama_gc":
        return _case("llama", "8bit", layers=layers, gc=True, clip=rng.choice([0.0, 1.0]), **sizes)
    return _case("llama", rng.choice(["8bit", "8bit", "compact"]), layers=layers, factored=True, **sizes)


# ---------------------------------------------------------------------------- parameter lists
def _shapes(c):
    """The case's parameter shapes, in the order that a model lists them."""
    w, f = c["width"], c["ffn"]
    if c["model"] == "mlp":
        # layers - 1 hidden layers of `width` units over `ffn` inputs, and an output of 10
        s = [(w, f), (w,)]
        for _ in range(c["layers"] - 2):
            s += [(w, w), (w,)]
        return s + [(10, w), (10,)]
    if c["model"] == "gpt":
        s = [(c["vocab"], w), (c["context"], w)]
        for _ in range(c["layers"]):
            s += [(w,), (w,), (w, 3 * w), (3 * w,), (w, w), (w,), (w,), (w,), (w, f), (f,), (f, w), (w,)]
        return s
    if c["model"] == "llama":
        s = [(c["vocab"], w)] if c["vocab"] else []
        for _ in range(c["layers"]):
            s += [(w, w), (c["kv"], w), (c["kv"], w), (w, w), (f, w), (f, w), (w, f), (w,), (w,)]
        return s + ([(w,), (c["vocab"], w)] if c["vocab"] else [])
    if c["model"] == "conv":
        # bottleneck blocks: 1 x 1, 3 x 3, 1 x 1 convolutions and their norms; the width doubles every quarter
        s = [(w, 3, 7, 7), (w,), (w,)]
        inp = w
        for i in range(c["layers"]):
            b = w << (4 * i // c["layers"])
            s += [(b, inp, 1, 1), (b,), (b,), (b, b, 3, 3), (b,), (b,), (4 * b, b, 1, 1), (4 * b,), (4 * b,)]
            inp = 4 * b
        return s + [(c["vocab"], inp), (c["vocab"],)]
    # ragged: element counts log-uniform in [64, 2^20], about half of them 2-D where they divide
    g = torch.Generator().manual_seed(c["shapes"])
    n = torch.exp(torch.rand(c["count"], generator=g, dtype=torch.float64) * math.log(2 ** 14) + math.log(64))
    twod = (torch.rand(c["count"], generator=g) < 0.5).tolist()
    s = []
    for k, t in zip(n.floor().long().tolist(), twod):
        r = 8
        while r * r < k and k % (r * 2) == 0:
            r *= 2
        s.append((r, k // r) if t and k % r == 0 else (k,))
    return s


def _numel(shape):
    return math.prod(shape)


def _goes_to_muon(c, shape):
    """Which parameters a case's Muon groups hold: every block matrix of the transformers and
    MLPs but embeddings and the output layer."""
    if not c["muon"] or len(shape) < 2 or min(shape) < 32:
        return False
    return not (c["model"] == "gpt" and shape in ((c["vocab"], c["width"]), (c["context"], c["width"])))


def _offsets(sizes, itemsize):
    """Element offsets of tensors of these sizes in one flat buffer, and its length."""
    unit = ALIGN // itemsize
    at, out = 0, []
    for n in sizes:
        out.append(at)
        at += (n + unit - 1) // unit * unit
    return out, at


# ---------------------------------------------------------------------------- inputs
def _tensors(case, seed, device):
    """(shapes, flat parameters, flat grads, their offsets): parameters ~N(0, 0.02); grads ~N(0, 1e-3)
    with a scale per tensor log-uniform in [0.1, 10], some of the ragged list's all zero; times the
    loss scale under GradScaler."""
    dt = DTYPES[case["dtype"]]
    shapes = _shapes(case)
    at, total = _offsets([_numel(s) for s in shapes], torch.tensor([], dtype=dt).element_size())
    gen = torch.Generator(device=device).manual_seed(seed)
    host = torch.Generator().manual_seed(seed)
    p = torch.empty(total, dtype=dt, device=device).normal_(0.0, 0.02, generator=gen)
    g = torch.empty(total, dtype=dt, device=device).normal_(0.0, 1e-3, generator=gen)
    scale = torch.exp((torch.rand(len(shapes), generator=host, dtype=torch.float64) * 2 - 1) * math.log(10.0))
    if case["model"] == "ragged":
        scale[torch.rand(len(shapes), generator=host) < 0.05] = 0.0
    if case["amp"]:
        scale *= AMP_SCALE
    torch._foreach_mul_([g[o:o + _numel(s)] for s, o in zip(shapes, at)], scale.tolist())
    return shapes, p, g, at


def _params(case, shapes, p, g, at):
    # 8-bit: plain shards whose grads the program assigns (as flat-sharding programs hold them), stepped
    # by step(); trainable ones would be stepped inside the backward
    out = []
    for s, o in zip(shapes, at):
        q = torch.nn.Parameter(p[o:o + _numel(s)].view(s), requires_grad=case["precision"] != "8bit")
        q.grad = g[o:o + _numel(s)].view(s)
        out.append(q)
    return out


def _optimizer(case, params):
    kw = dict(lr=LR, weight_decay=WD, eps=EPS, stochastic_rounding=case["sr"],
              clip_grad_norm=case["clip"] or None, grad_centralization=case["gc"])
    if case["muon"]:
        yes = [p for p in params if _goes_to_muon(case, tuple(p.shape))]
        no = [p for p in params if not _goes_to_muon(case, tuple(p.shape))]
        return apexw_amd.ApexW([dict(params=yes, use_muon=True), dict(params=no, use_muon=False)], use_muon=True,
                               lr=LR, weight_decay=WD, precision=case["precision"])
    return apexw_amd.ApexW(params, adamw_compat=True, precision=case["precision"], factored_v=case["factored"], **kw)


def _step(s):
    if s["amp"] is not None:
        # what torch's GradScaler hands to an optimizer that takes its scale
        s["opt"].grad_scale, s["opt"].found_inf = s["amp"]
    s["opt"].step()


def prepare(case, seed):
    device = torch.device("cuda", 0)
    shapes, p, g, at = _tensors(case, seed, device)
    torch.manual_seed(seed)      # the optimizer draws its rounding seed from torch's generator
    amp = None
    if case["amp"]:
        amp = (torch.full((), AMP_SCALE, device=device), torch.zeros((), device=device))
    # the run's first step, then its state moved into flat buffers, as a resumed run holds it
    first = _params(case, shapes, p, g, at)
    s = {"opt": _optimizer(case, first), "amp": amp}
    _step(s)
    states = [s["opt"].state[q] for q in first]
    flat = {}
    for st in states:
        for k, v in st.items():
            if torch.is_tensor(v) and v.is_cuda:
                flat.setdefault((k, v.dtype), []).append((st, k, v))
    out = {"p": p}
    for (k, dt), members in flat.items():
        offs, total = _offsets([v.numel() for _, _, v in members], members[0][2].element_size())
        buf = out["%s.%s" % (k, str(dt).replace("torch.", ""))] = torch.zeros(total, dtype=dt, device=device)
        for (st, key, v), o in zip(members, offs):
            view = buf[o:o + v.numel()].view(v.shape)
            view.copy_(v)
            st[key] = view
    params = _params(case, shapes, p, g, at)
    s = {"opt": _optimizer(case, params), "amp": amp, "out": out, "params": params, "grads": g}
    for q, st in zip(params, states):
        s["opt"].state[q] = dict(st)
    for _ in range(STEPS_BEFORE - 1):
        _step(s)
    return s


def run(state):
    _step(state)
    return state["out"]


# ---------------------------------------------------------------------------- what a pass needs
def _layouts(c):
    """Per parameter, how its second moment is held ("muon": none; "factored", "quad": one value for four
    consecutive elements, "full") and the bytes of its whole state."""
    shapes = _shapes(c)
    rest = [s for s in shapes if not _goes_to_muon(c, s)]
    thin = any(len(s) == 2 and min(s) <= 64 and max(s) >= 256 for s in rest)   # adapter-like models
    fp32_only = c["dtype"] == "fp32" and not c["amp"]
    v_bytes = 4 if not c["sr"] and not c["muon"] else 2       # beta2 = 0.999 without stochastic rounding
    out = []
    for s in shapes:
        n, rows = _numel(s), s[0]
        large = len(s) >= 2 or n >= 65536
        quads = n >= 16384 and n % 4 == 0 and (len(s) < 2 or min(s) >= 8)
        factored = c["factored"] and not thin and len(s) >= 2 and min(rows, n // rows) >= 128
        if _goes_to_muon(c, s):
            out.append(("muon", 4 * n))
        elif c["precision"] == "full" or (c["precision"] == "auto" and (fp32_only and not thin or not large)):
            out.append(("full", 8 * n))
        elif c["precision"] == "ultra":
            out.append(("full", (1 + v_bytes) * n + 4 * -(-n // (2048 if n >= 2048 else 256)) if large else 8 * n))
        elif c["precision"] == "8bit" and n >= 64:
            blocks = -(-n // next((b for b in (2048, 1024, 512, 256, 128) if n >= b), 64))
            if factored and n >= 65536:
                out.append(("factored", n + 4 * blocks + 4 * (rows + n // rows)))
            else:
                out.append(("quad", 3 * n // 4 + 8 * blocks) if quads else ("full", 2 * n + 8 * blocks))
        elif factored and n >= 524288:
            out.append(("factored", 2 * n + 4 * (rows + n // rows)))
        elif quads and v_bytes == 2 and c["precision"] != "8bit" and (thin or len(rest) >= 8):
            out.append(("quad", 2 * n + n // 2))
        else:
            out.append(("full", (2 + v_bytes) * n))
    return out


def work(case):
    """Bytes: p and the state read and written, the grad read, each once.  FLOPs of Muon: five
    Newton-Schulz iterations of A = X X^T, B = c A A + b A and X' = B X + a X on the m x k work
    matrix (m <= k), half of each symmetric product."""
    size = torch.tensor([], dtype=DTYPES[case["dtype"]]).element_size()
    bytes_, flops = 0, 0
    for s, (kind, state) in zip(_shapes(case), _layouts(case)):
        n = _numel(s)
        bytes_ += 3 * n * size + 2 * state
        if kind == "muon":
            m, k = min(s[0], n // s[0]), max(s[0], n // s[0])
            flops += 5 * (m * m * k + m ** 3 + 2 * m * m * k)
        else:
            flops += 12 * n
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """About four times what the same step shows when it is compiled with fused multiply-adds where the
    compiler sees them, and with the two halves of each matrix-core step of Newton-Schulz exchanged:
    single units of the 16-bit parameters and moments (rel up to 1.3e-5, max 0.0085 over a parameter's
    root mean square), codes on their boundary (6e-6 of them), bf16 products (rel 2e-3, max 0.03), and
    for fp32 states the order of the clip's sums."""
    if case["muon"]:
        return {"rel": 8e-3, "max": 0.12}
    if case["precision"] in ("8bit", "ultra"):
        return {"rel": 1e-4, "max": 3.5e-2, "differ": 3e-5}
    if case["dtype"] == "fp32" and case["precision"] == "full":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 1e-4, "max": 3.5e-2}


# ---------------------------------------------------------------------------- in 64 bits
def _newton_schulz(g):
    """The orthogonalised update of a 2-D grad."""
    x = g if g.shape[0] <= g.shape[1] else g.t()
    x = x / (x.norm() + 1e-7)
    for _ in range(5):
        a = x @ x.t()
        x = (2.0315 * (a @ a) - 4.7750 * a) @ x + 3.4445 * x
    return x if g.shape[0] <= g.shape[1] else x.t()


def exact(case, seed):
    """The parameters after the prepared steps and one pass, and the 16- and 32-bit moments, from the same
    grad at every step: then m = (1 - b1^t) g and v = (1 - b2^t) g^2.  Quantized moments and the scaled
    ones of fp16 parameters have no such value."""
    if sum(map(_numel, _shapes(case))) > 1_000_000_000:
        return None
    device = torch.device("cuda", 0)
    shapes, p, g, at = _tensors(case, seed, device)
    layouts = _layouts(case)
    p = p.double()
    steps, eight = STEPS_BEFORE + 1, case["precision"] == "8bit"
    b1, b2, mu = 0.9, 0.99 if case["muon"] else 0.999, 0.95
    grads = []
    for s, o in zip(shapes, at):
        x = g[o:o + _numel(s)].double().view(s) / (AMP_SCALE if case["amp"] else 1.0)
        if case["gc"] and len(s) >= 2:
            x = x - x.mean(dim=tuple(range(1, len(s))), keepdim=True)
        grads.append(x)
    if case["clip"]:
        norm = float(torch.stack([x.square().sum() for x in grads]).sum().sqrt())
        coef = min(case["clip"] / (norm + 1e-6), 1.0)
        grads = [x * coef for x in grads]
    moments = {"momentum": [], "exp_avg": [], "exp_avg_sq": []}
    for s, o, x, (kind, _) in zip(shapes, at, grads, layouts):
        n = _numel(s)
        q = p[o:o + n].view(s)
        if kind == "muon":
            # the rms-matched update at five times the learning rate
            u = _newton_schulz(x) * (0.2 * math.sqrt(max(s)))
            for _ in range(steps):
                q.mul_(1.0 - 5 * LR * WD).sub_(u, alpha=5 * LR)
            moments["momentum"].append((1.0 - mu ** steps) * x)
            continue
        second = x.square()
        if kind == "factored":
            row, col = second.view(s[0], -1).mean(1, keepdim=True), second.view(s[0], -1).mean(0, keepdim=True)
            second = (row / row.mean().clamp_min(1e-300) * col).view(s)
        elif kind == "quad":
            second = second.view(-1, 4).mean(1)
        moments["exp_avg"].append((1.0 - b1 ** steps) * x)
        moments["exp_avg_sq"].append((1.0 - b2 ** steps) * second)
        if kind == "quad":
            second = second.repeat_interleave(4).view(s)
        # the 8-bit step takes the lookahead lerp(g, m, b1), raised where m and g agree
        ahead = eight and n >= 64 and kind != "factored"
        decay = 1.0 if case["muon"] and len(s) < 2 else 1.0 - LR * WD
        for t in range(1, steps + 1):
            c1, c2 = 1.0 - b1 ** t, 1.0 - b2 ** t
            num = (1.0 - b1 ** (t + 1)) * (1.0 + 0.2 * b1) * x if ahead else c1 * x
            q.mul_(decay).sub_(num / ((c2 * second).sqrt() + EPS * math.sqrt(c2)), alpha=LR * math.sqrt(c2) / c1)
    out = {"p": p}
    if case["precision"] not in ("compact", "full") or case["dtype"] == "fp16" or case["factored"]:
        return out
    dense = "float32" if case["precision"] == "full" else "bfloat16"
    v_dense = dense if case["sr"] or case["muon"] else "float32"
    for k, dt in (("momentum", "float32"), ("exp_avg", dense), ("exp_avg_sq", v_dense)):
        if moments[k]:
            offs, total = _offsets([x.numel() for x in moments[k]], 2 if dt == "bfloat16" else 4)
            buf = out["%s.%s" % (k, dt)] = torch.zeros(total, dtype=torch.float64, device=device)
            for x, o in zip(moments[k], offs):
                buf[o:o + x.numel()] = x.reshape(-1)
    return out
