"""Performance cases of the optimizer step: what a training program has this package do.

listed() names the cases, draw() gives more over the same ranges; prepare() makes what
the program holds before the call (parameters, state, gradients, the optimizer), run()
makes one pass through the public entry points and returns everything that it updated.
exact() is the same pass in float64 with plain torch.

Kinds:
  adamw   one FusedAdamW step (detector, unscale, AdamW, export) over a list of tensors
  grads   the stage-gradient window: every micro-batch accumulated, flag and norm
  fp8     block-scaled FP8 transport of weights: pack, then unpack
  orth    orthogonalize() of one gradient or a list
  hybrid  one HybridMuonAdamW step of a model of SwiGLU blocks, its norms and its embedding
  disk    the [3, N] state update of a host array, chunk by chunk (DiskState.update)
"""
import math

import numpy as np
import torch

from morph_amd import DynamicLossScale, FusedAdamW
from morph_amd.disk import gpu_disk_update
from morph_amd.fp8 import pack_fp8, unpack_fp8
from morph_amd.grads import StageGradients
from morph_amd.muon import HybridMuonAdamW, orthogonalize

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
HYPER = dict(lr=3e-4, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.1)
STEP = 100  # steps taken before the measured one: moments and bias corrections are past the start
COEFFS = (3.4445, -4.775, 2.0315)


# ---------------------------------------------------------------- the cases --
def listed():
    return [
        # a small model's parameter group, FP32 gradients left in p.grad, weight decay on
        # its 2-D tensors only: latency, launches and host work
        dict(name="adamw_small", kind="adamw", shapes="256x64,64x256,256,512x256,256x512,512",
             grad="f32", export="none", scale=0.0, arena=False, rows="all"),
        # the norms and biases of a 5B model, one tensor each: hundreds of small tensors
        dict(name="adamw_vectors", kind="adamw", shapes="3072*326", grad="f32", export="none",
             scale=0.0, arena=False, rows="all"),
        # one stage of the 5B model (gate, up, down), FP16 gradients under a dynamic loss
        # scale, FP16 compute copy: the step that a streamed training loop repeats
        dict(name="adamw_window", kind="adamw", shapes="6144x3072*2,3072x6144", grad="f16",
             export="f16", scale=65536.0, arena=True, rows="all"),
        # the tied embedding, BF16 gradients on the rows of a batch's tokens: the largest tensor
        dict(name="adamw_embedding", kind="adamw", shapes="65536x3072", grad="bf16", export="bf16",
             scale=0.0, arena=True, rows="tokens"),
        # the gradient window of one 5B stage over four micro-batches
        dict(name="grads_window", kind="grads", shapes="6144x3072*2,3072x6144", grad="f16",
             scale=65536.0, micro=4),
        # the FP8 transport of one 5B stage's weights, out and in
        dict(name="fp8_window", kind="fp8", shapes="6144x3072*2,3072x6144", dtype="f16"),
        # one small ragged gradient
        dict(name="orth_small", kind="orth", shapes="200x96"),
        # one feed-forward gradient of the 5B model
        dict(name="orth_ffn", kind="orth", shapes="6144x3072"),
        # a small model's whole step
        dict(name="hybrid_small", kind="hybrid", layers=4, d=192, ff=448, vocab=1000, stacked=False),
        # an ordinary model's whole step
        dict(name="hybrid_mid", kind="hybrid", layers=12, d=768, ff=2048, vocab=8192, stacked=False),
        # the 42 hidden matrices of the 5B model and a million other parameters: the largest step
        dict(name="hybrid_5b", kind="hybrid", layers=14, d=3072, ff=6144, vocab=310, stacked=True),
        # one feed-forward state file's update, state and gradient in host memory
        dict(name="disk_update", kind="disk", n=18874368, chunk=1048576),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _matrices(rng, most):
    """Shapes of one stage: gate, up, down of any width, and its norm."""
    d = _log(rng, 32, 3072)
    ff = min(6144, max(d, int(d * rng.uniform(1.3, 4))))
    if rng.random() < 0.5:
        d, ff = d // 8 * 8, ff // 8 * 8  # widths in use are multiples of 8, though not all
    layers = rng.randint(1, 3)
    while layers > 1 and layers * 3 * d * ff > most:
        layers -= 1
    return ",".join(f"{ff}x{d}*2,{d}x{ff},{d}" for _ in range(layers))


def draw(rng):
    kind = rng.choice(["adamw", "adamw", "grads", "fp8", "orth", "orth", "hybrid", "hybrid", "disk"])
    if kind == "adamw":
        form = rng.choice(["stage", "vectors", "embedding"])
        if form == "vectors":
            return dict(kind=kind, shapes=f"{_log(rng, 33, 6144)}*{_log(rng, 4, 400)}", grad="f32",
                        export="none", scale=0.0, arena=False, rows="all")
        if form == "embedding":
            return dict(kind=kind, shapes=f"{_log(rng, 300, 65536)}x{_log(rng, 32, 3072)}",
                        grad="bf16", export="bf16", scale=0.0, arena=True, rows="tokens")
        grad = rng.choice(["f16", "bf16", "f32"])
        return dict(kind=kind, shapes=_matrices(rng, 1 << 26), grad=grad,
                    export=rng.choice(["f16", "bf16"]) if grad != "f32" else "none",
                    scale=rng.choice([65536.0, 1024.0]) if grad == "f16" else 0.0,
                    arena=rng.random() < 0.5, rows="all")
    if kind == "grads":
        return dict(kind=kind, shapes=_matrices(rng, 1 << 26), grad=rng.choice(["f16", "bf16"]),
                    scale=rng.choice([65536.0, 128.0]), micro=rng.randint(1, 8))
    if kind == "fp8":
        d, ff = _log(rng, 32, 3072), _log(rng, 64, 6144)
        return dict(kind=kind, shapes=f"{ff}x{d}*2,{d}x{ff}", dtype=rng.choice(["f16", "bf16", "f32"]))
    if kind == "orth":
        d = _log(rng, 48, 3072)
        n = min(6144, int(d * rng.uniform(1, 4)))
        return dict(kind=kind, shapes=rng.choice([f"{d}x{n}", f"{n}x{d}", f"{n}x{d}*2,{d}x{n}"]))
    if kind == "hybrid":
        d = _log(rng, 64, 2048)
        ff = int(d * rng.uniform(1.5, 4))
        if rng.random() < 0.5:
            d, ff = d // 16 * 16, ff // 16 * 16
        return dict(kind=kind, layers=rng.randint(1, 12), d=d, ff=ff, vocab=_log(rng, 100, 16384),
                    stacked=rng.random() < 0.3)
    return dict(kind=kind, n=_log(rng, 5000, 18874368), chunk=1048576)


# ------------------------------------------------------------------ helpers --
def _shapes(text):
    """'6144x3072*2,3072' -> [(6144, 3072), (6144, 3072), (3072,)]"""
    out = []
    for item in text.split(","):
        size, _, count = item.partition("*")
        out += [tuple(int(x) for x in size.split("x"))] * int(count or 1)
    return out


def _numels(text):
    return [math.prod(s) for s in _shapes(text)]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _flat_views(shapes, gen, std):
    """One buffer that holds the tensors one after the other (each on 256 bytes), N(0, std)."""
    at, offsets = 0, []
    for s in shapes:
        offsets.append(at)
        at += -(-math.prod(s) // 64) * 64
    flat = torch.zeros(at, device="cuda")
    views = [flat[o:o + math.prod(s)].view(s) for o, s in zip(offsets, shapes)]
    for v in views:
        v.normal_(0.0, std, generator=gen)
    return flat, views


def _adamw_inputs(case, seed):
    """Masters, moments (as flat buffers with views) and gradients of an adamw case."""
    gen = _gen(seed)
    shapes = _shapes(case["shapes"])
    masters, ps = _flat_views(shapes, gen, 0.02)
    first, ms = _flat_views(shapes, gen, 2e-5)
    second, vs = _flat_views(shapes, gen, 1e-4)
    second.square_()
    dtype, scale = DTYPES[case["grad"]], case["scale"] or 1.0
    grads = []
    for s in shapes:
        std = 1e-4 * scale if case["scale"] else 1e-3
        if case["rows"] == "tokens":  # rows of a batch's tokens, Zipf-distributed
            p = torch.arange(1, s[0] + 1, device="cuda", dtype=torch.float64).pow(-1.1)
            ids = torch.multinomial(p / p.sum(), min(4096, s[0] * 4), replacement=True,
                                    generator=gen).unique()
            g = torch.zeros(s, dtype=dtype, device="cuda")
            g[ids] = (torch.randn((ids.numel(), s[1]), generator=gen, device="cuda") * std).to(dtype)
        else:
            g = (torch.randn(s, generator=gen, device="cuda") * std).to(dtype)
        grads.append(g)
    return dict(shapes=shapes, flat=(masters, first, second), ps=ps, ms=ms, vs=vs, grads=grads)


def _groups(ps):
    """Weight decay on the matrices only."""
    groups = [dict(params=[p for p in ps if p.dim() > 1]),
              dict(params=[p for p in ps if p.dim() == 1], weight_decay=0.0)]
    return [g for g in groups if g["params"]]


def _decays(case, p):
    return p.dim() > 1 and case["rows"] == "all"


class _Block(torch.nn.Module):
    def __init__(self, gate, up, down, norm=None):
        super().__init__()
        for name, w in (("gate", gate), ("up", up), ("down", down)):
            layer = torch.nn.Linear(w.shape[1], w.shape[0], bias=False, device="meta")
            layer.weight = torch.nn.Parameter(w)
            setattr(self, name, layer)
        if norm is not None:
            self.norm = torch.nn.Parameter(norm)


class _Model(torch.nn.Module):
    """SwiGLU blocks, each with its norm (or all norms stacked in one parameter), an embedding."""

    def __init__(self, views, layers, stacked):
        super().__init__()
        per = 3 if stacked else 4
        self.blocks = torch.nn.ModuleList(_Block(*views[per * i:per * (i + 1)]) for i in range(layers))
        self.embedding = torch.nn.Parameter(views[-1])
        if stacked:
            self.norms = torch.nn.Parameter(views[-2])


def _hybrid_shapes(case):
    d, ff, layers = case["d"], case["ff"], case["layers"]
    block = [(ff, d), (ff, d), (d, ff)]
    if case["stacked"]:
        return block * layers + [(layers, d), (case["vocab"], d)]
    return (block + [(d,)]) * layers + [(case["vocab"], d)]


def _hybrid_inputs(case, seed):
    gen = _gen(seed)
    shapes = _hybrid_shapes(case)
    flat, views = _flat_views(shapes, gen, 0.02)
    grads = [torch.randn(s, generator=gen, device="cuda") * 1e-3 for s in shapes]
    per = 3 if case["stacked"] else 4
    is_muon = [i % per < 3 and i < per * case["layers"] for i in range(len(shapes))]
    momenta = [torch.randn(s, generator=gen, device="cuda") * 2e-4
               for s, muon in zip(shapes, is_muon) if muon]
    return flat, views, grads, is_muon, momenta


def _disk_inputs(case, seed):
    rng = np.random.default_rng(seed)
    n = case["n"]
    state = rng.standard_normal((3, n), dtype=np.float32)
    state *= np.array([[0.02], [2e-5], [1e-4]], np.float32)
    state[2] *= state[2]
    return state, rng.standard_normal(n, dtype=np.float32) * np.float32(1e-4)


def _fp8_weights(case, seed):
    gen = _gen(seed)
    return [(torch.randn(s, generator=gen, device="cuda") * 0.02).to(DTYPES[case["dtype"]])
            for s in _shapes(case["shapes"])]


def _orth_grads(case, seed):
    gen = _gen(seed)
    return [torch.randn(s, generator=gen, device="cuda") * 1e-3 for s in _shapes(case["shapes"])]


def _micro_grads(case, seed):
    gen = _gen(seed)
    return [[(torch.randn(s, generator=gen, device="cuda") * 1e-4 * case["scale"])
             .to(DTYPES[case["grad"]]) for s in _shapes(case["shapes"])]
            for _ in range(case["micro"])]


# ------------------------------------------------------------ prepare and run --
def prepare(case, seed):
    kind = case["kind"]
    if kind == "adamw":
        x = _adamw_inputs(case, seed)
        ps = x["ps"]
        export = DTYPES.get(case["export"])
        scaler = DynamicLossScale(case["scale"]) if case["scale"] else None
        groups = _groups(ps) if case["rows"] == "all" else [dict(params=ps, weight_decay=0.0)]
        opt = FusedAdamW(groups, loss_scale=scaler, export_dtype=export, arena=case["arena"], **HYPER)
        order = [p for g in opt.param_groups for p in g["params"]]
        at = {id(p): i for i, p in enumerate(ps)}
        saved = opt.state_dict()
        for k, p in enumerate(order):
            i = at[id(p)]
            if not case["arena"]:  # the program keeps its moments in flat buffers of its own
                opt.state[p]["exp_avg"], opt.state[p]["exp_avg_sq"] = x["ms"][i], x["vs"][i]
            saved["state"][k] = dict(step=torch.tensor(float(STEP)), exp_avg=x["ms"][i],
                                     exp_avg_sq=x["vs"][i])
        opt.load_state_dict(saved)
        grads = [x["grads"][at[id(p)]] for p in order]
        if case["grad"] == "f32":
            for p, g in zip(order, grads):
                p.grad = g
            grads = None
        if case["arena"]:
            outs = dict(params=order, exp_avg=[opt.state[p]["exp_avg"] for p in order],
                        exp_avg_sq=[opt.state[p]["exp_avg_sq"] for p in order])
        else:
            outs = dict(zip(("params", "exp_avg", "exp_avg_sq"), x["flat"]))
        outs["exports"] = opt.exports
        return dict(kind=kind, opt=opt, grads=grads, outs=outs)
    if kind == "grads":
        micro = _micro_grads(case, seed)
        return dict(kind=kind, micro=micro, scale=case["scale"],
                    window=StageGradients(_shapes(case["shapes"]), "cuda"))
    if kind == "fp8":
        return dict(kind=kind, weights=_fp8_weights(case, seed), dtype=DTYPES[case["dtype"]])
    if kind == "orth":
        gs = _orth_grads(case, seed)
        return dict(kind=kind, grads=gs if len(gs) > 1 else gs[0])
    if kind == "hybrid":
        flat, views, grads, is_muon, momenta = _hybrid_inputs(case, seed)
        model = _Model(views, case["layers"], case["stacked"])
        opt = HybridMuonAdamW(model, lr=1e-3, muon_lr=0.02, weight_decay=0.01)
        of = {v.data_ptr(): g for v, g in zip(views, grads)}
        for p in model.parameters():
            p.grad = of[p.data_ptr()]
        state = opt.state_dict()
        order = {p.data_ptr(): i for i, p in enumerate(opt.muon)}
        muon_views = [v for v, muon in zip(views, is_muon) if muon]
        state["momentum"] = {order[v.data_ptr()]: m for v, m in zip(muon_views, momenta)}
        opt.load_state_dict(state)
        adam = [p for g in opt.adam.param_groups for p in g["params"]]
        return dict(kind=kind, opt=opt, flat=flat, model=model, adam=adam,
                    momenta=[order[v.data_ptr()] for v in muon_views])
    state, grad = _disk_inputs(case, seed)
    return dict(kind=kind, state=state, grad=torch.from_numpy(grad), chunk=case["chunk"])


def run(state):
    kind = state["kind"]
    if kind == "adamw":
        state["opt"].step(state["grads"])
        return state["outs"]
    if kind == "grads":
        window = state["window"].zero_()
        last = len(state["micro"]) - 1
        for k, grads in enumerate(state["micro"]):
            window.accumulate(grads, state["scale"], final=k == last)
        return dict(window=window.flat, norm_squared=window.norm_squared_tensor())
    if kind == "fp8":
        packed = [pack_fp8(w) for w in state["weights"]]
        return dict(packed=packed, weights=[unpack_fp8(b, s, state["dtype"]) for b, s in packed])
    if kind == "orth":
        return orthogonalize(state["grads"])
    if kind == "hybrid":
        opt = state["opt"]
        opt.step()
        return dict(params=state["flat"], momenta=[opt.momentum[i] for i in state["momenta"]],
                    exp_avg=[opt.adam.state[p]["exp_avg"] for p in state["adam"]],
                    exp_avg_sq=[opt.adam.state[p]["exp_avg_sq"] for p in state["adam"]])
    gpu_disk_update(state["state"], state["grad"], STEP, 1e-4, 0.75, state["chunk"])
    return state["state"]


# ------------------------------------------------------- work and tolerance --
def _ns_flops(rows, cols):
    """Five iterations of A = X X^T and B = c A A + b A (symmetric: half of each), X' = B X."""
    m, n = min(rows, cols), max(rows, cols)
    return 5 * (3 * m * m * n + m ** 3)


def work(case):
    kind = case["kind"]
    size = {"f32": 4, "f16": 2, "bf16": 2, "none": 0}
    if kind == "adamw":
        n = sum(_numels(case["shapes"]))
        return dict(bytes=n * (size[case["grad"]] + 24 + size[case["export"]]), flops=15 * n)
    if kind == "grads":
        n = sum(_numels(case["shapes"]))
        return dict(bytes=n * (case["micro"] * size[case["grad"]] + 4), flops=(2 * case["micro"] + 2) * n)
    if kind == "fp8":
        n = sum(_numels(case["shapes"]))
        return dict(bytes=n * (2 * size[case["dtype"]] + 2) + n // 256 * 8, flops=5 * n)
    if kind == "orth":
        n = sum(_numels(case["shapes"]))
        return dict(bytes=8 * n, flops=sum(_ns_flops(*s) for s in _shapes(case["shapes"])))
    if kind == "hybrid":
        layers, d, ff = case["layers"], case["d"], case["ff"]
        muon, adam = 3 * layers * d * ff, (layers + case["vocab"]) * d
        return dict(bytes=20 * muon + 28 * adam, flops=3 * layers * _ns_flops(d, ff) + 15 * adam)
    return dict(bytes=28 * case["n"], flops=15 * case["n"])


def tolerance(case):
    # AdamW, the gradient window, FP8 and the disk update round where torch's CPU ops do:
    # the same bits from every correct implementation (the FP64 norm up to its order).
    # Newton-Schulz is bf16: another order of the same FP32 sums moves roundings through
    # five iterations.
    kind = case["kind"]
    if kind == "grads":
        return {"rel": 1e-12, "max": 1e-11}
    if kind == "orth":  # measured: permuted sums move 0.1-0.55% of the norm, 4.5% of an element
        return {"rel": 0.02, "max": 0.2}
    if kind == "hybrid":  # the same of an update of lr / sqrt(d) = .02 / sqrt(d) beside masters of .02
        return {"rel": 0.02 / math.sqrt(case["d"]), "max": 0.2 / math.sqrt(case["d"])}
    return "exact"


# ------------------------------------------------------------- in 64 bits --
def _adamw64(p, m, v, g, lr, betas, eps, wd, step):
    b1, b2 = betas
    p, m, v, g = (t.double() for t in (p, m, v, g))
    p = p * (1 - lr * wd)
    m = m + (1 - b1) * (g - m)
    v = v * b2 + (1 - b2) * g * g
    d = v.sqrt() / math.sqrt(1 - b2 ** step) + eps
    return p - lr / (1 - b1 ** step) * m / d, m, v


def _orth64(g):
    x = g.double()
    x = x.t() if g.shape[0] > g.shape[1] else x
    x = x / (x.norm() + 1e-7)
    a, b, c = COEFFS
    for _ in range(5):
        s = x @ x.t()
        x = a * x + (b * s + c * s @ s) @ x
    return x.t() if g.shape[0] > g.shape[1] else x


def exact(case, seed):
    kind = case["kind"]
    if kind == "adamw":
        x = _adamw_inputs(case, seed)
        scale = case["scale"] or 1.0
        done = [_adamw64(p, m, v, g.double() / scale, HYPER["lr"], HYPER["betas"], HYPER["eps"],
                         HYPER["weight_decay"] if _decays(case, p) else 0.0, STEP + 1)
                for p, m, v, g in zip(x["ps"], x["ms"], x["vs"], x["grads"])]
        if not case["arena"]:
            outs = {}
            for k, name in enumerate(("params", "exp_avg", "exp_avg_sq")):
                flat = torch.zeros_like(x["flat"][0], dtype=torch.float64)
                at = 0
                for s, d in zip(x["shapes"], done):
                    n = math.prod(s)
                    flat[at:at + n] = d[k].reshape(-1)
                    at += -(-n // 64) * 64
                outs[name] = flat
        else:
            outs = None
        order = [i for i, p in enumerate(x["ps"]) if p.dim() > 1]
        order += [i for i, p in enumerate(x["ps"]) if p.dim() == 1]
        if outs is None:
            outs = {name: [done[i][k] for i in order]
                    for k, name in enumerate(("params", "exp_avg", "exp_avg_sq"))}
        outs["exports"] = [done[i][0] for i in order] if case["export"] != "none" else []
        return outs
    if kind == "grads":
        micro = _micro_grads(case, seed)
        flat = torch.cat([sum(g.double() / case["scale"] for g in gs).reshape(-1)
                          for gs in zip(*micro)])
        return dict(window=flat, norm_squared=flat.square().sum())
    if kind == "fp8":
        packed = [(None, torch.nn.functional.pad(w.double().reshape(-1), (0, -w.numel() % 256))
                   .view(-1, 256).abs().amax(1) / 448) for w in _fp8_weights(case, seed)]
        return dict(packed=packed, weights=[w.double().reshape(-1) for w in _fp8_weights(case, seed)])
    if kind == "orth":
        outs = [_orth64(g).contiguous() for g in _orth_grads(case, seed)]
        return outs if len(outs) > 1 else outs[0]
    if kind == "hybrid":
        flat, views, grads, is_muon, momenta = _hybrid_inputs(case, seed)
        out = torch.zeros_like(flat, dtype=torch.float64)
        new_momenta, first, second = [], [], []
        left = iter(momenta)
        for p, g, muon in zip(views, grads, is_muon):
            at = (p.data_ptr() - flat.data_ptr()) // 4
            if muon:
                g64, m = g.double(), next(left).double()
                m = m + 0.05 * (g64 - m)
                new_momenta.append(m)
                u = _orth64(g64 + 0.95 * (m - g64)) * math.sqrt(max(1.0, p.shape[0] / p.shape[1]))
                new = p.double() * (1 - 0.02 * 0.01) - 0.02 * u
            else:
                zero = torch.zeros_like(g)
                new, m, v = _adamw64(p, zero, zero, g, 1e-3, (0.9, 0.95), 1e-8, 0.01, 1)
                first.append(m)
                second.append(v)
            out[at:at + p.numel()] = new.reshape(-1)
        # model.parameters() puts the model's own tensors first: the embedding, then the norms
        first, second = first[-1:] + first[:-1], second[-1:] + second[:-1]
        return dict(params=out, momenta=new_momenta, exp_avg=first, exp_avg_sq=second)
    state, grad = _disk_inputs(case, seed)
    s = torch.from_numpy(state)
    g = torch.from_numpy(grad).double() * 0.75
    done = _adamw64(*s, g, 1e-4, (0.9, 0.999), 1e-8, 0.01, STEP)
    return torch.stack(done).numpy()
