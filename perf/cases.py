"""The work a user of this package has it do, as cases that can be timed one by one.

Each case is one layer's share of a training step (its gradient dot products and train
gradients, or its gradient projection) through the functions the engines' backward hooks
call, or one whole engine step.  Sizes are those of the benchmark configurations (an MLP, the
Linear microbench, GPT-2-small, GPT-2-medium projections, Pythia-1B) and, in ``draw``, the
ranges around them: sequence lengths from one token up, batches of any train / val split,
feature counts that are odd or ragged, bf16 and fp32.

``exact`` forms the same results in float64 with plain torch.
"""
from __future__ import annotations

import contextlib
import math
from types import SimpleNamespace

import torch
import torch.nn.functional as F
from torch import nn

from ghostsuite_amd import GradDotProdEngine, _native
from ghostsuite_amd import autograd_grad_sample_dotprod as hooks
from ghostsuite_amd import supported_layers_grad_samplers_dotprod as samplers
from ghostsuite_amd.gradProjection.autograd_gradproj import create_projection_hooks
from ghostsuite_amd.gradProjection.projection_utils import choose_ki_ko
from ghostsuite_amd.workloads import MLP, CausalLM, LMConfig

DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


# ------------------------------------------------------------------------------ the cases
def _linear(n_train, n_val, T, d_in, d_out, dtype="bf16", bias=True, conv1d=False):
    """One Linear (or HF Conv1D) layer's backward hook.  T = 0: 2-D inputs [N, d]."""
    return {"kind": "linear", "n_train": n_train, "n_val": n_val, "T": T, "d_in": d_in,
            "d_out": d_out, "dtype": dtype, "bias": bias, "conv1d": conv1d}


def _pairs(n_train, n_val, T, d_in, d_out):
    return {"kind": "pairs", "n_train": n_train, "n_val": n_val, "T": T, "d_in": d_in,
            "d_out": d_out, "dtype": "bf16"}


def _layernorm(n_train, n_val, T, d, dtype="bf16"):
    return {"kind": "layernorm", "n_train": n_train, "n_val": n_val, "T": T, "d": d,
            "dtype": dtype}


def _embedding(n_train, n_val, T, d, vocab, dtype="bf16", pad=0.0):
    return {"kind": "embedding", "n_train": n_train, "n_val": n_val, "T": T, "d": d,
            "vocab": vocab, "dtype": dtype, "pad": pad}


def _kron(B, T, n_i, n_o, k_i, k_o, dtype="bf16"):
    return {"kind": "kron", "B": B, "T": T, "n_i": n_i, "n_o": n_o, "k_i": k_i, "k_o": k_o,
            "dtype": dtype}


def _kron_embedding(B, T, vocab, d, k_i, k_o, dtype="bf16"):
    return {"kind": "kron_embedding", "B": B, "T": T, "vocab": vocab, "d": d, "k_i": k_i,
            "k_o": k_o, "dtype": dtype}


def listed():
    """The listed cases, smallest first."""
    def named(name, case):
        return dict(case, name=name)

    # choose_ki_ko's answer for a GPT-2-medium qkv layer at the documented rank 512, k_min 8
    k_i, k_o = choose_ki_ko(1024, 3072, 512, 8)
    return [
        # The CPU-runnable plumbing configuration: a whole engine step of a small fp32 MLP,
        # where launches and host work count.
        named("mlp_step", {"kind": "mlp_step", "n_train": 64, "n_val": 16,
                           "dims": "512,1024,1024,10"}),
        # GPT-2-small's LayerNorm (25 of them a step), 16 train + 4 val rows.
        named("layernorm", _layernorm(16, 4, 1024, 768)),
        # GPT-2-small's token embedding: dot and untied train gradient.
        named("embedding", _embedding(16, 4, 1024, 768, 50257)),
        # A short-sequence batch (the microbench's T = 128 point) through the whole hook.
        named("linear_short", _linear(24, 8, 128, 768, 3072)),
        # A tokenised batch padded to its own longest row: an odd T and an odd split.
        named("linear_ragged", _linear(13, 3, 777, 768, 2304)),
        # The fp32 mode on a GPT-2-small projection at T = 256.
        named("linear_fp32", _linear(16, 4, 256, 768, 768, dtype="fp32")),
        # GPT-2-small's MLP input layer: the flagship training step's largest layer.
        named("linear_fc", _linear(16, 4, 1024, 768, 3072)),
        # Gradient projection of a GPT-2-medium MLP input layer, 16 x 16 per layer.
        named("kron_fc", _kron(32, 1024, 1024, 4096, 16, 16)),
        # ... and of its qkv layer at the projection sizes the rank rule picks.
        named("kron_rank", _kron(32, 1024, 1024, 3072, k_i, k_o)),
        # The Linear microbench: every val x train pair, val rows first in the batch.
        named("linear_pairs", _pairs(24, 8, 1024, 768, 3072)),
        # Pythia-1B's MLP input layer at T = 2048.
        named("linear_pythia_fc", _linear(8, 2, 2048, 2048, 8192)),
        # A whole bf16 GradDotProd step of a four-layer GPT-2 (width 768, T = 512).
        named("lm_step", {"kind": "lm_step", "n_train": 8, "n_val": 2, "T": 512, "layers": 4,
                          "vocab": 8192}),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges."""
    limit = max(work(c)["flops"] for c in listed())
    while True:
        case = _draw(rng)
        if work(case)["flops"] <= limit and work(case)["bytes"] <= 1.5e9:
            return case


def _draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "pairs", "layernorm",
                       "embedding", "kron", "kron", "kron_embedding", "mlp_step"])
    n_train, n_val = _log_int(rng, 2, 48), rng.randint(1, 8)
    T = _log_int(rng, 16, 2048)
    if rng.random() < 0.4:                     # a power of two or a multiple of 64
        T = rng.choice([32, 64, 128, 192, 256, 384, 512, 768, 1024, 2048])
    width = rng.choice([256, 320, 512, 640, 768, 1000, 1024, 1280, 1536, 2048])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
    if kind in ("linear", "pairs"):
        d_in, d_out = width, rng.choice([width, 3 * width, 4 * width])
        if rng.random() < 0.3:
            d_in, d_out = d_out, d_in
        if kind == "pairs":
            return _pairs(min(n_train, 24), n_val, min(T, 1024), min(d_in, 2048),
                          min(d_out, 3072))
        if rng.random() < 0.15:                # a 2-D classifier layer or head
            return _linear(_log_int(rng, 16, 512), rng.randint(4, 64), 0, width,
                           rng.choice([10, 100, 1000, width]), dtype="fp32")
        if dtype == "fp32":
            T = min(T, 512)
        return _linear(n_train, n_val, T, d_in, d_out, dtype, bias=rng.random() < 0.8,
                       conv1d=rng.random() < 0.25)
    if kind == "layernorm":
        return _layernorm(n_train, n_val, T, rng.choice([width, width + 12, 4 * width]), dtype)
    if kind == "embedding":
        return _embedding(n_train, n_val, T, width, rng.choice([1024, 8192, 30522, 50257]),
                          dtype, pad=rng.choice([0.0, 0.0, 0.3, 0.9]))
    if kind in ("kron", "kron_embedding"):
        B, n_o = _log_int(rng, 4, 48), rng.choice([width, 3 * width, 4 * width])
        rank = rng.choice([64, 256, 512, 1024])
        T = min(T, 1024)
        if kind == "kron_embedding":
            vocab = rng.choice([1024, 8192, 50257])
            return _kron_embedding(B, T, vocab, width, *choose_ki_ko(vocab, width, rank, 8),
                                   dtype)
        return _kron(B, T, width, n_o, *choose_ki_ko(width, n_o, rank, 8), dtype)
    hidden = rng.choice([128, 256, 500, 1024])
    return {"kind": "mlp_step", "n_train": _log_int(rng, 16, 256), "n_val": rng.randint(4, 64),
            "dims": "%d,%d,%d,10" % (rng.choice([64, 512, 784]), hidden, hidden)}


def _dims(case):
    return [int(d) for d in case["dims"].split(",")]


def work(case):
    """Bytes (each input read once, each output written once) and flops of one pass, the
    dots by the cheapest algorithm of the same semantics."""
    k = case["kind"]
    e = 4 if case.get("dtype", "bf16") == "fp32" else 2
    if k in ("linear", "pairs"):
        n_t, n_v, T = case["n_train"], case["n_val"], max(case["T"], 1)
        d, p = case["d_in"], case["d_out"]
        rows = (n_t + n_v) * T
        gemm = 2.0 * T * d * p                       # one sample's gradient
        if k == "pairs":
            flops = min(2.0 * n_t * n_v * T * T * (d + p),
                        (n_t + n_v) * gemm + 2.0 * n_t * n_v * d * p)
            return {"bytes": rows * (d + p) * e + 4.0 * n_t * (n_v + 1), "flops": flops}
        nv = n_v if _pairwise(case) else 1
        # the train gradient, then the dots from V or from the token Grams
        flops = n_t * gemm + min(nv * gemm + 2.0 * n_t * d * p,
                                 2.0 * n_t * nv * T * T * (d + p))
        return {"bytes": rows * (d + p) * e + d * p * e + 8.0 * n_t, "flops": flops}
    if k == "layernorm":
        n = (case["n_train"] + case["n_val"]) * case["T"] * case["d"]
        return {"bytes": 2.0 * n * e + 2.0 * case["d"] * e, "flops": 10.0 * n}
    if k == "embedding":
        n = (case["n_train"] + case["n_val"]) * case["T"]
        return {"bytes": n * (case["d"] * e + 8.0) + case["vocab"] * case["d"] * e,
                "flops": 3.0 * n * case["d"]}
    if k == "kron":
        n = case["B"] * case["T"]
        return {"bytes": n * (case["n_i"] + case["n_o"]) * e +
                4.0 * case["B"] * case["k_i"] * case["k_o"],
                "flops": 2.0 * n * (case["n_i"] * case["k_i"] + case["n_o"] * case["k_o"] +
                                    case["k_i"] * case["k_o"])}
    if k == "kron_embedding":
        n = case["B"] * case["T"]
        return {"bytes": n * (case["d"] * e + 8.0 + case["k_i"] * e) +
                4.0 * case["B"] * case["k_i"] * case["k_o"],
                "flops": 2.0 * n * (case["d"] * case["k_o"] + case["k_i"] * case["k_o"])}
    if k == "mlp_step":
        d, N = _dims(case), case["n_train"] + case["n_val"]
        w = sum(a * b + b for a, b in zip(d, d[1:]))
        return {"bytes": 4.0 * (2 * w + N * (d[0] + d[-1])), "flops": 6.0 * N * w}
    N, T, L, V = case["n_train"] + case["n_val"], case["T"], case["layers"], case["vocab"]
    w = L * 12 * 768 * 768 + V * 768
    # forward, input gradients, train gradients, and the val half of the dots
    return {"bytes": 2.0 * (2 * w + N * T * V),
            "flops": 6.0 * w * N * T + L * 12.0 * T * T * 768 * N}


def tolerance(case):
    """What another correct implementation at the same precision shows, times about four."""
    k = case["kind"]
    if k == "lm_step":
        # 16-bit activations through four layers: 0.9% measured against float64
        return {"rel": 4e-2}
    if k in ("mlp_step", "kron", "kron_embedding") or case["dtype"] == "fp32":
        # 32-bit results of 32-bit sums: up to 1e-6 measured
        return {"rel": 1e-5, "max": 1e-3}
    # bf16 results of 32-bit sums (0.17%); dots through a term held in bf16 (up to 0.26%)
    return {"rel": 8e-3, "max": 5e-2}


# ------------------------------------------------------------------------ states and passes
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, shape, scale, dtype):
    return (torch.randn(shape, generator=g, device="cuda") * scale).to(dtype)


def _hooked(layer, precision):
    """The layer as an engine leaves it: its trainability noted on its parameters."""
    for p in layer.parameters():
        p.initially_requires_grad = True
    return layer, precision


def _make_layer(case, dtype):
    with torch.device("cuda"):
        if case["kind"] == "layernorm":
            return nn.LayerNorm(case["d"], dtype=dtype)
        if case["kind"] == "embedding":
            return nn.Embedding(case["vocab"], case["d"], dtype=dtype)
        if case["conv1d"]:
            from transformers.pytorch_utils import Conv1D
            layer = Conv1D(case["d_out"], case["d_in"]).to(dtype)
            if not case["bias"]:
                layer.register_parameter("bias", None)
            return layer
        return nn.Linear(case["d_in"], case["d_out"], bias=case["bias"], dtype=dtype)


def _acts(case, seed):
    """Layer inputs ~ N(0, 1) and output gradients ~ N(0, 1e-3^2), as in the microbench; the
    rows share a weak common direction, so that a dot holds signal and noise alike."""
    g = _gen(seed)
    dtype = DTYPES[case["dtype"]]
    N = case["n_train"] + case["n_val"]
    d_in = case["d_in"] if "d_in" in case else case["d"]
    d_out = case["d_out"] if "d_out" in case else case["d"]
    rows = (N, case["T"]) if case["T"] else (N,)
    common = torch.randn(d_out, generator=g, device="cuda") * 2e-5
    A = _randn(g, rows + (d_in,), 1.0, torch.float32)
    A += 0.02
    G = _randn(g, rows + (d_out,), 1e-3, torch.float32)
    G += common
    return A.to(dtype), G.to(dtype)


def _tokens(case, seed):
    """Uniform ids, a share `pad` of them one padding id."""
    g = _gen(seed + 1)
    n = (case.get("B") or case["n_train"] + case["n_val"], case["T"])
    ids = torch.randint(0, case["vocab"], n, generator=g, device="cuda")
    if case.get("pad"):
        ids[torch.rand(n, generator=g, device="cuda") < case["pad"]] = 0
    return ids


def _projections(case, seed):
    g = _gen(seed + 2)
    n_i = case["n_i"] if case["kind"] == "kron" else case["vocab"]
    n_o = case["n_o"] if case["kind"] == "kron" else case["d"]
    return (_randn(g, (case["k_i"], n_i), case["k_i"] ** -0.5, torch.float32),
            _randn(g, (case["k_o"], n_o), case["k_o"] ** -0.5, torch.float32))


def _kron_inputs(case, seed):
    g = _gen(seed)
    dtype = DTYPES[case["dtype"]]
    B, T = case["B"], case["T"]
    if case["kind"] == "kron_embedding":
        return _tokens(case, seed), _randn(g, (B, T, case["d"]), 1e-3, dtype)
    return (_randn(g, (B, T, case["n_i"]), 1.0, dtype),
            _randn(g, (B, T, case["n_o"]), 1e-3, dtype))


def prepare(case, seed):
    k = case["kind"]
    s = SimpleNamespace(kind=k, case=case)
    torch.manual_seed(seed)
    if k in ("linear", "layernorm"):
        s.A, s.G = _acts(case, seed)
    elif k == "embedding":
        s.A, s.G = _tokens(case, seed), _acts(case, seed)[1]
    elif k == "pairs":
        s.A, s.G = _acts(case, seed)
    elif k in ("kron", "kron_embedding"):
        s.A, s.G = _kron_inputs(case, seed)
        P_i, P_o = _projections(case, seed)
        with torch.device("meta"):
            s.module = nn.Linear(case["n_i"], case["n_o"]) if k == "kron" else \
                nn.Embedding(case["vocab"], case["d"])
        s.hooks = create_projection_hooks(s.module, k, P_i, P_o)
    elif k == "mlp_step":
        _prepare_mlp(s, seed)
    else:
        _prepare_lm(s, seed)
    if k in ("linear", "layernorm", "embedding"):
        s.layer, s.precision = _hooked(_make_layer(case, DTYPES[case["dtype"]]),
                                       "fp32" if case["dtype"] == "fp32" else "reference")
    return s


def _prepare_mlp(s, seed):
    dims, N = _dims(s.case), s.case["n_train"] + s.case["n_val"]
    with torch.device("cuda"):
        s.model = MLP(dims)
    g = _gen(seed)
    s.X = torch.randn(N, dims[0], generator=g, device="cuda")
    s.Y = torch.randint(0, dims[-1], (N,), generator=g, device="cuda")
    s.opt = torch.optim.SGD(s.model.parameters(), lr=0.1)
    s.engine = GradDotProdEngine(s.model, val_batch_size=s.case["n_val"], use_dummy_bias=False,
                                 precision="fp32")
    s.engine.attach(s.opt)


def _lm_config(case):
    return LMConfig(n_layer=case["layers"], vocab=case["vocab"], n_ctx=case["T"])


def _prepare_lm(s, seed):
    N, T = s.case["n_train"] + s.case["n_val"], s.case["T"]
    with torch.device("cuda"):
        s.model = CausalLM(_lm_config(s.case)).to(torch.bfloat16)
    tokens = torch.randint(0, s.case["vocab"], (N, T + 1), generator=_gen(seed), device="cuda")
    s.X, s.Y = tokens[:, :T].contiguous(), tokens[:, 1:].contiguous()
    s.opt = torch.optim.SGD(s.model.parameters(), lr=0.1)
    s.engine = GradDotProdEngine(s.model, val_batch_size=s.case["n_val"], use_dummy_bias=True)
    s.engine.attach(s.opt)


@contextlib.contextmanager
def _options(**values):
    """The sampler options of one layer's hook, put back afterwards."""
    saved = dict(samplers.options)
    samplers.options.update(samplers.DEFAULT_OPTIONS)
    samplers.options.update(values)
    try:
        yield
    finally:
        samplers.options.update(saved)


def _run_hook(s):
    """The two stages of a layer's backward hook, on the current stream, as a training loop
    that owns its streams calls them."""
    layer, n_val = s.layer, s.case["n_val"]
    with _options(overlap=False, precision=s.precision):
        hooks._capture_activations(layer, (s.A,), None)
        hooks._prepare_sample_grad_or_dotprod(layer, (s.G,), n_val)
        hooks._apply_train_grad(layer, n_val)
    out = []
    for p in layer.parameters():
        out += [p.grad_dot_prod, p.train_grad]
        del p.grad_dot_prod, p.train_grad
    return out


def _run_step(s, loss_of):
    """One engine step up to the optimizer's update: logits, the logged dot products (one
    per train row) and every parameter's gradient."""
    n_t = s.case["n_train"]
    s.opt.zero_grad(set_to_none=True)
    s.engine.attach_train_batch(s.X[:n_t], s.Y[:n_t], 0, 0)
    logits = s.model(s.X)
    loss_of(logits, s.Y).backward()
    s.engine.prepare_gradients()
    named = [(n, p) for n, p in s.model.named_parameters() if "dummy_bias" not in n]
    total = named[0][1].grad_dot_prod          # the aggregate is summed into the first
    s.engine.aggregate_and_log()
    s.engine.clear_gradients()
    s.engine.dot_product_log.clear()
    return [logits.detach(), total] + [p.grad for _, p in named]


def _mlp_loss(logits, Y):
    return F.cross_entropy(logits, Y)


def _lm_loss(logits, Y):
    return F.cross_entropy(logits.float().view(-1, logits.shape[-1]), Y.reshape(-1))


def run(s):
    k, c = s.kind, s.case
    if k in ("linear", "layernorm", "embedding"):
        return _run_hook(s)
    if k == "pairs":
        return _native.ops().linear_dot(s.A, s.G, c["n_val"], val_start=0, want_pair=True)
    if k == "kron":
        s.hooks._compute_dense_proj(s.module, s.A, s.G)
        return s.module._ghost_grad_proj
    if k == "kron_embedding":
        s.hooks._compute_embedding_proj(s.module, s.A, s.G)
        return s.module._ghost_grad_proj
    return _run_step(s, _mlp_loss if k == "mlp_step" else _lm_loss)


# ----------------------------------------------------------------------------- float64 forms
def _pairwise(case):
    """The reference's rule for a Linear's val term: pairwise up to 2 T^2 = the weight's size,
    else the val rows summed first (always, for a Conv1D)."""
    T = max(case["T"], 1)
    return not case["conv1d"] and 2 * T * T <= case["d_in"] * case["d_out"]


def _rows3(x):
    return x.reshape(x.shape[0], -1, x.shape[-1]).double()


def _per_sample(A, G):
    """[N, d_out, d_in] per-sample weight gradients, one at a time."""
    return (g.t() @ a for a, g in zip(_rows3(A), _rows3(G)))


def _linear_exact(A, G, n_val, pairwise):
    """Weight dots, weight gradient (scaled N / n_train), bias dots, bias gradient."""
    N = A.shape[0]
    n_t = N - n_val
    if pairwise:
        V = sum(_per_sample(A[n_t:], G[n_t:]))
    else:
        V = _rows3(G[n_t:]).sum(0).t() @ _rows3(A[n_t:]).sum(0)
    dots, W = [], torch.zeros_like(V)
    for M in _per_sample(A[:n_t], G[:n_t]):
        dots.append((M * V).sum())
        W += M
    b = _rows3(G).sum(1)
    return (torch.stack(dots), W * (N / n_t), b[:n_t] @ b[n_t:].sum(0),
            b[:n_t].sum(0) * (N / n_t))


def _embedding_exact(ids, G, n_val, vocab):
    N, d = G.shape[0], G.shape[-1]
    n_t = N - n_val
    G3, ids2 = _rows3(G), ids.reshape(N, -1)
    zeros = torch.zeros(vocab, d, dtype=torch.float64, device=G.device)
    V = zeros.index_add(0, ids2[n_t:].reshape(-1), G3[n_t:].reshape(-1, d))
    dots = torch.stack([(V[i] * g).sum() for i, g in zip(ids2[:n_t], G3[:n_t])])
    W = zeros.index_add(0, ids2[:n_t].reshape(-1), G3[:n_t].reshape(-1, d))
    return dots, W * (N / n_t)


def _layernorm_exact(X, G, n_val, eps):
    N = X.shape[0]
    n_t = N - n_val
    G3 = _rows3(G)
    gx = (G3 * F.layer_norm(_rows3(X), (X.shape[-1],), eps=eps)).sum(1)
    gb = G3.sum(1)
    out = []
    for x in (gx, gb):
        out += [x[:n_t] @ x[n_t:].sum(0), x[:n_t].sum(0) * (N / n_t)]
    return out


def _mlp_exact(case, seed):
    s = SimpleNamespace(case=case)
    torch.manual_seed(seed)
    _prepare_mlp(s, seed)
    lin = [m for m in s.model.modules() if isinstance(m, nn.Linear)]
    x, acts, zs = s.X.double(), [], []
    for i, m in enumerate(lin):
        acts.append(x)
        z = (x @ m.weight.detach().double().t() + m.bias.detach().double()).requires_grad_()
        zs.append(z)
        x = z.relu() if i + 1 < len(lin) else z
    grads = torch.autograd.grad(F.cross_entropy(zs[-1], s.Y), zs)
    total, out = 0, []
    for a, g in zip(acts, grads):
        dw, gw, db, gb = _linear_exact(a.detach(), g, case["n_val"], True)
        total = total + dw + db
        out += [gw, gb]
    s.engine.detach()
    return [zs[-1].detach(), total] + out


def _lm_exact(case, seed):
    """The GPT-2 forward in float64 from the bf16 weights, every sampled layer's input and
    output gradient kept, then the layers' closed forms."""
    s = SimpleNamespace(case=case)
    torch.manual_seed(seed)
    _prepare_lm(s, seed)
    n_v, T, cfg = case["n_val"], case["T"], _lm_config(case)
    params = {n: p.detach().double() for n, p in s.model.named_parameters()}
    eps = s.model.ln_f.eps
    names = [n for n in params if "dummy_bias" not in n]
    s.engine.detach()
    N, d, H = s.X.shape[0], cfg.d_model, cfg.n_head
    taps = []                                       # (kind, layer, input, output)

    def tap(kind, name, x, y):
        y.retain_grad()
        taps.append((kind, name, x.detach(), y))
        return y

    def linear(name, x):
        b = params.get(name + ".bias")
        y = x @ params[name + ".weight"].t()
        return tap("linear", name, x, y if b is None else y + b)

    def norm(name, x):
        return tap("layernorm", name, x, F.layer_norm(
            x, (d,), params[name + ".weight"], params[name + ".bias"], eps))

    def embed(name, ids):
        return tap("embedding", name, ids, params[name + ".weight"][ids].requires_grad_())

    pos = torch.arange(T, device="cuda").repeat(N, 1)
    x = embed("wte", s.X) + embed("wpe", pos)
    causal = torch.full((T, T), float("-inf"), dtype=torch.float64, device="cuda").triu(1)
    for i in range(cfg.n_layer):
        q, kk, v = (t.reshape(N, T, H, d // H).transpose(1, 2).contiguous() for t in
                    linear(f"h.{i}.qkv", norm(f"h.{i}.ln_1", x)).split(d, dim=-1))
        att = (q @ kk.transpose(-1, -2).contiguous()) / math.sqrt(d // H) + causal
        y = (att.softmax(-1) @ v).transpose(1, 2).reshape(N, T, d)
        x = x + linear(f"h.{i}.proj", y)
        h = F.gelu(linear(f"h.{i}.fc", norm(f"h.{i}.ln_2", x)), approximate="tanh")
        x = x + linear(f"h.{i}.fc_out", h)
    h = norm("ln_f", x)
    logits = h @ params["wte.weight"].t()           # the tied head
    logits.retain_grad()
    F.cross_entropy(logits.reshape(-1, logits.shape[-1]), s.Y.reshape(-1)).backward()

    total = 0
    grads = {"wte.weight": _linear_exact(h.detach(), logits.grad, n_v, True)[1]}
    for kind, name, inp, out in taps:
        w, b = name + ".weight", name + ".bias"
        if kind == "linear":
            dw, gw, db, gb = _linear_exact(inp, out.grad, n_v, True)
        elif kind == "layernorm":
            dw, gw, db, gb = _layernorm_exact(inp, out.grad, n_v, eps)
        else:
            (dw, gw), db = _embedding_exact(inp, out.grad, n_v, params[w].shape[0]), 0
        total = total + dw + db
        grads[w] = grads[w] + gw if w in grads else gw
        if kind != "embedding":
            grads[b] = gb
    return [logits.detach(), total] + [grads[n] for n in names]


def exact(case, seed):
    k = case["kind"]
    if k == "mlp_step":
        return _mlp_exact(case, seed)
    if k == "lm_step":
        return _lm_exact(case, seed)
    if k == "linear":
        A, G = _acts(case, seed)
        dw, gw, db, gb = _linear_exact(A, G, case["n_val"], _pairwise(case))
        gw = gw.t() if case["conv1d"] else gw
        return [dw, gw] + ([db, gb] if case["bias"] else [])
    if k == "layernorm":
        A, G = _acts(case, seed)
        return _layernorm_exact(A, G, case["n_val"], nn.LayerNorm(1).eps)
    if k == "embedding":
        return list(_embedding_exact(_tokens(case, seed), _acts(case, seed)[1], case["n_val"],
                                     case["vocab"]))
    if k == "pairs":
        A, G = _acts(case, seed)
        n_v = case["n_val"]
        vals = list(_per_sample(A[:n_v], G[:n_v]))
        pair = torch.stack([torch.stack([(M * V).sum() for V in vals])
                            for M in _per_sample(A[n_v:], G[n_v:])], dim=1)
        return pair.sum(0), pair
    A, G = _kron_inputs(case, seed)
    P_i, P_o = (p.to(DTYPES[case["dtype"]]).double() for p in _projections(case, seed))
    out = []
    for a, g in zip(A, G):
        a = a.double() @ P_i.t() if k == "kron" else P_i.t()[a]
        out.append((g.double() @ P_o.t()).t() @ a)
    return torch.stack(out) * (float(case["B"]) if k == "kron" else 1.0)
