"""End-to-end GPU parity through the reference API: engines and hooks on small models, with
the HIP kernels underneath, checked against brute-force per-sample gradients (float64, CPU)."""
import copy

import pytest
import torch
import torch.nn.functional as F
from torch import nn

from ghostsuite_amd import GradDotProdEngine, GradProjLoraEngine
from ghostsuite_amd import supported_layers_grad_samplers_dotprod as S
from ghostsuite_amd.workloads import CausalLM, LMConfig, MLP, synthetic_tokens
from oracle import brute
from tests.helpers import BF16_TOL, FP32_TOL, assert_close, gen

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _reset_options():
    saved = dict(S.options)
    yield
    S.options.clear()
    S.options.update(saved)


def _lm_loss(T):
    return lambda m, x, y: m(x, y) * T


@pytest.mark.parametrize("precision,tol", [("fp32", FP32_TOL), ("reference", BF16_TOL)])
@pytest.mark.parametrize("algo", ["ghost", "valgrad"])
def test_gpt2_engine_on_gpu_matches_per_sample_gradients(gpu, precision, tol, algo):
    torch.manual_seed(12)
    T, vocab = 16, 64
    cfg = LMConfig(n_layer=2, n_head=2, d_model=32, d_mlp=64, vocab=vocab, n_ctx=T)
    model = CausalLM(cfg)
    untied = copy.deepcopy(model)
    untied.lm_head.weight = nn.Parameter(model.wte.weight.detach().clone())
    tied_ref = copy.deepcopy(model).double()
    untied = untied.double()
    n_t, n_v = 5, 2
    X, Y = synthetic_tokens(n_t + n_v, T, vocab, seed=13)
    model = model.to(gpu)
    opt = torch.optim.SGD(model.parameters(), lr=0.0)
    print(f"gpt2 engine precision={precision} algo={algo}", flush=True)
    eng = GradDotProdEngine(model, val_batch_size=n_v, use_dummy_bias=True, precision=precision,
                            linear_algo=algo)
    eng.attach(opt)
    eng.attach_train_batch(X[:n_t], Y[:n_t], 0, 0)
    model(X.to(gpu), Y.to(gpu)).backward()
    torch.cuda.synchronize()
    dots = {n: p.grad_dot_prod.cpu() for n, p in model.named_parameters()
            if hasattr(p, "grad_dot_prod")}
    semantics = {n: m.use_ghost_computation for n, m in model.named_modules()
                 if hasattr(m, "use_ghost_computation")}
    eng.prepare_gradients()
    grads = {n: p.grad.cpu() for n, p in model.named_parameters()
             if p.grad is not None and "dummy_bias" not in n}
    eng.aggregate_and_log()
    eng.detach()

    N = n_t + n_v
    g_untied = brute.per_sample_grads(untied, X, Y, _lm_loss(T), 1.0 / (N * T))
    g_tied = brute.per_sample_grads(tied_ref, X, Y, _lm_loss(T), 1.0 / (N * T))
    total = 0
    for name, d in dots.items():
        layer = name.rsplit(".", 1)[0]
        gr = g_untied[name]
        if semantics.get(layer, True):
            want = brute.pairwise_dots(gr, n_v)
        else:   # materialised branch: presum over val rows, <g_i, sum_j g_j> is the same here
            want = brute.pairwise_dots(gr, n_v) if n_v == 1 else None
        if want is None:
            continue
        assert_close(d, want, tol, f"dot {name}")
        total = total + want
    for name, gr in grads.items():
        assert_close(gr, brute.train_mean(g_tied[name], n_v, N), tol, f"grad {name}")


def _random_lm_configs(n, seed):
    g = torch.Generator().manual_seed(seed)
    pick = lambda opts: opts[int(torch.randint(0, len(opts), (1,), generator=g))]
    out = []
    for _ in range(n):
        n_head, hd = pick([1, 2, 4]), pick([8, 16])
        T = pick([3, 7, 12, 24])
        cfg = LMConfig(n_layer=pick([1, 2]), n_head=n_head, d_model=n_head * hd,
                       d_mlp=n_head * hd * pick([2, 4]), vocab=pick([20, 57, 120]), n_ctx=T,
                       rotary=pick([False, True]), tied=pick([False, True]))
        out.append((cfg, pick([3, 4, 6]), pick([1, 2, 3]), int(torch.randint(0, 1000, (1,),
                                                                            generator=g))))
    return out


@pytest.mark.parametrize("case", _random_lm_configs(6, 2032))
def test_random_lm_configs_engine_matches_per_sample_gradients(gpu, case):
    """Seeded random causal-LM configurations (layers, heads, widths, vocabulary, T, rotary or
    learned positions, tied or untied head, 1-3 val rows) through the engine in fp32 against
    float64 per-sample gradients: every parameter's dot (presum layers at n_v = 1, where
    presum equals the pairwise sum) and every train gradient."""
    cfg, n_t, n_v, seed = case
    torch.manual_seed(seed)
    T, vocab = cfg.n_ctx, cfg.vocab
    model = CausalLM(cfg)
    untied = copy.deepcopy(model)
    if cfg.tied:
        untied.lm_head.weight = nn.Parameter(model.wte.weight.detach().clone())
    ref = copy.deepcopy(model).double()
    untied = untied.double()
    X, Y = synthetic_tokens(n_t + n_v, T, vocab, seed=seed + 1)
    model = model.to(gpu)
    print(f"random lm engine cfg={cfg} n_t={n_t} n_v={n_v}", flush=True)
    eng = GradDotProdEngine(model, val_batch_size=n_v, use_dummy_bias=True, precision="fp32")
    eng.attach(torch.optim.SGD(model.parameters(), lr=0.0))
    eng.attach_train_batch(X[:n_t], Y[:n_t], 0, 0)
    model(X.to(gpu), Y.to(gpu)).backward()
    torch.cuda.synchronize()
    dots = {n: p.grad_dot_prod.cpu() for n, p in model.named_parameters()
            if hasattr(p, "grad_dot_prod")}
    semantics = {n: m.use_ghost_computation for n, m in model.named_modules()
                 if hasattr(m, "use_ghost_computation")}
    eng.prepare_gradients()
    grads = {n: p.grad.cpu() for n, p in model.named_parameters()
             if p.grad is not None and "dummy_bias" not in n}
    eng.detach()
    N = n_t + n_v
    g_dot = brute.per_sample_grads(untied, X, Y, _lm_loss(T), 1.0 / (N * T))
    g_grad = brute.per_sample_grads(ref, X, Y, _lm_loss(T), 1.0 / (N * T))
    checked = 0
    for name, d in dots.items():
        layer = name.rsplit(".", 1)[0]
        if not semantics.get(layer, True) and n_v > 1:
            continue   # presum: not a function of the per-sample gradients
        assert_close(d, brute.pairwise_dots(g_dot[name], n_v), FP32_TOL, f"dot {name}")
        checked += 1
    assert checked > 0
    assert grads
    for name, gr in grads.items():
        assert_close(gr, brute.train_mean(g_grad[name], n_v, N), FP32_TOL, f"grad {name}")


def test_mlp_engine_on_gpu_ten_steps(gpu):
    """configs[0] in small: 10 SGD steps, per-step aggregated dots vs brute force."""
    torch.manual_seed(14)
    dims = (64, 48, 32, 10)
    model = MLP(dims).to(gpu)
    ref = copy.deepcopy(model).cpu().double()
    n_t, n_v = 24, 8
    X = torch.randn(n_t + n_v, dims[0], generator=gen(15))
    Y = torch.randint(0, 10, (n_t + n_v,), generator=gen(16))
    opt = torch.optim.SGD(model.parameters(), lr=0.1)
    eng = GradDotProdEngine(model, val_batch_size=n_v, use_dummy_bias=False, precision="fp32")
    eng.attach(opt)
    for step in range(10):
        print(f"mlp step {step}", flush=True)
        eng.attach_train_batch(X[:n_t], Y[:n_t], step, 0)
        loss = F.cross_entropy(model(X.to(gpu)), Y.to(gpu))
        opt.zero_grad(set_to_none=True)
        loss.backward()
        eng.aggregate_and_log()
        eng.prepare_gradients()
        opt.step()
        eng.clear_gradients()
        g = brute.per_sample_grads(
            ref, X.double(), Y, lambda m, x, y: F.cross_entropy(m(x), y, reduction="sum"),
            1.0 / X.shape[0])
        want = sum(brute.pairwise_dots(gr, n_v) for gr in g.values())
        assert_close(eng.dot_product_log[-1]["dot_product"], want, FP32_TOL, f"step {step}")
        with torch.no_grad():
            for name, p in ref.named_parameters():
                p -= 0.1 * brute.train_mean(g[name], n_v, X.shape[0])
    eng.detach()
    for (n1, p1), (n2, p2) in zip(model.named_parameters(), ref.named_parameters()):
        assert_close(p1.detach().cpu(), p2.detach(), 1e-4, f"weights {n1}")


def test_hf_conv1d_layers_use_presum(gpu):
    transformers = pytest.importorskip("transformers")
    Conv1D = transformers.pytorch_utils.Conv1D
    torch.manual_seed(17)

    class Net(nn.Module):
        def __init__(self):
            super().__init__()
            self.c1 = Conv1D(24, 16)   # nf=24 out, nx=16 in
            self.c2 = Conv1D(8, 24)

        def forward(self, x):
            return self.c2(torch.tanh(self.c1(x)))

    net = Net()
    ref = copy.deepcopy(net).double()
    N, n_v, T = 6, 1, 5
    X = torch.randn(N, T, 16, generator=gen(18))
    head = torch.randn(8, generator=gen(19))
    net = net.to(gpu)
    eng = GradDotProdEngine(net, val_batch_size=n_v, use_dummy_bias=False, precision="fp32")
    eng.attach(torch.optim.SGD(net.parameters(), lr=0.0))
    ((net(X.to(gpu)) * head.to(gpu)).reshape(N, -1).sum(1).mean()).backward()
    torch.cuda.synchronize()
    dots = {n: p.grad_dot_prod.cpu() for n, p in net.named_parameters()}
    eng.detach()
    g = brute.per_sample_grads(ref, X.double(), X, lambda m, x, y: (m(x) * head.double()).sum(),
                               1.0 / N)
    for name, d in dots.items():   # n_val = 1: presum equals <g_i, g_val>
        assert_close(d, brute.pairwise_dots(g[name], n_v), FP32_TOL, f"conv1d {name}")


@pytest.mark.parametrize("n_v", [1, 2])
def test_hf_conv1d_bf16_fused_path(gpu, n_v, monkeypatch):
    """A bf16 HF Conv1D model at tile-aligned sizes takes the fused dot + train-gradient pass
    (operands swapped, [d_in, d_out] gradient popped into train_grad): dots and weights'
    gradients against the unfused passes on the same run, and at n_v = 1 (presum equals
    pairwise) the dots against brute force."""
    transformers = pytest.importorskip("transformers")
    Conv1D = transformers.pytorch_utils.Conv1D
    torch.manual_seed(31)

    class Net(nn.Module):
        def __init__(self):
            super().__init__()
            self.c1 = Conv1D(128, 64)   # nf=128 out, nx=64 in
            self.c2 = Conv1D(64, 128)

        def forward(self, x):
            return self.c2(torch.tanh(self.c1(x)))

    net = Net().to(torch.bfloat16).float()   # the reference starts from the bf16 weights
    ref = copy.deepcopy(net).double()
    N, T = 3 + n_v, 64
    X = torch.randn(N, T, 64, generator=gen(32)).to(torch.bfloat16).float()
    head = torch.randn(64, generator=gen(33)).to(torch.bfloat16).float()
    net = net.to(gpu, torch.bfloat16)
    opt = torch.optim.SGD(net.parameters(), lr=0.0)
    eng = GradDotProdEngine(net, val_batch_size=n_v, use_dummy_bias=False, record_algorithms=True)

    def run():
        S.ALGO_LOG.clear()
        eng.attach(opt)
        loss = (net(X.to(gpu, torch.bfloat16)) * head.to(gpu, torch.bfloat16))
        loss.reshape(N, -1).float().sum(1).mean().backward()
        torch.cuda.synchronize()
        dots = {n: p.grad_dot_prod.float().cpu() for n, p in net.named_parameters()}
        eng.prepare_gradients()
        grads = {n: p.grad.float().cpu() for n, p in net.named_parameters()}
        eng.clear_gradients()
        eng.detach()
        return dots, grads, dict(S.ALGO_LOG)

    print(f"hf conv1d bf16 fused n_v={n_v}", flush=True)
    dots, grads, log = run()
    assert sorted(k for k, v in log.items() if v[1] == "valgrad+train_grad") == ["c1", "c2"], log
    assert grads["c1.weight"].shape == (64, 128) and grads["c2.weight"].shape == (128, 64)
    monkeypatch.setattr(S, "_fused_dot_train_grad", lambda *a, **k: False)
    dots2, grads2, log2 = run()
    assert not any(v[1] == "valgrad+train_grad" for v in log2.values()), log2
    for name in dots:
        assert_close(dots[name], dots2[name], 1e-2, f"fused vs unfused dot {name}")
        assert_close(grads[name], grads2[name], 1e-2, f"fused vs unfused grad {name}")
    if n_v == 1:
        g = brute.per_sample_grads(ref, X.double(), X,
                                   lambda m, x, y: (m(x) * head.double()).sum(), 1.0 / N)
        for name, d in dots.items():
            assert_close(d, brute.pairwise_dots(g[name], n_v), BF16_TOL, f"conv1d {name}")
            want = brute.train_mean(g[name], n_v, N)
            assert_close(grads[name], want, BF16_TOL, f"conv1d grad {name}")


@pytest.mark.parametrize("dummy", [False, True])
def test_hf_gpt2_model_through_the_engine(gpu, dummy):
    """The reference LM example's model family: a tiny Hugging Face GPT2LMHeadModel (Conv1D
    attention and MLP layers, LayerNorms, wte / wpe, tied lm_head), per-sample position ids
    passed explicitly, fp32, one val row (presum equals the pairwise sum), against float64
    per-sample gradients: every parameter's dot and train gradient; with `dummy` through the
    documented dummy-bias setup (embeddings listed in ghost_embeddings, weights frozen for
    autograd)."""
    transformers = pytest.importorskip("transformers")
    torch.manual_seed(41)
    cfg = transformers.GPT2Config(n_layer=2, n_embd=32, n_head=2, vocab_size=50, n_positions=16,
                                  resid_pdrop=0.0, embd_pdrop=0.0, attn_pdrop=0.0,
                                  bos_token_id=0, eos_token_id=0)
    model = transformers.GPT2LMHeadModel(cfg).eval()
    untied = copy.deepcopy(model)
    untied.lm_head.weight = nn.Parameter(model.transformer.wte.weight.detach().clone())
    untied = untied.double()
    ref = copy.deepcopy(model).double()
    N, n_v, T = 5, 1, 12
    X = torch.randint(0, 50, (N, T), generator=gen(42))
    pos = torch.arange(T).expand(N, T).contiguous()

    def sample_loss(m, x, y):   # the batch loss is the mean of the per-sample token means
        return m(input_ids=x, position_ids=torch.arange(T)[None], labels=x).loss

    model = model.to(gpu)
    opt = torch.optim.SGD(model.parameters(), lr=0.0)
    if dummy:
        model.ghost_embeddings = ["transformer.wte", "transformer.wpe"]
    eng = GradDotProdEngine(model, val_batch_size=n_v, use_dummy_bias=dummy, precision="fp32")
    eng.attach(opt)
    print(f"hf gpt2 engine dummy={dummy}", flush=True)
    model(input_ids=X.to(gpu), position_ids=pos.to(gpu), labels=X.to(gpu)).loss.backward()
    torch.cuda.synchronize()
    dots = {n: p.grad_dot_prod.cpu() for n, p in model.named_parameters()
            if hasattr(p, "grad_dot_prod")}
    eng.prepare_gradients()
    grads = {n: p.grad.cpu() for n, p in model.named_parameters()
             if p.grad is not None and "dummy_bias" not in n}
    eng.detach()
    assert len(grads) == len(list(ref.named_parameters()))
    g_dot = brute.per_sample_grads(untied, X, X, sample_loss, 1.0 / N)
    g_grad = brute.per_sample_grads(ref, X, X, sample_loss, 1.0 / N)
    assert any(".attn.c_attn." in n for n in dots) and "transformer.wpe.weight" in dots
    for name, d in dots.items():
        assert_close(d, brute.pairwise_dots(g_dot[name], n_v), FP32_TOL, f"dot {name}")
    for name, gr in grads.items():
        assert_close(gr, brute.train_mean(g_grad[name], n_v, N), FP32_TOL, f"grad {name}")


def test_hf_gpt2_bf16_conv1d_layers_take_the_fused_pass(gpu, monkeypatch):
    """A bf16 Hugging Face GPT2LMHeadModel at tile-aligned sizes: its four Conv1D layers take
    the fused dot + train-gradient pass (gs_conv1d_dot_train_grad, bias included), and the
    dots and gradients equal those of the separate passes on the same run."""
    transformers = pytest.importorskip("transformers")
    torch.manual_seed(43)
    cfg = transformers.GPT2Config(n_layer=1, n_embd=64, n_head=2, vocab_size=50, n_positions=64,
                                  resid_pdrop=0.0, embd_pdrop=0.0, attn_pdrop=0.0,
                                  bos_token_id=0, eos_token_id=0)
    model = transformers.GPT2LMHeadModel(cfg).eval().to(gpu, torch.bfloat16)
    N, n_v, T = 6, 2, 64
    X = torch.randint(0, 50, (N, T), generator=gen(44)).to(gpu)
    pos = torch.arange(T, device=gpu).expand(N, T).contiguous()
    eng = GradDotProdEngine(model, val_batch_size=n_v, use_dummy_bias=False, record_algorithms=True)
    opt = torch.optim.SGD(model.parameters(), lr=0.0)

    def run():
        S.ALGO_LOG.clear()
        eng.attach(opt)
        model(input_ids=X, position_ids=pos, labels=X).loss.backward()
        torch.cuda.synchronize()
        dots = {n: p.grad_dot_prod.float().cpu() for n, p in model.named_parameters()
                if hasattr(p, "grad_dot_prod")}
        eng.prepare_gradients()
        grads = {n: p.grad.float().cpu() for n, p in model.named_parameters()
                 if p.grad is not None}
        eng.clear_gradients()
        eng.detach()
        return dots, grads, dict(S.ALGO_LOG)

    print("hf gpt2 bf16 fused", flush=True)
    dots, grads, log = run()
    fused = sorted(k for k, v in log.items() if v[1] == "valgrad+train_grad")
    assert fused == ["transformer.h.0.attn.c_attn", "transformer.h.0.attn.c_proj",
                     "transformer.h.0.mlp.c_fc", "transformer.h.0.mlp.c_proj"], log
    monkeypatch.setattr(S, "_fused_dot_train_grad", lambda *a, **k: False)
    dots2, grads2, _ = run()
    for name in dots:
        assert_close(dots[name], dots2[name], 1e-2, f"fused vs separate dot {name}")
    for name in grads:
        assert_close(grads[name], grads2[name], 1e-2, f"fused vs separate grad {name}")


def test_gradproj_engine_on_gpu_naive_check(gpu, tmp_path):
    torch.manual_seed(20)
    model = nn.Sequential(nn.Linear(10, 20), nn.ReLU(), nn.Linear(20, 5)).to(gpu)
    X = torch.randn(4, 10, generator=gen(21)).to(gpu)
    Y = torch.randint(0, 5, (4,), generator=gen(22)).to(gpu)
    eng = GradProjLoraEngine(model, proj_layers="0,2", proj_rank_total=16, proj_rank_min=2,
                             proj_seed=42, proj_dtype="float32", proj_dir=str(tmp_path))
    eng.attach()
    F.cross_entropy(model(X), Y).backward()
    proj = eng.collect_batch().cpu()
    eng.detach()
    naive = []
    for b in range(4):
        model.zero_grad()
        F.cross_entropy(model(X[b:b + 1]), Y[b:b + 1]).backward()
        parts = []
        for name in sorted(eng.matched_layers):
            P_i, P_o = eng.projection_matrices[name]
            W = eng.matched_layers[name].weight.grad.double()
            parts.append((P_o.double() @ W @ P_i.double().t()).reshape(-1))
        naive.append(torch.cat(parts).cpu())
    assert_close(proj, torch.stack(naive), FP32_TOL, "gradproj naive")


def test_gradproj_embedding_on_gpu_matches_naive(gpu, tmp_path):
    torch.manual_seed(23)
    emb = nn.Embedding(40, 12)
    model = nn.Sequential(emb, nn.Flatten(), nn.Linear(12 * 5, 3)).to(gpu)
    X = torch.randint(0, 40, (4, 5), generator=gen(24)).to(gpu)
    Y = torch.randint(0, 3, (4,), generator=gen(25)).to(gpu)
    eng = GradProjLoraEngine(model, proj_layers="0", proj_rank_total=12, proj_rank_min=2,
                             proj_seed=6, proj_dtype="float32", proj_dir=str(tmp_path),
                             include_embeddings=True)
    eng.attach()
    F.cross_entropy(model(X), Y).backward()
    got = eng.matched_layers["0"]._ghost_grad_proj.cpu()
    eng.detach()
    P_i, P_o = (p.double().cpu() for p in eng.projection_matrices["0"])
    for b in range(4):
        model.zero_grad()
        F.cross_entropy(model(X[b:b + 1]), Y[b:b + 1], reduction="sum").backward()
        W = emb.weight.grad.double().cpu()
        # the reference applies no batch-size factor to embedding projections
        assert_close(got[b].double() * 4, P_o @ W.t() @ P_i.t(), FP32_TOL, f"emb proj {b}")


def test_side_stream_overlap_gives_identical_results(gpu):
    """The dot kernels on the side stream (default) and on the autograd stream give the same
    bits over several optimizer steps of a model large enough to recycle memory (no
    attention, whose backward need not be bit-reproducible)."""
    vocab, d, T = 512, 128, 128

    class Net(nn.Module):
        def __init__(self):
            super().__init__()
            self.emb = nn.Embedding(vocab, d)
            self.blocks = nn.ModuleList(
                nn.Sequential(nn.LayerNorm(d), nn.Linear(d, 4 * d), nn.GELU(), nn.Linear(4 * d, d))
                for _ in range(3))
            self.ln_f = nn.LayerNorm(d)
            self.head = nn.Linear(d, vocab)

        def forward(self, x, y):
            h = self.emb(x)
            for b in self.blocks:
                h = h + b(h)
            logits = self.head(self.ln_f(h)).float()
            return F.cross_entropy(logits.reshape(-1, vocab), y.reshape(-1))

    X = torch.randint(0, vocab, (10, T), generator=gen(31))
    Y = torch.randint(0, vocab, (10, T), generator=gen(32))

    def run(overlap):
        torch.manual_seed(30)
        model = Net().to(gpu).bfloat16()
        opt = torch.optim.SGD(model.parameters(), lr=1e-2)
        eng = GradDotProdEngine(model, val_batch_size=2, use_dummy_bias=False,
                                precision="reference", overlap=overlap)
        eng.attach(opt)
        for step in range(3):
            eng.attach_train_batch(X[:8], Y[:8], step, 0)
            model(X.to(gpu), Y.to(gpu)).backward()
            eng.prepare_gradients()
            opt.step()
            eng.aggregate_and_log()
            eng.clear_gradients()
        eng.detach()
        dots = torch.stack([r["dot_product"] for r in eng.dot_product_log])
        return dots, [p.detach().float().cpu() for p in model.parameters()]

    d_on, w_on = run(True)
    d_off, w_off = run(False)
    print(f"overlap dots {d_on[-1, :3].tolist()}", flush=True)
    assert torch.isfinite(d_on).all()
    assert torch.equal(d_on, d_off)
    for a, b in zip(w_on, w_off):
        assert torch.equal(a, b)


def test_async_host_copies_and_files_match_device_results(gpu, tmp_path):
    """The dot log's host copies and the projection files are written off the critical
    path; what a reader sees equals the device results, and the saved files are the
    reference's plain formats (loadable with weights_only=True)."""
    torch.manual_seed(40)
    model = MLP((32, 64, 10)).to(gpu)
    X = torch.randn(12, 32, generator=gen(41)).to(gpu)
    Y = torch.randint(0, 10, (12,), generator=gen(42)).to(gpu)
    eng = GradDotProdEngine(model, val_batch_size=4, precision="fp32",
                            dot_prod_save_path=str(tmp_path))
    eng.attach(torch.optim.SGD(model.parameters(), lr=0.0))
    device_totals = []
    for step in range(3):
        eng.attach_train_batch(X[:8], Y[:8], step, step)
        F.cross_entropy(model(X), Y).backward()
        dots = [p.grad_dot_prod.clone() for _, p in model.named_parameters()
                if hasattr(p, "grad_dot_prod")]
        device_totals.append(sum(dots).cpu())
        eng.prepare_gradients()
        eng.aggregate_and_log()
        eng.clear_gradients()
    assert len(eng.dot_product_log) == 3
    for rec, want in zip(eng.dot_product_log, device_totals):
        assert rec["dot_product"].device.type == "cpu"
        assert_close(rec["dot_product"], want, 1e-6, "async log")
        assert torch.equal(rec["X_train"], X[:8].cpu())
    eng.save_dot_product_log(iter_num=7)
    saved = torch.load(tmp_path / "dot_prod_log_iter_7.pt", weights_only=True)
    assert type(saved) is list and len(saved) == 3
    assert set(saved[0]) == {"dot_product", "X_train", "Y_train", "iter_num", "batch_idx"}
    assert saved[2]["iter_num"] == 2 and saved[2]["dot_product"].dtype == torch.float32
    # clear() drops records whose copies may still be in flight, without waiting; the
    # records logged afterwards read back finished values.
    for step in range(3, 6):
        eng.attach_train_batch(X[:8], Y[:8], step, step)
        F.cross_entropy(model(X), Y).backward()
        want = sum(p.grad_dot_prod.clone() for _, p in model.named_parameters()
                   if hasattr(p, "grad_dot_prod")).cpu()
        eng.prepare_gradients()
        eng.aggregate_and_log()
        eng.clear_gradients()
        if step < 5:
            eng.dot_product_log.clear()
    assert len(eng.dot_product_log) == 1
    assert_close(eng.dot_product_log[0]["dot_product"], want, 1e-6, "log after clear")
    eng.detach()

    proj_dir = tmp_path / "proj"
    net = nn.Sequential(nn.Linear(16, 24), nn.ReLU(), nn.Linear(24, 8)).to(gpu)
    Xp = torch.randn(6, 16, generator=gen(43)).to(gpu)
    peng = GradProjLoraEngine(net, proj_layers="0,2", proj_rank_total=16, proj_rank_min=2,
                              proj_seed=3, proj_dtype="float16", proj_dir=str(proj_dir))
    peng.attach()
    outs = []
    for it in range(2):
        net.zero_grad()
        net(Xp).square().mean().backward()
        outs.append(peng.collect_batch(batch_indices=list(range(6))).cpu())
    peng.detach()   # waits for the writer
    for it, want in enumerate(outs):
        d = torch.load(proj_dir / f"proj_iter_{it:06d}.pt", weights_only=True)
        assert set(d) == {"proj", "iter", "batch_size", "batch_idx"}
        assert d["proj"].dtype == torch.float16 and d["iter"] == it and d["batch_size"] == 6
        assert torch.equal(d["proj"], want)
    assert (proj_dir / "metadata.json").exists()


@pytest.mark.parametrize("precision,tol", [("fp32", FP32_TOL), ("reference", BF16_TOL)])
@pytest.mark.parametrize("n_val", [1, 3])
def test_conv2d_engine_on_gpu(gpu, precision, tol, n_val):
    """Conv2d samplers: unfold to token-major rows, presum dots on the Linear kernels, the
    bias dot and train gradient from the bias kernel."""
    from oracle import ghost_ref as R
    from tests.helpers import conv_net, run_conv_engine
    torch.manual_seed(60)
    model = conv_net()
    ref = copy.deepcopy(model).double()
    N = 7
    X = torch.randn(N, 3, 8, 8, generator=gen(61))
    Y = torch.randint(0, 5, (N,), generator=gen(62))
    model = model.to(gpu)
    caps = {}
    for idx in (0, 2):
        model[idx].register_forward_hook(
            lambda m, i, o, k=idx: caps.__setitem__(("A", k), i[0].detach().cpu()))
        model[idx].register_full_backward_hook(
            lambda m, gi, go, k=idx: caps.__setitem__(("B", k), go[0].detach().cpu()))
    print(f"conv2d engine precision={precision} n_val={n_val}", flush=True)
    dots, grads = run_conv_engine(model, X, Y, n_val, gpu, precision)
    g = brute.per_sample_grads(ref, X.double(), Y,
                               lambda m, x, y: F.cross_entropy(m(x), y, reduction="sum"),
                               1.0 / N)
    for idx in (0, 2):
        layer = model[idx]
        conv = dict(kernel_size=layer.kernel_size, dilation=layer.dilation,
                    padding=layer.padding, stride=layer.stride)
        want = R.conv2d_dot_exact(caps[("A", idx)], caps[("B", idx)], n_val, conv)
        assert_close(dots[f"{idx}.weight"], want, tol, f"conv{idx} dot")
        if n_val == 1:
            # A, B captured from the fp32 GPU model: fp32-level agreement
            assert_close(want, brute.pairwise_dots(g[f"{idx}.weight"], 1), 1e-5, "closed form")
    for name, gr in grads.items():
        assert_close(gr, brute.train_mean(g[name], n_val, N), tol, f"grad {name}")


@pytest.mark.parametrize("precision", ["fp32", "reference"])
@pytest.mark.parametrize("n_val", [1, 2])
def test_conv2d_reference_ghost_on_gpu(gpu, precision, n_val):
    """reference_conv2d_ghost through the HIP ghost kernel: the Conv2d layer on the ghost
    branch (C_in*kh*kw == C_out) against the reference's bf16 op sequence
    (oracle.conv2d_ghost_ref, precision 'reference') or the quantity in float64 (fp32); the
    layer on the materialised branch keeps the presum dot."""
    from oracle import ghost_ref as R
    from tests.helpers import conv_net_square, run_conv_engine
    torch.manual_seed(63)
    model = conv_net_square().to(gpu)
    N = 6
    X = torch.randn(N, 4, 8, 8, generator=gen(64))
    Y = torch.randint(0, 5, (N,), generator=gen(65))
    caps = {}
    for idx in (0, 2):
        model[idx].register_forward_hook(
            lambda m, i, o, k=idx: caps.__setitem__(("A", k), i[0].detach().cpu()))
        model[idx].register_full_backward_hook(
            lambda m, gi, go, k=idx: caps.__setitem__(("B", k), go[0].detach().cpu()))
    print(f"conv2d reference ghost precision={precision} n_val={n_val}", flush=True)
    dots, _ = run_conv_engine(model, X, Y, n_val, gpu, precision, reference_conv2d_ghost=True)
    assert model[0].use_ghost_computation and not model[2].use_ghost_computation
    convs = {idx: dict(kernel_size=model[idx].kernel_size, dilation=model[idx].dilation,
                       padding=model[idx].padding, stride=model[idx].stride) for idx in (0, 2)}
    A0, B0 = caps[("A", 0)], caps[("B", 0)]
    exact = R.conv2d_ghost_exact(A0, B0, n_val, convs[0])
    if precision == "fp32":
        assert_close(dots["0.weight"], exact, FP32_TOL, "ghost branch")
        tol = FP32_TOL
    else:
        assert dots["0.weight"].dtype == torch.float32
        assert_close(dots["0.weight"], R.conv2d_ghost_ref(A0, B0, n_val, convs[0]).double(),
                     BF16_TOL, "ghost branch vs the reference's op sequence")
        assert_close(dots["0.weight"], exact, BF16_TOL, "ghost branch vs float64")
        tol = BF16_TOL
    assert_close(dots["2.weight"], R.conv2d_dot_exact(caps[("A", 2)], caps[("B", 2)], n_val,
                                                      convs[2]), tol, "materialised branch")


@pytest.mark.parametrize("n_v", [1, 2])
def test_gpt2_engine_fused_bias_path_on_gpu(gpu, n_v, monkeypatch):
    """Tile-aligned shapes (T and every d_out multiples of 256) route each Linear with a bias
    through the fused weight + bias pass: dots against brute force, and dots and train grads
    against the separate weight and bias passes on the same bf16 run."""
    torch.manual_seed(21)
    T, vocab = 256, 64
    cfg = LMConfig(n_layer=1, n_head=4, d_model=256, d_mlp=512, vocab=vocab, n_ctx=T)
    model = CausalLM(cfg).to(torch.bfloat16).float()   # references start from the bf16 weights
    untied = copy.deepcopy(model)
    untied.lm_head.weight = nn.Parameter(model.wte.weight.detach().clone())
    untied = untied.double()
    n_t = 3
    X, Y = synthetic_tokens(n_t + n_v, T, vocab, seed=22)
    model = model.to(gpu, torch.bfloat16)

    opt = torch.optim.SGD(model.parameters(), lr=0.0)
    # the kernels' own fp32 dots for the arithmetic checks; the reference-dtype hand-over is
    # checked against them below
    eng = GradDotProdEngine(model, val_batch_size=n_v, use_dummy_bias=True,
                            record_algorithms=True, linear_algo="valgrad", dot_dtypes="fp32")

    def run():
        S.ALGO_LOG.clear()
        eng.attach(opt)
        eng.attach_train_batch(X[:n_t], Y[:n_t], 0, 0)
        model(X.to(gpu), Y.to(gpu)).backward()
        torch.cuda.synchronize()
        dots = {n: p.grad_dot_prod.cpu() for n, p in model.named_parameters()
                if hasattr(p, "grad_dot_prod")}
        eng.prepare_gradients()
        grads = {n: p.grad.float().cpu() for n, p in model.named_parameters()
                 if p.grad is not None and "dummy_bias" not in n}
        eng.aggregate_and_log()
        eng.clear_gradients()
        eng.detach()
        return dots, grads, dict(S.ALGO_LOG)

    print(f"gpt2 fused-bias engine n_v={n_v}", flush=True)
    linears = ["h.0.fc", "h.0.fc_out", "h.0.proj", "h.0.qkv"]
    # default: weight + bias dots and both train grads from one pass over the train rows
    dots, grads, log = run()
    assert sorted(k for k, v in log.items() if v[1] == "valgrad+train_grad") == linears, log
    # the default hand-over: each dot in the dtype the reference returns (a Linear's
    # materialised-branch weight dot and its bias dot in bf16, the rest fp32), the fp32 value
    # rounded once
    eng.options["dot_dtypes"] = "reference"
    dots_ref, _, _ = run()
    eng.options["dot_dtypes"] = "fp32"
    modules = dict(model.named_modules())
    for name, d in dots.items():
        mod = modules[name.rsplit(".", 1)[0]]
        bf = isinstance(mod, nn.Linear) and (name.endswith("bias") or
                                             not mod.use_ghost_computation)
        assert d.dtype == torch.float32, name
        assert dots_ref[name].dtype == (torch.bfloat16 if bf else torch.float32), name
        assert torch.equal(dots_ref[name], d.to(dots_ref[name].dtype)), name
    # without it: the fused weight + bias dot pass, train grad separately
    monkeypatch.setattr(S, "_fused_dot_train_grad", lambda *a, **k: False)
    dots1, grads1, log1 = run()
    assert sorted(k for k, v in log1.items() if v[1] == "valgrad+bias") == linears, log1
    # without both: separate weight and bias passes
    monkeypatch.setattr(S, "_fused_bias_dot", lambda *a, **k: False)
    dots2, grads2, log2 = run()
    assert not any(v[1] in ("valgrad+bias", "valgrad+train_grad") for v in log2.values()), log2
    for name, d in dots1.items():
        assert_close(d, dots2[name], 1e-2, f"fused bias vs separate dot {name}")
    for name in grads1:
        assert_close(grads1[name], grads2[name], 1e-2, f"fused bias vs separate grad {name}")
    semantics = {n: m.use_ghost_computation for n, m in model.named_modules()
                 if hasattr(m, "use_ghost_computation")}
    N = n_t + n_v
    g_untied = brute.per_sample_grads(untied, X, Y, _lm_loss(T), 1.0 / (N * T))
    for name, d in dots.items():
        assert_close(d, dots2[name], 1e-2, f"fused vs separate dot {name}")
        layer = name.rsplit(".", 1)[0]
        if not semantics.get(layer, True) and n_v > 1:
            continue   # presum: not a function of the per-sample gradients
        assert_close(d, brute.pairwise_dots(g_untied[name], n_v), BF16_TOL, f"dot {name}")
    block = [n for n in grads if n.startswith("h.")]
    assert block and all(n in grads2 for n in block), (sorted(grads), sorted(grads2))
    for name in block:
        assert_close(grads[name], grads2[name], 1e-2, f"fused vs separate grad {name}")


def test_manager_step_contract_on_gpu(gpu, tmp_path):
    """The reference's training step (Examples/GradDotProd_LM/training_loop.py:99-166) through
    GhostEngineManager on the GPU: attach_train_batch -> save metrics on their interval ->
    prepare_forward_input -> forward/backward -> prepare_gradients -> optimizer step ->
    aggregate_and_log -> clear_gradients -> zero_grad, with config.ghost_options reaching
    the engine (fp32 dots here).  Over four steps: every logged dot vector and the weights
    against per-sample gradients of float64 copies; then the files the loop leaves
    (valset.pt, dot_prod_log_iter_2.pt, and dot_prod_log_iter_-1.pt from cleanup)."""
    import types
    from ghostsuite_amd import GhostEngineManager
    torch.manual_seed(50)
    T, vocab, n_t, n_v, lr = 16, 64, 4, 2, 0.05
    cfg_m = LMConfig(n_layer=2, n_head=2, d_model=32, d_mlp=64, vocab=vocab, n_ctx=T)
    model = CausalLM(cfg_m)
    ref = copy.deepcopy(model).double()       # tied, follows the same SGD updates
    model = model.to(gpu)
    Xv, Yv = synthetic_tokens(n_v, T, vocab, seed=51)
    opt = torch.optim.SGD(model.parameters(), lr=lr)
    cfg = types.SimpleNamespace(method="GradDotProd", result_dir=str(tmp_path),
                                val_batch_size=n_v, dot_prod_save_interval=2,
                                ghost_options={"precision": "fp32"})
    mgr = GhostEngineManager(cfg, model, opt, {"master_process": True, "device": gpu},
                             (Xv.to(gpu), Yv.to(gpu)))
    assert S.options["precision"] == "fp32"
    N = n_t + n_v
    for it in range(4):
        print(f"manager step {it}", flush=True)
        X, Y = synthetic_tokens(n_t, T, vocab, seed=60 + it)
        mgr.attach_train_batch(X.to(gpu), Y.to(gpu), it, list(range(it * n_t, (it + 1) * n_t)))
        if it > 0 and mgr.should_save_metrics(it):
            mgr.save_metrics(it)
        Xf, Yf = mgr.prepare_forward_input(X.to(gpu), Y.to(gpu))
        assert torch.equal(Xf[n_t:].cpu(), Xv)
        model(Xf, Yf).backward()
        mgr.prepare_gradients()
        opt.step()
        mgr.aggregate_and_log()
        mgr.clear_gradients()
        opt.zero_grad(set_to_none=True)
        # expected: per-sample gradients on the same concatenated batch
        Xc, Yc = torch.cat((X, Xv)), torch.cat((Y, Yv))
        untied = copy.deepcopy(ref)
        untied.lm_head.weight = nn.Parameter(ref.wte.weight.detach().clone())
        g_untied = brute.per_sample_grads(untied, Xc, Yc, _lm_loss(T), 1.0 / (N * T))
        g_tied = brute.per_sample_grads(ref, Xc, Yc, _lm_loss(T), 1.0 / (N * T))
        names = [n for n, _ in ref.named_parameters()]
        want = sum(brute.pairwise_dots(g_untied[n], n_v) for n in names)
        assert_close(mgr.engine.dot_product_log[-1]["dot_product"], want, FP32_TOL,
                     f"step {it} logged dots")
        with torch.no_grad():
            for n, p in ref.named_parameters():
                p -= lr * brute.train_mean(g_tied[n], n_v, N)
        ref_params = dict(ref.named_parameters())
        for n, p in model.named_parameters():
            if "dummy_bias" not in n:
                assert_close(p.detach().cpu(), ref_params[n].detach(), FP32_TOL,
                             f"step {it} weight {n}")
    mgr.cleanup()
    d = tmp_path / "grad_dotprods"
    vs = torch.load(d / "valset.pt", weights_only=True)
    assert torch.equal(vs["X_val"], Xv) and torch.equal(vs["Y_val"], Yv)
    log2 = torch.load(d / "dot_prod_log_iter_2.pt", weights_only=True)
    assert [r["iter_num"] for r in log2] == [0, 1]
    assert log2[1]["batch_idx"] == [4, 5, 6, 7] and log2[0]["dot_product"].shape == (n_t,)
    rest = torch.load(d / "dot_prod_log_iter_-1.pt", weights_only=True)
    assert [r["iter_num"] for r in rest] == [2, 3]
    assert not hasattr(model, "autograd_grad_sample_hooks")


@pytest.mark.parametrize("promote", [False, True])
def test_embedding_id_promotion_on_gpu(gpu, promote):
    """GPT-2-small wte [50257, 768] and wpe [1024, 768] tables, bf16, 16 train + 4 val rows of
    T = 1024, through the engine and the HIP embedding kernels.  reference_id_promotion=True
    runs the dots on the ids the reference's hook makes (int64 -> bf16 -> int64,
    autograd_grad_sample_dotprod.py:116-123): wte against the reference's own op sequence on
    those ids; wpe's position 1023 rounds to 1024, past the 1024-row table (where the
    reference's index_add_ would raise), and such a token takes no part, as any out-of-range
    id.  The train gradients use the ids as given in both settings."""
    from oracle import ghost_ref as R
    N, n_val, T, d, V = 20, 4, 1024, 768, 50257
    n_t = N - n_val

    class Embeddings(nn.Module):
        def __init__(self):
            super().__init__()
            self.wte = nn.Embedding(V, d)
            self.wpe = nn.Embedding(T, d)

        def forward(self, ids):
            pos = torch.arange(T, device=ids.device).repeat(ids.shape[0], 1)
            return self.wte(ids) + self.wpe(pos)

    torch.manual_seed(5)
    model = Embeddings().to(gpu, torch.bfloat16)
    ids = torch.randint(0, V, (N, T), generator=gen(501))
    ids[0, :4] = torch.tensor([1023, 50000, 50256, 257])   # ids that round in bf16
    head = (torch.randn(N, T, d, generator=gen(502)) * 1e-2).to(torch.bfloat16)
    eng = GradDotProdEngine(model, val_batch_size=n_val, use_dummy_bias=False,
                            reference_id_promotion=promote)
    eng.attach(torch.optim.SGD(model.parameters(), lr=0.0))
    print(f"embedding id promotion promote={promote}", flush=True)
    (model(ids.to(gpu)).float() * head.to(gpu).float()).sum().backward()
    torch.cuda.synchronize()
    got_te = model.wte.weight.grad_dot_prod.cpu()
    got_pe = model.wpe.weight.grad_dot_prod.cpu()
    grad_te = model.wte.weight.train_grad.float().cpu()
    grad_pe = model.wpe.weight.train_grad.float().cpu()
    eng.detach()
    B = head.float()
    pos = torch.arange(T).repeat(N, 1)
    if promote:
        p_ids = ids.to(torch.bfloat16).long()
        assert not torch.equal(p_ids, ids)
        assert_close(got_te, R.embedding_dot_ref(p_ids.to(torch.bfloat16), B, n_val, V),
                     BF16_TOL, "wte dot, reference sequence on promoted ids")
        p_pos = pos.to(torch.bfloat16).long()
        past = p_pos >= T
        assert past.any() and int(p_pos.max()) == T   # 1023 -> 1024
        Bz = B.clone()
        Bz[past] = 0
        assert_close(got_pe, R.embedding_dot_exact(p_pos.clamp(max=T - 1), Bz, n_val), BF16_TOL,
                     "wpe dot on promoted positions")
        assert not torch.allclose(got_te.double(), R.embedding_dot_exact(ids, B, n_val),
                                  rtol=1e-3)
    else:
        assert_close(got_te, R.embedding_dot_exact(ids, B, n_val), BF16_TOL, "wte dot")
        assert_close(got_pe, R.embedding_dot_exact(pos, B, n_val), BF16_TOL, "wpe dot")
    for tab, x, got in ((V, ids, grad_te), (T, pos, grad_pe)):
        want = torch.zeros(tab, d, dtype=torch.float64)
        want.index_add_(0, x[:n_t].reshape(-1), B[:n_t].double().reshape(-1, d) * N / n_t)
        assert_close(got.double(), want, BF16_TOL, f"train grad [{tab}]")


@pytest.mark.parametrize("first", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [16, 1000])
def test_ordered_sum_matches_sequential_in_place_adds(gpu, first, n):
    """gs_ordered_sum, the engine's aggregation of the per-parameter dots, against torch's
    in-place adds in the same order on the same GPU tensors (graddotprod_engine.py:204-211),
    bit for bit: 600 sources of scales 1e-3..1e3 (three chained launches of at most 256),
    bf16 and fp32 mixed, the total in the first source's dtype and in its memory."""
    from ghostsuite_amd import _native
    g = gen(600 + n)
    dts = [first] + [torch.bfloat16 if i % 3 else torch.float32 for i in range(599)]
    scales = 10.0 ** torch.randint(-3, 4, (600,), generator=g).double()
    srcs = [(torch.randn(n, generator=g) * float(sc)).to(dt) for dt, sc in zip(dts, scales)]
    print(f"ordered sum first={first} n={n}", flush=True)
    a = [s.to(gpu) for s in srcs]
    want = srcs[0].to(gpu)
    for s in srcs[1:]:
        want += s.to(gpu)
    got = _native.ops().ordered_sum_(a)
    torch.cuda.synchronize()
    assert got.data_ptr() == a[0].data_ptr() and got.dtype == first
    assert torch.equal(got, want)
    # a different order gives different bits: the order is the reference's, not any order
    rev = [s.to(gpu) for s in srcs[:1] + srcs[:0:-1]]
    assert not torch.equal(_native.ops().ordered_sum_(rev), want)



def test_side_stream_with_layers_on_both_sides_of_its_line(gpu):
    """One weight shared by a Linear call small enough for the autograd stream, one that runs on
    the side stream and an embedding: the same bits as without overlap, whichever comes first."""
    from ghostsuite_amd import autograd_grad_sample_dotprod as hooks
    d, T = 512, 256

    class Net(nn.Module):
        def __init__(self, small_first):
            super().__init__()
            self.small_first = small_first
            self.emb = nn.Embedding(d, d)
            self.big, self.small = nn.Linear(d, d), nn.Linear(d, d)
            self.big.weight = self.small.weight = self.emb.weight

        def forward(self, x):
            h = self.emb(x)
            if self.small_first:
                return self.big(h + self.small(h[:, :2]).mean(1, keepdim=True)).float()
            return self.small(torch.tanh(self.big(h))[:, :2]).float()

    x = torch.randint(0, d, (12, T), generator=gen(33)).to(gpu)
    big = torch.empty(12, T, d, device="meta")
    assert hooks._worth_overlapping(nn.Linear(1, 1), big, big)
    assert not hooks._worth_overlapping(nn.Linear(1, 1), big[:, :2], big[:, :2])
    for small_first in (False, True):
        res = []
        for overlap in (True, False):
            torch.manual_seed(34)
            model = Net(small_first).to(gpu).bfloat16()
            opt = torch.optim.SGD(model.parameters(), lr=1e-2)
            eng = GradDotProdEngine(model, val_batch_size=2, use_dummy_bias=False,
                                    precision="reference", overlap=overlap)
            eng.attach(opt)
            for step in range(3):
                eng.attach_train_batch(x[:10], x[:10], step, 0)
                model(x).square().mean().backward()
                eng.prepare_gradients()
                opt.step()
                eng.aggregate_and_log()
                eng.clear_gradients()
            eng.detach()
            res.append([r["dot_product"] for r in eng.dot_product_log] +
                       [p.detach().float().cpu() for p in model.parameters()])
        for a, b in zip(*res):
            assert torch.isfinite(a).all() and torch.equal(a, b)
