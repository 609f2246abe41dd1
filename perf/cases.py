"""The calls whose speed matters to a program that uses this package, with their inputs, their least work and the accuracy
they are held to.

Three kinds of program use it: one that serves a language model (`FlashSTU.generate`, or `FlashSTU.forward` with a prompt
and then token by token against the caches it returned), one that evaluates the model or the STU operator over whole
sequences (`FlashSTU.forward`, `STU.forward` in both modes, the dense LDS recurrence), and one that trains through the
operator (`STU.forward_differentiable` and its backward pass).  `listed()` has each of them at the sizes of the
repository's own configurations and some ragged ones, `draw()` anywhere in between."""
import functools
import math
import os
import sys
import tempfile

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "flash-stu-2_amd"))
from flash_stu import STU, FlashSTU, FlashSTUConfig, _hip  # noqa: E402
from flash_stu.utils.stu_utils import save_spectral_filters  # noqa: E402

VOCAB, FILTERS, STATE = 50257, 24, 64     # vocabulary, Hankel filters per STU, modes of the decode recurrence

# The language models: the repository's tiny, 768-d and 2048-d configurations (the last one with a third of its layers,
# so that a model is made in a few seconds: every layer pair costs the same).
MODELS = {
    "tiny": dict(n_embd=256, n_layers=4, n_heads=4, window_size=128, seq_len=1024, torch_dtype=torch.float32),
    "base": dict(n_embd=768, n_layers=12, n_heads=12, window_size=512, seq_len=2048, torch_dtype=torch.bfloat16),
    "large": dict(n_embd=2048, n_layers=8, n_heads=16, window_size=1024, seq_len=8192, torch_dtype=torch.bfloat16),
}
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def listed():
    return [
        # one request on the small fp32 model: a chain of the shortest launches there are
        dict(name="generate_tiny_fp32_1row", kind="generate", model="tiny", rows=1, prompt=64, new=64, top_k=0),
        # one interactive request, a short prompt and a short answer: latency
        dict(name="generate_base_1row", kind="generate", model="base", rows=1, prompt=37, new=64, top_k=0),
        # a batch of requests, greedy: the repository's headline workload with its prompt
        dict(name="generate_base_8rows", kind="generate", model="base", rows=8, prompt=512, new=128, top_k=0),
        # a full batch on the wide model with sampling; the prompt is no multiple of anything
        dict(name="generate_large_32rows_topk", kind="generate", model="large", rows=32, prompt=300, new=64, top_k=40),
        # a ragged prompt whose caches the program keeps
        dict(name="prompt_base_ragged", kind="prompt", model="base", rows=3, prompt=777),
        # long documents scored in one pass: every position's logits
        dict(name="score_large_long", kind="score", model="large", rows=4, prompt=4096),
        # a program that picks its tokens itself: a prompt, then one forward call per token on the caches
        dict(name="steps_base_4rows", kind="steps", model="base", rows=4, prompt=600, new=24),
        # the operator on its own: one long sequence (the shape the reference records a time for) ...
        dict(name="stu_long_1row", kind="stu", rows=1, length=4096, width=2048, dtype="bf16"),
        # ... and the smallest call of it in earnest: short, ragged, fp32
        dict(name="stu_short_fp32", kind="stu", rows=2, length=100, width=256, dtype="fp32"),
        # the operator with one projection per filter (use_approx=False) at the repository's benchmark shape
        dict(name="stu_exact_long", kind="exact", rows=4, length=8192, width=1024),
        # a training step of the operator: forward, and gradients of the input and of both weights
        dict(name="stu_train", kind="train", rows=8, length=2048, width=768, dtype="bf16"),
        # the dense LDS over a batch of sequences, the state carried: the repository's benchmark shape
        dict(name="lds_sequence", kind="lds", rows=64, length=4096, width=1024, state=160),
    ]


def _between(rng, lo, hi):
    """A whole number of lo..hi, spread over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    """One more case of the same kinds, anywhere between the smallest sizes in use and the largest listed ones."""
    kind = rng.choice(["generate", "generate", "prompt", "score", "steps", "stu", "stu", "exact", "train", "lds"])
    if kind == "generate":
        model = rng.choice(["tiny", "base", "base", "large"])
        rows = _between(rng, 1, 8 if model == "tiny" else 32)
        prompt = _between(rng, 16, 300 if model == "large" else 512 if rows <= 8 else 128)
        new = _between(rng, 16, 64 if model != "base" else 128)
        return dict(kind=kind, model=model, rows=rows, prompt=prompt, new=new, top_k=rng.choice([0, 40]))
    if kind == "prompt":     # longer than the attention window, so that the rings it returns are full
        rows = _between(rng, 1, 8)
        return dict(kind=kind, model="base", rows=rows, prompt=_between(rng, 514, 2048))
    if kind == "score":
        model = rng.choice(["base", "large"])
        rows = _between(rng, 1, 8)
        return dict(kind=kind, model=model, rows=rows, prompt=_between(rng, 40, min(2048 if model == "base" else 4096, 16384 // rows)))
    if kind == "steps":
        return dict(kind=kind, model="base", rows=_between(rng, 1, 16), prompt=_between(rng, 514, 1024), new=rng.randint(4, 24))
    if kind == "stu":
        width = rng.choice([256, 384, 512, 768, 1024, 1536, 2048])
        rows = _between(rng, 1, 8)
        return dict(kind=kind, rows=rows, length=_between(rng, 16, 8192), width=width, dtype=rng.choice(["bf16", "bf16", "fp32"]))
    if kind == "exact":
        return dict(kind=kind, rows=_between(rng, 1, 4), length=_between(rng, 64, 8192), width=rng.choice([256, 512, 768, 1024]))
    if kind == "train":
        rows = _between(rng, 1, 8)
        return dict(kind=kind, rows=rows, length=_between(rng, 64, 2048), width=rng.choice([256, 512, 768]), dtype=rng.choice(["bf16", "bf16", "fp32"]))
    return dict(kind=kind, rows=_between(rng, 1, 64), length=_between(rng, 64, 4096), width=rng.choice([256, 512, 1024]), state=rng.choice([32, 64, 96, 128, 160]))


# ---------------------------------------------------------------- what a program has in hand before the call
@functools.lru_cache(maxsize=None)
def _filters(length):
    """(length, FILTERS) float64 on the host: the leading eigenvectors of the Hankel matrix 2/(s^3-s), scaled by the
    fourth root of their eigenvalues, by subspace iteration (the spectrum falls so fast that a few rounds do; a
    full decomposition of 8192 rows takes minutes)."""
    i = torch.arange(1, length + 1, dtype=torch.float64, device="cuda")
    s = i[:, None] + i[None, :]
    z = 2.0 / (s * s * s - s)
    q = torch.randn(length, FILTERS + 16, dtype=torch.float64, generator=torch.Generator().manual_seed(0))
    for _ in range(8):
        q = torch.linalg.qr((z @ q.cuda()).cpu())[0]
    zq = (z @ q.cuda()).cpu()
    sigma, w = torch.linalg.eigh(q.T @ zq)
    sigma, w = sigma[-FILTERS:].clamp_min(1e-300), w[:, -FILTERS:]
    return (q @ w) * sigma ** 0.25


@functools.lru_cache(maxsize=1)
def _model(name):
    """The model a serving program keeps.  Its weights are scaled so that it behaves like a trained one: every sub-layer
    adds a fraction of the stream's size, and the picks are clear ones (the embedding's own direction outweighs what
    chance gives the other tokens), so that a rounding does not change which token comes next."""
    with tempfile.TemporaryDirectory() as folder:
        kw = MODELS[name]
        path = os.path.join(folder, "filters.pt")
        save_spectral_filters(_filters(kw["seq_len"]), path)
        cfg = FlashSTUConfig(vocab_size=VOCAB, num_eigh=FILTERS, filter_path=path, **kw)
        torch.manual_seed(1)
        with torch.device("cuda"):
            model = FlashSTU(cfg)
    model = model.cuda().eval()
    with torch.no_grad():
        for n, p in model.named_parameters():
            if n.endswith("proj.weight") and ".mlp." in n:
                p.normal_(0.0, 0.5 * cfg.n_embd ** -0.5)
            elif n in ("tok_emb.weight", "lm_head.weight"):
                p.normal_(0.0, 1.0)
            elif "norm" in n:
                p.normal_(1.0, 0.1)
    return model


def _stu(case, gen, exact=False):
    """An STU of the case's width with weights of the usual scales."""
    dt, d = DTYPES[case.get("dtype", "bf16")], case["width"]
    length = max(512, 1 << (case["length"] - 1).bit_length())
    cfg = FlashSTUConfig(n_embd=d, n_heads=d // 64, n_layers=2, seq_len=length, num_eigh=FILTERS, vocab_size=64, torch_dtype=dt, use_approx=not exact)
    stu = STU(cfg, _filters(length).to("cuda", dt), 2 * length).cuda()
    with torch.no_grad():
        for p in stu.parameters():
            fan_in = d if exact or p is stu.M_inputs else FILTERS
            p.normal_(0.0, fan_in ** -0.5, generator=gen)
    return stu


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    kind, rows = case["kind"], case["rows"]
    if kind in ("generate", "prompt", "score", "steps"):
        model = _model(case["model"])
        count = case["prompt"] + (case["new"] if kind == "steps" else 0)
        ids = torch.randint(0, VOCAB, (rows, count), generator=gen, device="cuda")
        return dict(case=case, model=model, ids=ids)
    if kind == "lds":
        length, d, s = case["length"], case["width"], case["state"]
        a = 0.9 + 0.099 * torch.rand(s, generator=gen, device="cuda")
        b = (torch.randn(d, s, generator=gen, device="cuda") / d).bfloat16()
        c = (torch.randn(s, d, generator=gen, device="cuda") / s).bfloat16()
        x = torch.randn(length, rows, d, generator=gen, device="cuda", dtype=torch.bfloat16)
        return dict(case=case, a=a, b=b, c=c, x=x)
    stu = _stu(case, gen, exact=kind == "exact")
    dt = DTYPES[case.get("dtype", "bf16")]
    x = torch.randn(rows, case["length"], case["width"], generator=gen, device="cuda", dtype=dt)
    if kind != "train":
        return dict(case=case, stu=stu, x=x)
    gy = torch.randn(rows, case["length"], case["width"], generator=gen, device="cuda", dtype=dt)
    return dict(case=case, stu=stu, x=x.requires_grad_(True), gy=gy)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "generate":
        model, k = state["model"], case["top_k"]
        how = dict(do_sample=True, top_k=k, temperature=0.8, seed=7) if k else dict(do_sample=False)
        tokens = model.generate(state["ids"], max_length=case["prompt"] + case["new"], **how)
        return dict(tokens=tokens, last_logits=model.decode_engine().logits if case["new"] > 1 else None)
    if kind == "prompt":
        out = state["model"](state["ids"], use_cache=True)
        return dict(logits=out.logits, caches=out.past_key_values)
    if kind == "score":
        return state["model"](state["ids"], use_cache=False).logits
    if kind == "steps":
        model, ids, p = state["model"], state["ids"], case["prompt"]
        out = model(ids[:, :p], use_cache=True)
        logits, past = [out.logits], out.past_key_values
        for t in range(p, p + case["new"]):
            out = model(ids[:, t:t + 1], past_key_values=past, use_cache=True)
            logits.append(out.logits)
            past = out.past_key_values
        return dict(logits=logits, caches=past)
    if kind in ("stu", "exact"):
        return state["stu"](state["x"])
    if kind == "train":
        stu, x = state["stu"], state["x"]
        for p in (x, stu.M_inputs, stu.M_filters):
            p.grad = None
        y = stu.forward_differentiable(x)
        y.backward(state["gy"])
        return dict(y=y.detach(), x=x.grad, inputs=stu.M_inputs.grad, filters=stu.M_filters.grad)
    h = torch.zeros(case["rows"], case["state"], device="cuda")
    y = _hip.lds_steps(h, state["x"], state["a"], state["b"], state["c"])
    return dict(y=y, state=h)


# ---------------------------------------------------------------- the least it takes
def _conv_flops(length):
    """One causal convolution through real transforms of twice the length: forward, both sign branches, back."""
    n = 2 * length
    return 3 * 2.5 * n * math.log2(max(n, 2)) + 12 * n


def _pass_work(cfg, rows, length, logits):
    """A prompt of `length` positions through the layers and the head over `logits` positions of each row."""
    d, layers, w, m = cfg["n_embd"], cfg["n_layers"], 4 if cfg["torch_dtype"] == torch.float32 else 2, rows * length
    inner = 12 * d
    weights = layers * 3 * d * inner + (layers // 2) * 5 * d * d + VOCAB * d
    seen = min(cfg["window_size"], length)
    flops = 2.0 * m * (weights - VOCAB * d) + 2.0 * rows * logits * VOCAB * d
    flops += layers // 2 * (4.0 * m * d * (seen - seen * seen / (2.0 * length)) + rows * d * _conv_flops(length))
    return w * weights + rows * logits * VOCAB * w + 8 * m, flops


def _step_work(cfg, rows, position):
    """One new position of each row against the caches."""
    d, layers, w = cfg["n_embd"], cfg["n_layers"], 4 if cfg["torch_dtype"] == torch.float32 else 2
    weights = layers * 36 * d * d + (layers // 2) * 5 * d * d + VOCAB * d
    kv = layers // 2 * rows * 2 * d * w * min(position, cfg["window_size"] + 1)
    if w == 2:      # recurrence state (one parity bank read and written, the other read) and its output weights
        stu = layers // 2 * (rows * STATE * d * 4 * 3 + 2 * STATE * d * 4)
    else:           # the history of projected inputs and the filter
        stu = layers // 2 * (rows + 1) * position * d * w
    return w * weights + kv + stu + rows * VOCAB * w, 2.0 * rows * weights + 2.0 * kv / w + stu / 2


def work(case):
    kind, rows = case["kind"], case["rows"]
    if kind in ("generate", "prompt", "score", "steps"):
        cfg, p = MODELS[case["model"]], case["prompt"]
        nbytes, flops = _pass_work(cfg, rows, p, 1 if kind == "generate" else p)
        # the prompt's own pick is the first new token of generate(); the steps kind feeds every given token
        for t in range(case.get("new", 0) - (1 if kind == "generate" else 0)):
            b, f = _step_work(cfg, rows, p + t)
            nbytes, flops = nbytes + b, flops + f
        return {"bytes": nbytes, "flops": flops}
    d, length = case["width"], case["length"]
    m = rows * length
    if kind == "lds":
        return {"bytes": 2 * m * d * 2 + 2 * d * case["state"] * 2, "flops": 4.0 * m * d * case["state"] + 2.0 * m * case["state"]}
    w = 4 if case.get("dtype") == "fp32" else 2
    if kind == "exact":
        return {"bytes": 2 * m * d * w + 2 * FILTERS * d * d * w + length * FILTERS * w,
                "flops": 4.0 * m * d * FILTERS * d + rows * d * (1 + 2 * FILTERS) * 2.5 * 2 * length * math.log2(2 * length)}
    forward = 2.0 * m * d * d + rows * d * _conv_flops(length)
    if kind == "stu":
        return {"bytes": 2 * m * d * w + d * d * w + length * FILTERS * w + FILTERS * d * w, "flops": forward}
    # training: y, gy in; gradients of x and the weights out; each product of the forward pass has two in the backward pass
    return {"bytes": 4 * m * d * w + 2 * d * d * w + 2 * FILTERS * d * w, "flops": 3 * forward}


def tolerance(case):
    """About four times what was seen: for the models against themselves with the residual stream's and the MLP's features
    in another order (so that every sum is formed in another order), for the operators against their float64 form."""
    if case["kind"] in ("generate", "prompt", "score", "steps"):
        if case["model"] == "tiny":                          # seen: rel 2e-7, max 9e-7
            return {"rel": 1e-5, "max": 5e-5, "differ": 0.0}
        return {"rel": 0.03, "max": 0.23, "differ": 0.0}     # seen: rel 0.011, max 0.058, no pick differs
    if case.get("dtype") == "fp32":                          # seen: rel 6e-7, max 4e-6 (2 x 500 positions)
        return {"rel": 1e-5, "max": 5e-5}
    return {"rel": 0.013, "max": 0.08}                       # seen: rel 0.0033, max 0.021
