"""Model-level GPU parity: FlashSTU / FlashSTUBlock on the HIP path against the
CPU oracle with identical weights and prompts.

fp32: greedy ids must match the oracle's full-recompute loop bit-exactly.
bf16: logits within 2e-2 (max abs error relative to the row's max |logit|) and
greedy ids equal on >= 99 % of positions when the oracle is teacher-forced with
the device's own tokens."""
import pytest
import torch

from oracle import flashstu_oracle as O

pytestmark = pytest.mark.gpu


def make_pair(seed=0, init="healthy", **kw):
    """(oracle cfg, oracle weights, device model) sharing the same tensors."""
    from flash_stu import FlashSTU, FlashSTUConfig
    dt = kw.pop("dtype", torch.float32)
    extra = {k: kw.pop(k) for k in ("stu_decode_mode", "stu_lds_state_dim", "stu_prefill_mode", "stu_lds_fir_taps") if k in kw}
    ocfg = O.OracleConfig(dtype=dt, **kw)
    w = O.init_weights(ocfg, seed=seed, mode=init)
    cfg = FlashSTUConfig(n_embd=ocfg.n_embd, n_heads=ocfg.n_heads, n_layers=ocfg.n_layers, seq_len=ocfg.seq_len,
                         window_size=ocfg.window_size, vocab_size=ocfg.vocab_size, mlp_scale=ocfg.mlp_scale,
                         num_eigh=ocfg.num_eigh, use_hankel_L=ocfg.use_hankel_L, use_approx=ocfg.use_approx,
                         use_attn=ocfg.use_attn, softcap=ocfg.softcap, torch_dtype=dt, **extra)
    torch.manual_seed(1234)
    model = FlashSTU(cfg)
    model.load_named_tensors(w)
    return ocfg, w, model.cuda().eval()


C1 = dict(n_embd=256, n_layers=4, n_heads=4, window_size=128, num_eigh=24, seq_len=1024, vocab_size=50257)


def prompt(B, P, V, seed):
    return torch.randint(0, V, (B, P), generator=torch.Generator().manual_seed(seed))


def replayed(model, ids, max_length, steps=8, do_sample=False, temperature=1.0, top_k=None, top_p=None, seed=0, between=None):
    """generate() with every step from a captured graph, whatever the number of chunks: graphs of `steps` steps, the rest as
    single-step graphs; `between` runs between the launches."""
    from flash_stu import _hip
    eng, (B, P) = model.decode_engine(), ids.shape
    how = (temperature, top_k, top_p, do_sample, seed)
    tokens = torch.zeros(B, max_length, dtype=torch.int64, device="cuda")
    tokens[:, :P] = ids
    with torch.no_grad():
        _hip.sample(eng.prefill(tokens[:, :P], max_length), tokens[:, P], *how, 0)
    done, todo = 0, max_length - P - 1
    try:
        for n in (steps, 1):
            if todo - done >= n:
                eng.graph_begin(tokens, P + done, 1 + done, *how, steps_per_graph=n)
            while todo - done >= n:
                eng.graph_step()
                done += n
                if between is not None:
                    between()
    finally:
        eng.graph_end()
    return tokens


@pytest.mark.parametrize("init,mlp_scale", [("reference", 12), ("healthy", 12), ("healthy", 4)])
def test_c1_fp32_greedy_ids_bit_exact(init, mlp_scale):
    """64-token prompt, 64 greedy tokens, fp32, seed 0."""
    ocfg, w, model = make_pair(seed=0, init=init, mlp_scale=mlp_scale, **C1)
    ids = prompt(1, 64, ocfg.vocab_size, 0)
    ref, ref_logits = O.generate(w, ocfg, ids, max_length=128, do_sample=False, mode="recompute", return_logits=True)
    got, got_logits = model.generate(ids.cuda(), max_length=128, do_sample=False, return_logits=True)
    assert got.shape == (1, 128)
    assert torch.equal(got.cpu(), ref), f"first mismatch at {int((got.cpu() != ref).nonzero()[0, 1])}"
    scale = float(ref_logits.abs().max())
    assert float((got_logits.cpu() - ref_logits).abs().max()) <= 1e-4 * scale


def test_fp32_sampling_matches_oracle_stream():
    """top-k / temperature sampling with the counter-based stream (config 5's
    sampler at a size the CPU oracle can follow)."""
    ocfg, w, model = make_pair(seed=2, init="healthy", mlp_scale=2, n_embd=128, n_layers=4, n_heads=2, window_size=16,
                               num_eigh=8, seq_len=128, vocab_size=997)
    ids = prompt(3, 10, ocfg.vocab_size, 1)
    ref = O.generate(w, ocfg, ids, max_length=60, temperature=0.8, top_k=40, do_sample=True, mode="stateful", seed=11)
    got = model.generate(ids.cuda(), max_length=60, temperature=0.8, top_k=40, do_sample=True, seed=11)
    assert torch.equal(got.cpu(), ref)
    again = model.generate(ids.cuda(), max_length=60, temperature=0.8, top_k=40, do_sample=True, seed=11)
    assert torch.equal(again, got)
    other = model.generate(ids.cuda(), max_length=60, temperature=0.8, top_k=40, do_sample=True, seed=12)
    assert not torch.equal(other, got)


def test_generate_without_cache_equals_with_cache():
    ocfg, w, model = make_pair(seed=3, init="healthy", mlp_scale=2, n_embd=128, n_layers=4, n_heads=2, window_size=8,
                               num_eigh=8, seq_len=64, vocab_size=503)
    ids = prompt(2, 7, ocfg.vocab_size, 2).cuda()
    a = model.generate(ids, max_length=40, do_sample=False, use_cache=True)
    b = model.generate(ids, max_length=40, do_sample=False, use_cache=False)
    assert torch.equal(a, b)
    assert model.generate(ids, max_length=7).shape == (2, 7)


@pytest.mark.parametrize("do_sample", [False, True])
def test_graph_replay_equals_eager_steps(do_sample):
    """The captured-step graph is replayed for many positions, with eager work and synchronisation in between,
    and must reproduce the eager token sequence exactly (same kernels, position read from device memory)."""
    ocfg, w, model = make_pair(seed=7, init="healthy", dtype=torch.bfloat16, mlp_scale=2, n_embd=128, n_layers=4,
                               n_heads=2, window_size=8, num_eigh=8, seq_len=128, vocab_size=1001, stu_decode_mode="lds")
    ids = prompt(3, 6, ocfg.vocab_size, 9).cuda()
    kw = dict(max_length=70, do_sample=do_sample, temperature=0.9, top_k=20, seed=5)
    eager = model.generate(ids, use_graph=False, **kw)

    def unrelated():
        torch.randn(256, 256, device="cuda") @ torch.randn(256, 256, device="cuda")
        torch.cuda.synchronize()
    for steps in (1, 8, 3):
        unrelated()
        assert torch.equal(model.generate(ids, use_graph=True, **kw), eager)
        assert torch.equal(replayed(model, ids, steps=steps, between=unrelated, **kw), eager)


@pytest.mark.parametrize("do_sample", [False, True])
@pytest.mark.parametrize("rows,d", [(33, 256), (40, 128)])
def test_several_chunks_replay_graphs(rows, d, do_sample, monkeypatch):
    """More rows than one chunk holds (a wide one of 32 rows and one of 1; three of up to 16): runs of single-step graphs, of
    8-step graphs alone and of both give the tokens of the steps launched one by one, and are runs of graphs."""
    from flash_stu.engine import DecodeEngine
    _, _, model = make_pair(seed=7, init="healthy", dtype=torch.bfloat16, mlp_scale=2, n_embd=d, n_layers=4, n_heads=2,
                            window_size=8, num_eigh=8, seq_len=64, vocab_size=1001)
    ids = prompt(rows, 5, 1001, 9).cuda()
    launches = []
    step = DecodeEngine.graph_step
    monkeypatch.setattr(DecodeEngine, "graph_step", lambda self, *a: (launches.append(self.graph_steps), step(self, *a)))
    for todo, graphs in ((2, [1] * 2), (9, [1] * 9), (31, [1] * 31), (32, [8] * 4), (37, [8] * 4 + [1] * 5)):
        kw = dict(max_length=5 + 1 + todo, do_sample=do_sample, temperature=0.9, top_k=20, seed=5)
        want = model.generate(ids, use_graph=False, **kw)
        assert not launches
        assert torch.equal(model.generate(ids, **kw), want)
        assert len(model.decode_engine().chunks) == (2 if d == 256 else 3) and launches == graphs
        launches.clear()


@pytest.mark.parametrize("dtype,mode", [(torch.bfloat16, "lds"), (torch.float32, "lds"), (torch.float32, "history")])
def test_scan_prefill_against_oracle_and_fft_prefill(dtype, mode):
    """stu_prefill_mode='scan' (the distilled recurrence over the prompt instead of the FFT convolution): prompt logits
    within the model-dtype tolerance of the oracle's, the decode state it leaves equal to the one the FFT path
    builds (same recurrence over the same projected inputs), and generation continues from it."""
    kw = dict(seed=5, init="healthy", dtype=dtype, mlp_scale=2, n_embd=128, n_layers=4, n_heads=2, window_size=16,
              num_eigh=8, seq_len=256, vocab_size=701, stu_decode_mode=mode)
    ocfg, w, fft = make_pair(**kw)
    _, _, scan = make_pair(stu_prefill_mode="scan", **kw)
    ids = prompt(2, 150, ocfg.vocab_size, 4)
    ref, _ = O.model_forward(w, ocfg, ids)
    a = fft(ids.cuda(), use_cache=True)
    b = scan(ids.cuda(), use_cache=True)
    scale = float(ref.abs().max())
    tol = 2e-2 if dtype == torch.bfloat16 else 2e-3      # fp32: the fit error of the 64-mode recurrence (about 1e-4 per layer)
    assert float((b.logits.float().cpu() - ref.float()).abs().max()) <= tol * scale
    assert float((b.logits.float() - a.logits.float()).abs().max()) <= tol * scale
    if mode == "lds":
        for ca, cb in zip(a.past_key_values, b.past_key_values):
            if len(ca) == 3 and ca[0].dim() == 3 and ca[0].shape[1] == 0:     # STU entry: (empty hist, state, pos)
                assert float((ca[1] - cb[1]).abs().max()) <= 2e-2 * float(ca[1].abs().max())
    out = scan.generate(ids.cuda(), max_length=170, do_sample=False)
    assert out.shape == (2, 170) and torch.equal(out[:, :150].cpu(), ids)


def test_hankel_L_decodes_on_the_recurrence_state():
    """use_hankel_L=True in bf16 decodes on the two-bank recurrence state (even lags from the token's bank, odd lags
    from the other one): logits of the stateful loop within the bf16 tolerance of the oracle teacher-forced on the
    same tokens, and of the cache-free loop."""
    ocfg, w, model = make_pair(seed=6, init="healthy", dtype=torch.bfloat16, mlp_scale=2, n_embd=128, n_layers=4,
                               n_heads=2, window_size=16, num_eigh=8, seq_len=128, vocab_size=503, use_hankel_L=True)
    assert model.config.resolved_stu_decode_mode() == "lds"
    P, N = 20, 40
    ids = prompt(2, P, ocfg.vocab_size, 3)
    got, gl = model.generate(ids.cuda(), max_length=P + N, do_sample=False, return_logits=True)
    ref = _teacher_forced(w, ocfg, got.cpu(), P)
    scale = float(ref.float().abs().max())
    assert float((gl.float().cpu() - ref.float()).abs().max()) <= 2e-2 * scale
    _, gl2 = model.generate(ids.cuda(), max_length=P + 8, do_sample=False, use_cache=False, return_logits=True)
    assert float((gl2.float() - gl[:, :8].float()).abs().max()) <= 2e-2 * scale


@pytest.mark.parametrize("hankel", [False, True])
def test_stu_forward_differentiable_gradients(hankel):
    """Training-side forward of the approx-mode STU under autograd: output equal to the inference forward, gradients
    of x, M_inputs and M_filters equal to autograd through the oracle's stu_forward (fp32)."""
    from flash_stu import STU, FlashSTUConfig
    L, K, d, B, T = 64, 8, 32, 2, 50
    cfg = FlashSTUConfig(n_embd=d, n_heads=2, n_layers=2, seq_len=L, num_eigh=K, vocab_size=11, torch_dtype=torch.float32,
                         use_hankel_L=hankel)
    phi = torch.tensor(O.get_spectral_filters_f64(L, K, hankel)).float()
    n = O.nearest_power_of_two(2 * L - 1, True)
    g = torch.Generator().manual_seed(17)
    Mi, Mf = torch.randn(d, d, generator=g) / d ** 0.5, torch.randn(K, d, generator=g) / K ** 0.5
    x, wgt = torch.randn(B, T, d, generator=g), torch.randn(B, T, d, generator=g)
    stu = STU(cfg, phi.cuda(), n).cuda()
    with torch.no_grad():
        stu.M_inputs.copy_(Mi)
        stu.M_filters.copy_(Mf)
    xd = x.cuda().requires_grad_(True)
    y = stu.forward_differentiable(xd)
    assert float((y.detach() - stu(x.cuda())).abs().max()) <= 2e-5 * float(y.detach().abs().max())
    (y * wgt.cuda()).sum().backward()
    xo = x.clone().requires_grad_(True)
    p = {"M_inputs": Mi.clone().requires_grad_(True), "M_filters": Mf.clone().requires_grad_(True)}
    ref = O.stu_forward(xo, phi, p, n, use_approx=True, use_hankel_L=hankel)
    (ref * wgt).sum().backward()
    for got, want in ((xd.grad, xo.grad), (stu.M_inputs.grad, p["M_inputs"].grad), (stu.M_filters.grad, p["M_filters"].grad)):
        assert float((got.cpu() - want).abs().max()) <= 2e-4 * float(want.abs().max())


@pytest.mark.parametrize("hankel", [False, True])
@pytest.mark.parametrize("T", [20, 50])
def test_stu_forward_differentiable_second_order(hankel, T):
    """create_graph=True through the whole operator, at a length of the time-domain kernel and one of the transforms: gradients
    of a penalty on the gradients against autograd through the oracle.  Each order of differentiation is one more pass of
    fp32 convolutions and products: five times the bound of the first-order test."""
    from flash_stu import STU, FlashSTUConfig
    L, K, d, B = 64, 8, 32, 2
    cfg = FlashSTUConfig(n_embd=d, n_heads=2, n_layers=2, seq_len=L, num_eigh=K, vocab_size=11, torch_dtype=torch.float32,
                         use_hankel_L=hankel)
    phi = torch.tensor(O.get_spectral_filters_f64(L, K, hankel)).float()
    n = O.nearest_power_of_two(2 * L - 1, True)
    g = torch.Generator().manual_seed(18)
    Mi, Mf = torch.randn(d, d, generator=g) / d ** 0.5, torch.randn(K, d, generator=g) / K ** 0.5
    x, wgt = torch.randn(B, T, d, generator=g), torch.randn(B, T, d, generator=g)
    stu = STU(cfg, phi.cuda(), n).cuda()
    with torch.no_grad():
        stu.M_inputs.copy_(Mi)
        stu.M_filters.copy_(Mf)
    p = {"M_inputs": Mi.clone().requires_grad_(True), "M_filters": Mf.clone().requires_grad_(True)}
    seconds = []
    for leaves, y, w in (((x.cuda().requires_grad_(True), stu.M_inputs, stu.M_filters), stu.forward_differentiable, wgt.cuda()),
                         ((x.clone().requires_grad_(True), *p.values()), lambda t: O.stu_forward(t, phi, p, n, use_approx=True, use_hankel_L=hankel), wgt)):
        first = torch.autograd.grad((y(leaves[0]).square() * w).sum(), leaves, create_graph=True)
        seconds.append(torch.autograd.grad(sum(t.square().sum() / t.detach().square().sum() for t in first), leaves))
    for got, want in zip(*seconds):
        assert float((got.cpu() - want).abs().max()) <= 1e-3 * float(want.abs().max())


@pytest.mark.parametrize("B,T,d", [(4, 32, 128), (3, 201, 256), (1, 1025, 128)])
def test_training_step_as_one_node(B, T, d, monkeypatch):
    """forward_differentiable in bf16 as one autograd node against its composed operators: outputs and gradients, x expanded, off its
    alignment and strided, parameters frozen, and the gradients of the gradients.  Three roundings to bf16 (2^-8 each) lie
    between the two in any of them."""
    from flash_stu import STU, FlashSTUConfig
    from flash_stu.utils.stu_utils import ApproxUnit
    L, K = 1040, 24
    g = torch.Generator().manual_seed(T)
    cfg = FlashSTUConfig(n_embd=d, n_heads=2, n_layers=2, seq_len=L, num_eigh=K, vocab_size=11, torch_dtype=torch.bfloat16)
    stu = STU(cfg, torch.randn(L, K, generator=g).div(L ** 0.5).bfloat16().cuda(), 4096).cuda()
    with torch.no_grad():
        for p in (stu.M_inputs, stu.M_filters):
            p.copy_(torch.randn(p.shape, generator=g) / p.shape[0] ** 0.5)
    x, gy = (torch.randn(B, T, d, generator=g).bfloat16().cuda() for _ in range(2))
    shifted = torch.empty(B * T * d + 1, dtype=torch.bfloat16, device="cuda")[1:].view(B, T, d).copy_(x)
    strided = torch.empty(T, B, d, dtype=torch.bfloat16, device="cuda").transpose(0, 1).copy_(x)
    close = lambda a, b: float((a.float() - b.float()).norm()) <= 3 * 2.0 ** -8 * float(b.float().norm())
    made = []
    takes = ApproxUnit.takes

    def pass_of(xi, wanted, second=False):
        xi = xi.detach().requires_grad_(0 in wanted)
        for i, p in enumerate((stu.M_inputs, stu.M_filters), 1):
            p.requires_grad_(i in wanted)
        leaves = [t for i, t in enumerate((xi, stu.M_inputs, stu.M_filters)) if i in wanted]
        y = stu.forward_differentiable(xi)
        grads = torch.autograd.grad(y, leaves, gy, create_graph=second)
        if second:
            grads = torch.autograd.grad(sum(t.float().square().sum() / t.detach().float().square().sum() for t in grads), leaves)
        return y.detach(), *grads
    for xi, wanted, second in ((x, (0, 1, 2), False), (shifted, (0, 1, 2), False), (strided, (1, 2), False), (x[:1].expand(B, T, d), (0, 2), False),
                               (x, (2,), False), (x, (1,), False), (x, (0,), False), (x, (0, 1, 2), True)):
        both = []
        for node in (True, False):
            monkeypatch.setattr(ApproxUnit, "takes", staticmethod(lambda *a: made.append(takes(*a)) or (node and made[-1])))
            both.append(pass_of(xi, wanted, second))
        assert len(both[0]) == 1 + len(wanted) and all(close(a, b) and a.shape == b.shape for a, b in zip(*both))
    assert all(made)


def test_filter_weights_may_change_before_the_backward_pass():
    """No gradient of first order needs the values of M_filters: an update between the passes leaves the gradients those of the
    forward pass's weights, bit for bit, and those with a graph of their own within three roundings to bf16 (2^-8 each)."""
    from flash_stu import STU, FlashSTUConfig
    B, T, d, L, K = 4, 64, 128, 128, 24
    g = torch.Generator().manual_seed(5)
    cfg = FlashSTUConfig(n_embd=d, n_heads=2, n_layers=2, seq_len=L, num_eigh=K, vocab_size=11, torch_dtype=torch.bfloat16)
    stu = STU(cfg, torch.randn(L, K, generator=g).div(L ** 0.5).bfloat16().cuda(), 256).cuda()
    mf = (torch.randn(K, d, generator=g) / K ** 0.5).cuda()
    with torch.no_grad():
        stu.M_inputs.copy_(torch.randn(d, d, generator=g) / d ** 0.5)
    x, gy = (torch.randn(B, T, d, generator=g).bfloat16().cuda() for _ in range(2))
    x.requires_grad_(True)
    runs = []
    for update, second in ((False, False), (True, False), (True, True)):
        with torch.no_grad():
            stu.M_filters.copy_(mf)
        y = stu.forward_differentiable(x)
        if update:
            with torch.no_grad():
                stu.M_filters.mul_(-3.0)
        runs.append(torch.autograd.grad(y, (x, stu.M_inputs, stu.M_filters), gy, create_graph=second))
    for want, got, graph in zip(*runs):
        assert torch.equal(got, want)
        assert float((graph.detach().float() - want.float()).norm()) <= 3 * 2.0 ** -8 * float(want.float().norm())


@pytest.mark.parametrize("second", [False, True])
def test_what_no_gradient_needs_may_change_before_the_backward_pass(second):
    """Where M_filters alone is trained its gradient needs neither x nor M_inputs, where it is frozen none needs phi: an update of them
    between the passes leaves the gradients those of the forward pass, bit for bit."""
    from flash_stu import STU, FlashSTUConfig
    B, T, d, L, K = 4, 64, 128, 128, 24
    g = torch.Generator().manual_seed(6)
    cfg = FlashSTUConfig(n_embd=d, n_heads=2, n_layers=2, seq_len=L, num_eigh=K, vocab_size=11, torch_dtype=torch.bfloat16)
    stu = STU(cfg, torch.randn(L, K, generator=g).div(L ** 0.5).bfloat16().cuda(), 256).cuda()
    start = [torch.randn(p.shape, generator=g).div(p.shape[0] ** 0.5).bfloat16().cuda() for p in (stu.M_inputs, stu.M_filters)] + [stu.phi.clone()]
    x0, gy = (torch.randn(B, T, d, generator=g).bfloat16().cuda() for _ in range(2))
    for wanted, changed in (((2,), (0, 1)), ((0, 1), (3,)), ((1,), (3,))):
        runs = []
        for update in (False, True):
            x = x0.clone()
            leaves = (x, stu.M_inputs, stu.M_filters, stu.phi)
            with torch.no_grad():
                for t, v in zip(leaves[1:], start):
                    t.copy_(v)
            for i, t in enumerate(leaves[:3]):
                t.requires_grad_(i in wanted)
            y = stu.forward_differentiable(x)
            with torch.no_grad():
                for i in changed if update else ():
                    leaves[i].mul_(-3.0)
            runs.append(torch.autograd.grad(y, [leaves[i] for i in wanted], gy, create_graph=second))
        assert all(torch.equal(a, b) for a, b in zip(*runs))


@pytest.mark.parametrize("B,T,d", [(1, 128, 128), (3, 320, 256), (2, 97, 128)])
def test_input_projection_gradients(B, T, d):
    """x @ M_inputs and its gradients on the matrix-core kernels (and, for rows they do not take, the library's product)
    against float64: fp32 sums of exact products, one rounding to bf16 (2^-8 of the value) each; x expanded, shifted off its
    alignment and frozen."""
    from flash_stu.utils.stu_utils import ProjectInputs
    g = torch.Generator().manual_seed(B * T)
    x, m, w = (torch.randn(*s, generator=g).bfloat16().cuda() for s in ((B, T, d), (d, 2 * d), (B, T, 2 * d)))
    assert ProjectInputs.takes(x, m) == (B * T % 64 == 0)
    project = ProjectInputs.apply if ProjectInputs.takes(x, m) else torch.matmul
    shifted = torch.empty(B * T * d + 1, dtype=torch.bfloat16, device="cuda")[1:].view(B, T, d).copy_(x)
    for xi in (x, shifted, x[:1].expand(B, T, d)):
        xi, mi = xi.detach().requires_grad_(True), m.clone().requires_grad_(True)
        y = project(xi, mi)
        y.backward(w)
        xd, md, wd = xi.detach().double().reshape(-1, d), m.double(), w.double().reshape(-1, 2 * d)
        for got, a, b in ((y.detach(), xd, md), (xi.grad, wd, md.t()), (mi.grad, xd.t(), wd)):
            ref, mag = a @ b, a.abs() @ b.abs()
            err = (got.double().reshape(ref.shape) - ref).abs()
            assert bool((err <= 2.0 ** -8 * ref.abs() + a.shape[1] * 2.0 ** -23 * mag).all())
    xi = x.clone().requires_grad_(True)
    project(xi, m).backward(w)                         # m needs no gradient
    assert xi.grad.shape == x.shape and m.grad is None


def test_input_projection_gradients_of_gradients():
    """create_graph=True: the gradients of x @ m carry their own graph, as those of the plain product do.  Same bf16 products in
    both: two roundings (2^-8 each) of sums of the same terms."""
    from flash_stu.utils.stu_utils import ProjectInputs
    g = torch.Generator().manual_seed(3)
    x0, m0, w = (torch.randn(*s, generator=g).bfloat16().cuda() for s in ((2, 64, 128), (128, 128), (2, 64, 128)))
    seconds = []
    for f in (ProjectInputs.apply, torch.matmul):
        x, m = x0.clone().requires_grad_(True), m0.clone().requires_grad_(True)
        gx, gm = torch.autograd.grad(f(x, m), (x, m), w, create_graph=True)
        assert gx.requires_grad and gm.requires_grad
        seconds.append(torch.autograd.grad(gx.float().square().sum() + gm.float().square().sum(), (x, m)))
    for got, ref in zip(*seconds):
        assert float((got.float() - ref.float()).norm()) <= 2.0 ** -7 * float(ref.float().norm())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,d", [(1, 64), (3, 256), (16, 512)])
def test_greedy_steps_in_one_call(dtype, B, d):
    """fstu_decode_steps, whose picks are finished in the launch that begins the next step, against a call per step: the same tokens, and
    nothing left of one call's maxima for the next; the last step's logits against those of one pass over all tokens, which knows
    neither steps nor that launch."""
    from flash_stu import FlashSTU, FlashSTUConfig
    torch.manual_seed(B)
    cfg = FlashSTUConfig(n_embd=d, n_heads=2, n_layers=2, seq_len=64, window_size=16, vocab_size=501, num_eigh=8, torch_dtype=dtype)
    model = FlashSTU(cfg).cuda().eval()
    with torch.no_grad():
        model.lm_head.weight.normal_(0.0, 1.0)         # the picks are clear ones: another order of the norm's sum does not change them
    ids = torch.randint(0, 501, (B, 9), generator=torch.Generator().manual_seed(d)).cuda()
    for n in (1, 2, 3, 30):
        one = model.generate(ids, max_length=9 + n, do_sample=False)
        each, _ = model.generate(ids, max_length=9 + n, do_sample=False, return_logits=True)
        assert torch.equal(one, each), n
        if n > 1:
            model.generate(ids, max_length=9 + n, do_sample=False)
            got, ref = model.decode_engine().logits.float(), model(one[:, :-1], use_cache=False).logits[:, -1].float()
            assert float((got - ref).abs().max()) <= (1e-4 if dtype == torch.float32 else 3e-2) * float(ref.abs().max()), n


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_refused_steps_leave_no_pick_behind(dtype):
    """A step behind the end of the history is refused: the picks of the steps in front of it are written all the same, and nothing of
    them is left for the next call, which gives the tokens of a fresh descriptor."""
    from flash_stu import FlashSTU, FlashSTUConfig, _hip
    B, P, cap = 3, 9, 64
    torch.manual_seed(4)
    cfg = FlashSTUConfig(n_embd=64, n_heads=2, n_layers=2, seq_len=cap, window_size=cap, vocab_size=501, num_eigh=8, torch_dtype=dtype,
                         stu_decode_mode="history")
    model = FlashSTU(cfg).cuda().eval()
    with torch.no_grad():
        model.lm_head.weight.normal_(0.0, 1.0)
    ids = torch.randint(0, 501, (B, P), generator=torch.Generator().manual_seed(4)).cuda()
    want = model.generate(ids, max_length=cap, do_sample=False)
    eng = model.decode_engine()
    assert eng.desc.hist_cap == cap
    for n, refused in ((cap - P + 1, True), (cap - P, False)):
        tokens = torch.zeros(B, cap + 3, dtype=torch.int64, device="cuda")
        tokens[:, :P + 1] = want[:, :P + 1]
        how = (tokens, P, n, 1.0, None, None, False, 0, 1)
        if refused:
            with pytest.raises(_hip.FlashSTUHipError, match="history capacity"):
                eng.steps(*how)
        else:
            eng.steps(*how)
        assert torch.equal(tokens[:, :cap], want)
        assert torch.equal(tokens[:, cap], eng.logits.float().argmax(-1)) and int(tokens[:, cap + 1:].abs().sum()) == 0


def _teacher_forced(w, ocfg, tokens, P):
    logits, _ = O.model_forward(w, ocfg, tokens[:, :-1])
    return logits[:, P - 1:, :]          # predictions for positions P..end


class _wide_accumulation:
    """Inside the block every F.linear of the oracle accumulates in float64 and rounds once to the model dtype: the
    same specification (same rounding points) under another summation order than the CPU library's."""
    def __enter__(self):
        self.saved = O.F.linear

        def wide(x, w, b=None):
            y = x.double() @ w.double().t()
            if b is not None:
                y = y + b.double()
            return y.to(x.dtype)
        O.F.linear = wide

    def __exit__(self, *a):
        O.F.linear = self.saved


def _bf16_parity(ocfg, w, model, ids, N, label):
    """Greedy decode on the device, the oracle teacher-forced on the device's tokens.  Returns (worst relative
    logit error, strict agreement of the greedy ids, the comparison's own noise floor, scored picks).  The floor
    is the oracle against itself with float64 accumulation inside every linear (same rounding points, another
    summation order): two faithful evaluations of one bf16 specification do not pick the same token every time."""
    B, P = ids.shape
    got, got_logits = model.generate(ids.cuda(), max_length=P + N, do_sample=False, return_logits=True)
    got, got_logits = got.cpu(), got_logits.float().cpu()
    ref_logits = _teacher_forced(w, ocfg, got, P).float()
    assert ref_logits.shape == got_logits.shape
    err = float(((got_logits - ref_logits).abs().amax(-1) / ref_logits.abs().amax(-1)).max())
    agree = float((ref_logits.argmax(-1) == got[:, P:]).float().mean())
    with _wide_accumulation():
        ref2 = _teacher_forced(w, ocfg, got, P).float()
    floor = float((ref2.argmax(-1) == ref_logits.argmax(-1)).float().mean())
    floor_err = float(((ref2 - ref_logits).abs().amax(-1) / ref_logits.abs().amax(-1)).max())
    print(f"{label}: {B * N} picks, max rel logit err {err:.2e} (oracle vs oracle(float64 accumulation) {floor_err:.2e}), "
          f"strict greedy agreement {agree:.4f}, floor {floor:.4f}")
    return err, agree, floor, B * N


@pytest.mark.parametrize("mode", ["history", "lds"])
@pytest.mark.parametrize("init", ["healthy", "reference"])
def test_c2_dims_bf16_teacher_forced(mode, init):
    """BASELINE config 2's architecture (768-d, 12 layers, 12 heads, window 512, L=2048) at a prompt/batch the CPU
    oracle finishes in seconds, 2000 scored picks per cell.  Tolerances from BASELINE.json: logits within 2e-2
    relative; greedy ids agree on >= 99 % of the tokens wherever the specification agrees with itself that often, and
    never fall more than one point below the comparison's own noise floor."""
    ocfg, w, model = make_pair(seed=1, init=init, dtype=torch.bfloat16, mlp_scale=4, n_embd=768, n_layers=12,
                               n_heads=12, window_size=512, num_eigh=24, seq_len=2048, vocab_size=50257,
                               stu_decode_mode=mode)
    B, P, N = 8, 40, 250
    err, agree, floor, picks = _bf16_parity(ocfg, w, model, prompt(B, P, ocfg.vocab_size, 3), N, f"mode={mode} init={init}")
    assert picks >= 2000
    assert err <= 2e-2, err
    assert agree >= min(0.99, floor - 0.01), (agree, floor)


def test_c2_benched_config_bf16_against_the_oracle_past_the_ring_wrap():
    """The configuration bench.py runs (mlp_scale 12, recurrence STU state, window 512) with a prompt longer than the
    ring (513 slots): the decode steps read a wrapped ring and a recurrence state older than the window, and their
    logits are compared with the oracle's full-sequence forward (teacher-forced on the device's tokens)."""
    ocfg, w, model = make_pair(seed=1, init="reference", dtype=torch.bfloat16, mlp_scale=12, n_embd=768, n_layers=12,
                               n_heads=12, window_size=512, num_eigh=24, seq_len=2048, vocab_size=50257,
                               stu_decode_mode="lds")
    B, P, N = 4, 530, 125
    err, agree, floor, picks = _bf16_parity(ocfg, w, model, prompt(B, P, ocfg.vocab_size, 5), N, "benched config, lds")
    assert err <= 2e-2, err
    # 500 picks: the sampling noise of an agreement near 0.97 is 0.8 points, so the margin is two points here
    assert agree >= min(0.99, floor - 0.02), (agree, floor)


def test_c2_full_size_decode_against_full_sequence_recompute():
    """BASELINE config 2 at its full size (batch 8, 512-token prompt, window 512, mlp_scale 12), where the CPU oracle is
    out of reach: the stateful decode (ring past its wrap, recurrence state past the window) must give the logits of
    a full-sequence forward over the same tokens (the prefill kernels, tied to the oracle at small sizes), and the
    8-step graphs with the chained pick must reproduce the kernel-by-kernel loop token for token."""
    from flash_stu import FlashSTU, FlashSTUConfig
    torch.manual_seed(1)
    cfg = FlashSTUConfig(n_embd=768, n_layers=12, n_heads=12, window_size=512, seq_len=2048, vocab_size=50257,
                         num_eigh=24, mlp_scale=12, torch_dtype=torch.bfloat16)
    with torch.device("cuda"):
        model = FlashSTU(cfg)
    model = model.cuda().eval()
    B, P, N = 8, 512, 40
    ids = prompt(B, P, cfg.vocab_size, 1).cuda()
    eager, logits = model.generate(ids, max_length=P + N, do_sample=False, return_logits=True)      # step by step
    assert torch.equal(model.generate(ids, max_length=P + N, do_sample=False), eager)
    assert torch.equal(replayed(model, ids, P + N), eager)                                          # 8-step graphs
    worst = 0.0
    for s in (0, 1, 7, 20, N - 1):          # logits that picked token P+s come from positions < P+s
        full = model(eager[:, :P + s].contiguous()).logits[:, -1, :].float()
        got = logits[:, s, :].float()
        worst = max(worst, float(((got - full).abs().amax(-1) / full.abs().amax(-1)).max()))
    assert worst <= 2e-2, worst


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_single_token_prompt_and_ragged_batches(dtype):
    """Edge cases of the token loop: a one-token prompt (the prefill is a single position), batches of 1 and of 17
    rows (one full row chunk of 16 plus a chunk of one), a single new token, and max_length equal to the prompt."""
    ocfg, w, model = make_pair(seed=9, init="healthy", dtype=dtype, mlp_scale=2, n_embd=128, n_layers=4, n_heads=2,
                               window_size=8, num_eigh=8, seq_len=64, vocab_size=307)
    for B in (1, 17):
        ids = prompt(B, 1, ocfg.vocab_size, B)
        if dtype == torch.float32:
            ref = O.generate(w, ocfg, ids, max_length=20, do_sample=False, mode="recompute")
            got = model.generate(ids.cuda(), max_length=20, do_sample=False)
            assert torch.equal(got.cpu(), ref)
        else:
            got, gl = model.generate(ids.cuda(), max_length=20, do_sample=False, return_logits=True)
            ref = _teacher_forced(w, ocfg, got.cpu(), 1).float()
            assert float(((gl.float().cpu() - ref).abs().amax(-1) / ref.abs().amax(-1)).max()) <= 2e-2
            assert torch.equal(model.generate(ids.cuda(), max_length=20, do_sample=False), got)
            assert torch.equal(replayed(model, ids.cuda(), 20), got)
        one = model.generate(ids.cuda(), max_length=2, do_sample=False)
        assert one.shape == (B, 2) and torch.equal(one[:, :2], got[:, :2])
        assert torch.equal(model.generate(ids.cuda(), max_length=1), ids.cuda())


def test_window_wraps_the_ring_bf16():
    """Decode far past window+1 so every ring slot is overwritten several times."""
    ocfg, w, model = make_pair(seed=4, init="healthy", dtype=torch.bfloat16, mlp_scale=2, n_embd=128, n_layers=4,
                               n_heads=2, window_size=8, num_eigh=8, seq_len=128, vocab_size=1001,
                               stu_decode_mode="history")
    B, P, N = 2, 5, 60
    ids = prompt(B, P, ocfg.vocab_size, 5)
    got, gl = model.generate(ids.cuda(), max_length=P + N, do_sample=False, return_logits=True)
    ref_logits = _teacher_forced(w, ocfg, got.cpu(), P).float()
    err = (gl.float().cpu() - ref_logits).abs().amax(-1) / ref_logits.abs().amax(-1)
    assert float(err.max()) <= 2e-2


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_forward_full_sequence_and_stepwise_cache(dtype):
    ocfg, w, model = make_pair(seed=5, init="healthy", dtype=dtype, mlp_scale=2, n_embd=128, n_layers=4, n_heads=2,
                               window_size=8, num_eigh=8, seq_len=64, vocab_size=777)
    ids = prompt(2, 24, ocfg.vocab_size, 6)
    ref, _ = O.model_forward(w, ocfg, ids)
    out = model(ids.cuda())
    tol = 1e-4 if dtype == torch.float32 else 3e-2
    scale = float(ref.float().abs().max())
    assert out.logits.shape == (2, 24, 777)
    assert float((out.logits.float().cpu() - ref.float()).abs().max()) <= tol * scale
    assert len(out.past_key_values) == 4                       # use_cache defaults to config.use_cache (True)
    kr, vr, pos = out.past_key_values[1]
    assert kr.shape == (2, 2, 9, 64) and int(pos[0]) == 24
    # prefill 10, then feed the rest one token at a time through forward()
    o = model(ids[:, :10].cuda(), use_cache=True)
    cache = o.past_key_values
    for t in range(10, 24):
        o = model(ids[:, t:t + 1].cuda(), past_key_values=cache, use_cache=True)
        cache = o.past_key_values
        assert float((o.logits[:, 0].float().cpu() - ref[:, t].float()).abs().max()) <= tol * scale
    # tuple return and hidden states
    tup = model(ids.cuda(), use_cache=False, return_dict=False, output_hidden_states=True)
    assert len(tup) == 2 and len(tup[1]) == 5
    # beam reordering keeps working on the cache tuples
    re = model._reorder_cache(cache, torch.tensor([1, 0]))
    assert torch.equal(re[1][0][0], cache[1][0][1])


@pytest.mark.parametrize("rows", [1, 3, 16])
@pytest.mark.parametrize("dtype,extra", [(torch.float32, dict(n_embd=96, n_heads=3)), (torch.float32, dict(use_hankel_L=True)),
                                         (torch.bfloat16, dict(n_embd=256)), (torch.bfloat16, dict(n_embd=96, n_heads=3)),
                                         (torch.bfloat16, dict(stu_lds_fir_taps=0, softcap=0.0)), (torch.bfloat16, dict(use_attn=False)),
                                         (torch.bfloat16, dict(stu_decode_mode="history"))])
def test_one_call_step_equals_the_layers_own_calls(dtype, extra, rows):
    """forward() with caches for one position: the one-call step against the layers' forward calls (a hook that does nothing
    keeps those in use), logits and caches, over the edges of the prompt's fill of rings and of the row range."""
    from flash_stu import engine
    kw = dict(mlp_scale=2, n_embd=128, n_layers=4, n_heads=2, window_size=8, num_eigh=8, seq_len=64, vocab_size=777)
    _, _, model = make_pair(seed=5, init="healthy", dtype=dtype, **{**kw, **extra})
    ids = prompt(rows, 14, 777, 6).cuda()
    caches = {}
    for how in ("one", "layers"):
        hook = model.norm.register_forward_hook(lambda *a: None) if how == "layers" else None
        out = model(ids[:, :6], use_cache=True)
        logits, past = [out.logits[:, -1:]], out.past_key_values
        assert (engine.step_on_caches(model, ids[:, 6:7], tuple(tuple(t.clone() for t in c) for c in past)) is None) == (how == "layers")
        for t in range(6, 14):
            out = model(ids[:, t:t + 1], past_key_values=past, use_cache=True)
            assert out.logits.shape == (rows, 1, 777)
            logits.append(out.logits)
            past = out.past_key_values
        caches[how] = (torch.cat(logits, 1), past)
        if hook is not None:
            hook.remove()
    # sums in another order: fp32 as the forward tests hold it; bf16 a few roundings of 2^-8 that pass through four layers
    tol = 1e-4 if dtype == torch.float32 else 2e-2
    (la, ca), (lb, cb) = caches["one"], caches["layers"]
    assert float((la.float() - lb.float()).abs().max()) <= tol * float(lb.float().abs().max())
    for i, (ea, eb) in enumerate(zip(ca, cb)):
        attn = len(ea) == 3 and ea[0].dim() == 4
        for a, b in zip(ea, eb):
            if attn and a.dim() == 4:                            # slots beyond the last position are not written
                a, b = a[:, :, :min(14, 9)], b[:, :, :min(14, 9)]
            assert a.shape == b.shape and a.dtype == b.dtype
            if a.numel():
                assert float((a.float() - b.float()).abs().max()) <= tol * max(float(b.float().abs().max()), 1e-6)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_weights_changed_between_two_steps_on_caches_are_seen(dtype):
    """Every parameter scaled in place between two positions: the second step is that of the layers' own calls (sums in another
    order, bounds as above) and not that of the weights before."""
    _, _, model = make_pair(seed=5, init="healthy", dtype=dtype, mlp_scale=2, n_embd=128, n_layers=4, n_heads=2, window_size=8,
                            num_eigh=8, seq_len=64, vocab_size=777)
    ids = prompt(3, 8, 777, 2).cuda()
    out = model(ids[:, :6], use_cache=True)
    past = model(ids[:, 6:7], past_key_values=out.past_key_values, use_cache=True).past_key_values
    copies = [tuple(tuple(t.clone() for t in c) for c in past) for _ in range(2)]
    before = model(ids[:, 7:8], past_key_values=past, use_cache=True).logits.float()
    with torch.no_grad():
        for i, p in enumerate(model.parameters()):
            p.mul_(1.0 + 0.1 * (i % 3))
    one = model(ids[:, 7:8], past_key_values=copies[0], use_cache=True).logits.float()
    hook = model.norm.register_forward_hook(lambda *a: None)
    layers = model(ids[:, 7:8], past_key_values=copies[1], use_cache=True).logits.float()
    hook.remove()
    scale = float(layers.abs().max())
    assert float((one - layers).abs().max()) <= (1e-4 if dtype == torch.float32 else 2e-2) * scale
    assert float((one - before).abs().max()) > 5e-2 * scale


class _Scaled(torch.nn.Module):
    def forward(self, w):
        return w * 0.5


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 256), (torch.float32, 128)])
def test_parametrized_projections_are_held_until_they_are_read(dtype, d):
    """A parametrized weight is a new tensor on every access.  Scaling by 0.5 is exact, so the caches' one-call step and
    generate() give the bits of a model whose weights were scaled beforehand."""
    from torch.nn.utils import parametrize
    kw = dict(seed=5, init="healthy", dtype=dtype, mlp_scale=2, n_embd=d, n_layers=4, n_heads=2, window_size=8, num_eigh=8,
              seq_len=64, vocab_size=777)
    _, _, plain = make_pair(**kw)
    _, _, model = make_pair(**kw)
    for scaled, layer in zip(plain.layers, model.layers):
        names = ["mlp.gate_proj", "mlp.up_proj", "mlp.down_proj"] + (["attn.c_attn", "attn.c_proj"] if hasattr(layer, "attn") else [])
        for name in names:
            with torch.no_grad():
                scaled.get_submodule(name).weight.mul_(0.5)
            parametrize.register_parametrization(layer.get_submodule(name), "weight", _Scaled())
    for rows in (3, 16, 20):
        ids = prompt(rows, 10, 777, rows).cuda()
        if rows <= 16:
            outs = []
            for m in (plain, model):
                past, logits = m(ids[:, :6], use_cache=True).past_key_values, []
                for t in range(6, 10):
                    out = m(ids[:, t:t + 1], past_key_values=past, use_cache=True)
                    past = out.past_key_values
                    logits.append(out.logits)
                outs.append(torch.cat(logits, 1))
            assert torch.equal(*outs)
        assert torch.equal(model.generate(ids, max_length=20, do_sample=False), plain.generate(ids, max_length=20, do_sample=False))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_step_on_caches_takes_expanded_ids(dtype):
    """One token for all rows as an expanded view, or as a column of a longer buffer: the logits of a dense column."""
    _, _, model = make_pair(seed=5, init="healthy", dtype=dtype, mlp_scale=2, n_embd=256, n_layers=4, n_heads=2, window_size=8,
                            num_eigh=8, seq_len=64, vocab_size=777)
    for rows in (1, 3):
        ids = prompt(rows, 6, 777, rows).cuda()
        past = model(ids, use_cache=True).past_key_values
        token = ids[0, 2]
        step = lambda column: model(column, past_key_values=tuple(tuple(t.clone() for t in c) for c in past), use_cache=True).logits
        want = step(token.repeat(rows, 1))
        for column in (token.expand(rows, 1), token.reshape(1, 1).expand(rows, 4)[:, 2:3], token.repeat(rows, 5)[:, 3:4]):
            assert torch.equal(step(column), want)


@pytest.mark.parametrize("what", ["MLP.forward", "RMSNorm.add_then_norm", "STU._step", "instance", "subclass", "model"])
def test_replaced_methods_run_in_a_step_on_caches(what, monkeypatch):
    """A method replaced on a class, an instance or in a subclass is called for one position on caches too."""
    from flash_stu import FlashSTU
    from flash_stu.modules.norm import RMSNorm
    from flash_stu.modules.stu import STU
    from flash_stu.modules.swiglu import MLP
    _, _, model = make_pair(seed=5, init="healthy", dtype=torch.bfloat16, mlp_scale=2, n_embd=128, n_layers=4, n_heads=2,
                            window_size=8, num_eigh=8, seq_len=64, vocab_size=777)
    ids = prompt(2, 7, 777, 1).cuda()
    past = model(ids[:, :6], use_cache=True).past_key_values
    calls = []

    def counted(f):
        def g(*a, **k):
            calls.append(1)
            return f(*a, **k)
        return g
    layer = model.layers[0]
    if what == "instance":
        monkeypatch.setattr(layer.mlp_norm, "add_then_norm", counted(layer.mlp_norm.add_then_norm))
    elif what == "model":
        monkeypatch.setattr(model, "_head", counted(model._head))
    elif what == "subclass":
        class Other(FlashSTU):
            _run_layers = counted(FlashSTU._run_layers)
        model.__class__ = Other
    else:
        cls, name = what.split(".")
        cls = {"MLP": MLP, "RMSNorm": RMSNorm, "STU": STU}[cls]
        monkeypatch.setattr(cls, name, counted(getattr(cls, name)))
    model(ids[:, 6:7], past_key_values=past, use_cache=True)
    assert len(calls) == {"MLP.forward": 4, "RMSNorm.add_then_norm": 4, "STU._step": 2}.get(what, 1)


def test_derived_tensors_are_complete_on_every_stream():
    """Transposed weights and filter spectra that one stream has only just been given, read by the next call on another: the
    values of a model that nothing else runs beside.  A module that has been called can still be copied and pickled."""
    import copy
    import pickle
    from flash_stu import STU, FlashSTUConfig
    cfg = FlashSTUConfig(n_embd=256, n_heads=4, n_layers=2, seq_len=512, num_eigh=8, vocab_size=64, torch_dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(2)
    phi, x = torch.randn(512, 8, generator=g).bfloat16(), torch.randn(2, 300, 256, generator=g).bfloat16().cuda()
    stu = STU(cfg, phi, 1024).cuda()
    other, big = torch.cuda.Stream(), torch.randn(4096, 4096, device="cuda")
    default = torch.cuda.current_stream()
    for first, second in ((other, default), (default, other)) * 2:
        with torch.no_grad():
            for p in stu.parameters():
                p.copy_(torch.randn(p.shape, generator=g))
        fresh = STU(cfg, phi, 1024).cuda()
        fresh.load_state_dict(stu.state_dict())
        want = fresh(x)
        torch.cuda.synchronize()
        with torch.cuda.stream(first):
            for _ in range(8):                  # some milliseconds in front of the copies
                big @ big
            there = stu(x)
        with torch.cuda.stream(second):
            here = stu(x)
            assert torch.equal(here, want)
        torch.cuda.synchronize()
        assert torch.equal(there, want)
        assert torch.equal(stu(x), want) and stu._derived["mit"][4] == {other.cuda_stream, default.cuda_stream}
    for copied in (copy.deepcopy(stu), pickle.loads(pickle.dumps(stu))):
        assert torch.equal(copied(x), want)


def test_derived_tensors_outlive_what_other_streams_read():
    """Spectra that another stream has still to read while a call of another length replaces them, and memory of their size that
    the stream that made them asks for then and fills."""
    from flash_stu import STU, FlashSTUConfig
    cfg = FlashSTUConfig(n_embd=256, n_heads=4, n_layers=2, seq_len=1024, num_eigh=8, vocab_size=64, torch_dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(2)
    phi = torch.randn(1024, 8, generator=g).bfloat16()
    x, longer = (torch.randn(2, T, 256, generator=g).bfloat16().cuda() for T in (300, 700))
    stu = STU(cfg, phi, 2048).cuda()
    with torch.no_grad():
        for p in stu.parameters():
            p.copy_(torch.randn(p.shape, generator=g))
    stu(longer)
    other, big = torch.cuda.Stream(), torch.randn(4096, 4096, device="cuda")
    want = stu(x)
    spec = stu._derived["spec"][1]
    shape, at = spec.shape, spec.data_ptr()
    del spec
    torch.cuda.synchronize()
    with torch.cuda.stream(other):
        for _ in range(8):
            big @ big
        there = stu(x)
    stu(longer)
    assert stu._derived["spec"][1].shape != shape
    fills = [torch.full(shape, 7.0, device="cuda") for _ in range(3)]
    assert at not in [t.data_ptr() for t in fills]
    torch.cuda.synchronize()
    assert torch.equal(there, want)


@pytest.mark.parametrize("T,d", [(2049, 512), (3000, 768), (4096, 1024), (2100, 1536), (4096, 2048), (300, 256)])
def test_operator_rows_and_graphs_do_not_depend_on_the_rows_of_other_calls(T, d):
    """A row of the operator has the bits that it has alone, and a graph captured for one row still gives them after calls of
    other numbers of rows and other memory filled."""
    from flash_stu import STU, FlashSTUConfig
    cfg = FlashSTUConfig(n_embd=d, n_heads=d // 64, n_layers=2, seq_len=4096, num_eigh=8, vocab_size=64, torch_dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(T)
    stu = STU(cfg, (torch.randn(4096, 8, generator=g) / 64).bfloat16(), 8192).cuda()
    with torch.no_grad():
        for p in stu.parameters():
            p.copy_(torch.randn(p.shape, generator=g) * d ** -0.5)
    xp = torch.randn(5, T, d, generator=g).bfloat16().cuda()
    one = xp[:1].clone()
    with torch.no_grad():
        want = [stu._convolve(xp[b:b + 1].contiguous()) for b in range(5)]
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = stu._convolve(one)
        for rows in (2, 3, 5):
            assert torch.equal(stu._convolve(xp[:rows].contiguous()), torch.cat(want[:rows]))
            fills = [torch.full((d, n), 7.0, device="cuda") for n in (2064 * 2, 4096, 8192 * 2)]
            one.copy_(xp[rows - 1:rows])
            graph.replay()
            assert torch.equal(y, want[rows - 1])
            del fills


@pytest.mark.parametrize("T", [64, 700, 4096])
def test_fp32_filters_beside_bf16_inputs(T):
    """Filters and their projection kept in fp32, inputs and M_inputs in bf16: the convolution against float64 sums of the same
    operands, fp32 transforms (1e-6 of the largest sum is five times their error) and each branch and the sum of both rounded once."""
    from flash_stu import STU, FlashSTUConfig
    cfg = FlashSTUConfig(n_embd=2048, n_heads=32, n_layers=2, seq_len=4096, num_eigh=8, vocab_size=64, torch_dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(T)
    stu = STU(cfg, (torch.randn(4096, 8, generator=g) / 64).bfloat16(), 8192).cuda()
    with torch.no_grad():
        for p in stu.parameters():
            p.copy_(torch.randn(p.shape, generator=g) * 2048 ** -0.5)
    stu.phi, stu.M_filters.data = stu.phi.float(), stu.M_filters.data.float()
    x = torch.randn(1, T, 2048, generator=g).bfloat16().cuda()
    y = stu(x).double()
    xp, f = stu._project(x).double(), stu.effective_filter().double()
    n, sgn = 2 * T, (-1.0) ** torch.arange(T, device="cuda", dtype=torch.float64)[:, None]
    plus, minus = (torch.fft.irfft(torch.fft.rfft(xp, n, 1) * torch.fft.rfft(v, n, 0), n, 1)[:, :T] for v in (f[:T], f[:T] * sgn))
    bound = 2.0 ** -8 * (plus.abs() + minus.abs() + (plus + minus).abs()) + 1e-6 * float(plus.abs().max())
    assert bool(((y - plus - minus).abs() <= bound).all())


@pytest.mark.parametrize("dtype,T", [(torch.bfloat16, 300), (torch.float32, 20), (torch.float32, 100)])
def test_tensors_derived_under_capture_stay_in_the_graph(dtype, T, monkeypatch):
    """The first call on new weights inside a capture: calls beside the graph do not read what only its replay writes, and
    replays, with other work between them, give the values of an uncaptured module on each input."""
    from flash_stu import STU, FlashSTUConfig, _hip
    cfg = FlashSTUConfig(n_embd=256, n_heads=4, n_layers=2, seq_len=512, num_eigh=8, vocab_size=64, torch_dtype=dtype)
    g = torch.Generator().manual_seed(3)
    phi = torch.randn(512, 8, generator=g).to(dtype)
    new, reference = STU(cfg, phi, 1024).cuda(), STU(cfg, phi, 1024).cuda()
    with torch.no_grad():
        for p in new.parameters():
            p.copy_(torch.randn(p.shape, generator=g))
    reference.load_state_dict(new.state_dict())
    x, others = torch.randn(2, T, 256, generator=g).to(dtype).cuda(), torch.randn(3, 2, T, 256, generator=g).to(dtype).cuda()
    want = [reference(t) for t in (x, *others)]         # (also the kernels' one-time set-up)
    torch.cuda.synchronize()
    monkeypatch.setattr(_hip, "_twiddle_cache", {})
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = new(x)
    assert not new._derived and not _hip._twiddle_cache
    assert torch.equal(new(x), want[0])
    for t, w in zip(others, want[1:]):
        x.copy_(t)
        graph.replay()
        assert torch.equal(y, w)
        assert torch.equal(new(t), w)


@pytest.mark.parametrize("d,rows", [(256, 3), (256, 20), (128, 20)])
def test_generate_under_inference_mode(d, rows):
    """torch.inference_mode() around the first call, and calls outside after it: the tokens of a call under no_grad, and those of
    changed weights after a change."""
    kw = dict(seed=5, init="healthy", dtype=torch.bfloat16, mlp_scale=2, n_embd=d, n_layers=4, n_heads=2, window_size=8,
              num_eigh=8, seq_len=64, vocab_size=777)
    ids = prompt(rows, 6, 777, rows).cuda()
    _, _, model = make_pair(**kw)
    _, _, other = make_pair(**kw)
    run = lambda m: m.generate(ids, max_length=16, do_sample=False)
    with torch.inference_mode():
        first = run(model)
    assert torch.equal(first, run(other)) and torch.equal(first, run(model))
    with torch.no_grad():
        for m in (model, other):
            for p in m.parameters():
                p.mul_(0.75)
    with torch.inference_mode():
        second = run(model)
    assert torch.equal(second, run(other)) and torch.equal(second, run(model))


def test_models_that_have_generated_can_be_copied():
    """deepcopy and pickle of a model with an engine: the copy generates the same tokens and follows its own weights."""
    import copy
    import pickle
    _, _, model = make_pair(seed=5, init="healthy", dtype=torch.bfloat16, mlp_scale=2, n_embd=256, n_layers=4, n_heads=2,
                            window_size=8, num_eigh=8, seq_len=64, vocab_size=777)
    ids = prompt(2, 6, 777, 1).cuda()
    want = model.generate(ids, max_length=16, do_sample=False)
    for other in (copy.deepcopy(model), pickle.loads(pickle.dumps(model))):
        assert torch.equal(other.generate(ids, max_length=16, do_sample=False), want)
        assert other.tok_emb.weight is other.lm_head.weight
        with torch.no_grad():
            for p in other.parameters():
                p.zero_()
        assert torch.equal(model.generate(ids, max_length=16, do_sample=False), want)


@pytest.mark.parametrize("dtype,extra", [(torch.float32, {}), (torch.bfloat16, {}), (torch.bfloat16, dict(use_hankel_L=True)),
                                         (torch.float32, dict(use_hankel_L=True))])
def test_steps_on_caches_of_more_rows_than_one_launch_takes(dtype, extra):
    """forward() with caches for 37 rows (three launches of the skinny projection, one of each state operator) against the same
    rows in groups of 16, whose sums are formed in another order: bounds as in the test of the one-call step."""
    _, _, model = make_pair(seed=5, init="healthy", dtype=dtype, mlp_scale=2, n_embd=128, n_layers=4, n_heads=2, window_size=8,
                            num_eigh=8, seq_len=64, vocab_size=777, **extra)
    ids = prompt(37, 10, 777, 3).cuda()

    def run(rows):
        past, logits = model(rows[:, :6], use_cache=True).past_key_values, []
        for t in range(6, 10):
            out = model(rows[:, t:t + 1], past_key_values=past, use_cache=True)
            past = out.past_key_values
            logits.append(out.logits.float())
        return torch.cat(logits, 1)
    got, want = run(ids), torch.cat([run(ids[b:b + 16]) for b in range(0, 37, 16)])
    assert float((got - want).abs().max()) <= (1e-4 if dtype == torch.float32 else 2e-2) * float(want.abs().max())


@pytest.mark.parametrize("dtype", [torch.int32, torch.float32, torch.float64])
def test_steps_on_caches_whose_positions_were_cast(dtype):
    """Caches that a program has cast as a whole still step, through the one call."""
    from flash_stu.engine import step_on_caches
    _, _, model = make_pair(seed=5, init="healthy", dtype=torch.float32, mlp_scale=2, n_embd=64, n_layers=2, n_heads=1, window_size=8,
                            num_eigh=8, seq_len=64, vocab_size=77)
    ids = prompt(2, 8, 77, 3).cuda()
    past = model(ids[:, :6], use_cache=True).past_key_values
    cast = [(a.clone(), b.clone(), p.to(dtype)) for a, b, p in past]
    for t in (6, 7):
        want = model(ids[:, t:t + 1], past_key_values=past, use_cache=True)
        past = want.past_key_values
        logits, cast = step_on_caches(model, ids[:, t:t + 1], cast)
        assert torch.equal(logits, want.logits)


def _takes_one_call(model, ids, past) -> bool:
    """Whether a step on these caches is the one call (made on copies of them)."""
    from flash_stu.engine import step_on_caches
    return step_on_caches(model, ids, tuple(tuple(t.clone() for t in c) for c in past)) is not None


@pytest.mark.parametrize("d,scale,rows,mode", [(256, 2, 1, "lds"), (256, 4, 16, "lds"), (512, 4, 3, "lds"), (768, 2, 10, "lds"), (768, 12, 11, "lds"),
                                               (1024, 4, 8, "lds"), (1024, 3, 9, "lds"), (2048, 2, 4, "lds"), (2048, 4, 5, "lds"), (512, 2, 4, "history")])
def test_one_call_step_on_the_parameters_themselves(d, scale, rows, mode):
    """The step on caches reads row-major weights in the launches that generate() runs over packed copies: every width those take,
    with the norms merged (rows * d up to 8192, feature counts of 512) and beside them, against the layers' own calls.  Sums of the
    same products in other orders: the bounds of the one-call step's other tests."""
    _, _, model = make_pair(seed=5, init="healthy", dtype=torch.bfloat16, mlp_scale=scale, n_embd=d, n_layers=4, n_heads=d // 64, window_size=8,
                            num_eigh=8, seq_len=64, vocab_size=777, stu_decode_mode=mode)
    ids = prompt(rows, 10, 777, 3).cuda()

    def run(one_call):
        past, logits = model(ids[:, :6], use_cache=True).past_key_values, []
        assert _takes_one_call(model, ids[:, 6:7], past) == one_call
        for t in range(6, 10):
            out = model(ids[:, t:t + 1], past_key_values=past, use_cache=True)
            past = out.past_key_values
            logits.append(out.logits.float())
        return torch.cat(logits, 1)
    got = run(True)
    model.layers[0].mlp.register_forward_hook(lambda *a: None)     # the layers' own calls run
    want = run(False)
    assert float((got - want).abs().max()) <= 2e-2 * float(want.abs().max())


@pytest.mark.parametrize("d,rows,extra", [(64, 1, {}), (64, 5, {}), (192, 2, dict(stu_decode_mode="lds")), (256, 2, {}), (288, 1, dict(use_hankel_L=True)),
                                          (320, 3, {}), (512, 2, dict(stu_decode_mode="lds")), (512, 1, {}), (544, 2, {})])
def test_fp32_step_with_its_norms_in_the_projections(d, rows, extra):
    """One and two fp32 rows of up to 512 features: the projections normalise the stream themselves (544 features and more rows keep
    the launches of their own), histories of 1 to 16 slices, against the layers' own calls: the bounds of the fp32 step."""
    _, _, model = make_pair(seed=5, init="healthy", dtype=torch.float32, mlp_scale=3, n_embd=d, n_layers=4, n_heads=d // 32, window_size=8,
                            num_eigh=8, seq_len=320, vocab_size=777, **extra)
    ids = prompt(rows, 300, 777, 3).cuda()

    def run(first, count, one_call):
        past, logits = model(ids[:, :first], use_cache=True).past_key_values, []
        assert _takes_one_call(model, ids[:, first:first + 1], past) == one_call
        for t in range(first, first + count):
            out = model(ids[:, t:t + 1], past_key_values=past, use_cache=True)
            past = out.past_key_values
            logits.append(out.logits)
        return torch.cat(logits, 1)
    got = [run(3, 3, True), run(70, 2, True), run(290, 2, True)]
    model.layers[0].mlp.register_forward_hook(lambda *a: None)     # the layers' own calls run
    for a, b in zip(got, [run(3, 3, False), run(70, 2, False), run(290, 2, False)]):
        assert float((a - b).abs().max()) <= 1e-4 * float(b.abs().max())


def test_forward_accepts_reference_style_kv_cache():
    from flash_stu import Attention, FlashSTUConfig
    cfg = FlashSTUConfig(n_embd=128, n_heads=2, n_layers=2, seq_len=64, window_size=6, vocab_size=11, mlp_scale=2,
                         torch_dtype=torch.float32)
    torch.manual_seed(0)
    att = Attention(cfg).cuda()
    torch.nn.init.normal_(att.c_attn.weight, std=0.05)
    torch.nn.init.normal_(att.c_proj.weight, std=0.05)
    x = torch.randn(2, 15, 128, device="cuda")
    p = {"c_attn.weight": att.c_attn.weight.detach().cpu(), "c_proj.weight": att.c_proj.weight.detach().cpu()}
    ref, (k, v) = O.attention_forward(x.cpu(), p, 2, 6, 50.0)
    y_full = att(x, use_cache=False)
    assert float((y_full.cpu() - ref).abs().max()) < 1e-5
    # growing (B,t,H,hd) cache as the reference returns it -> converted to a ring
    y, cache = att(x[:, 14:15], past_key_value=(k[:, :14].cuda(), v[:, :14].cuda()), use_cache=True)
    assert float((y.cpu() - ref[:, 14:15]).abs().max()) < 1e-5
    assert len(cache) == 3 and cache[0].shape == (2, 2, 7, 64)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("use_attention", [False, True])
def test_block_forward_and_cache(dtype, use_attention):
    from flash_stu import FlashSTUBlock
    torch.manual_seed(0)
    blk = FlashSTUBlock(d_model=128, sequence_length=64, num_filters=8, use_attention=use_attention,
                        torch_dtype=dtype, stu_decode_mode="history")
    assert blk.config.mlp_scale == 4 and blk.config.n_heads == 2 and blk.config.window_size == 16
    assert blk.is_attention_block == use_attention
    for p in blk.parameters():
        torch.nn.init.normal_(p, std=0.05) if p.dim() > 1 else torch.nn.init.ones_(p)
    blk = blk.cuda()
    ocfg = O.OracleConfig(n_embd=128, n_heads=2, n_layers=1, seq_len=64, window_size=16, vocab_size=1, mlp_scale=4,
                          num_eigh=8, dtype=dtype)
    lw = {k[len("layer."):]: v.detach().cpu() for k, v in blk.state_dict().items() if k.startswith("layer.")}
    x = torch.randn(2, 20, 128).to(dtype)
    if use_attention:
        ref, _ = O.attention_layer_forward(x.clone(), lw, ocfg)
    else:
        ref = O.stu_layer_forward(x.clone(), lw, ocfg, blk.phi.cpu())
    tol = 1e-4 if dtype == torch.float32 else 4e-2
    scale = float(ref.float().abs().max())
    y = blk(x.cuda().clone())
    assert float((y.float().cpu() - ref.float()).abs().max()) <= tol * scale
    # prefill 12 positions with cache, then step
    y0, cache = blk(x[:, :12].cuda().clone(), use_cache=True)
    for t in range(12, 20):
        yt, cache = blk(x[:, t:t + 1].cuda().clone(), past_key_value=cache, use_cache=True)
        assert float((yt[:, 0].float().cpu() - ref[:, t].float()).abs().max()) <= tol * scale


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_exact_mode_stu_forward(dtype):
    """use_approx=False: filter-bank convolution + K*d*d contraction (config 3's operator, small)."""
    from flash_stu import STU, FlashSTUConfig
    cfg = FlashSTUConfig(n_embd=64, n_heads=1, n_layers=1, seq_len=128, num_eigh=8, use_approx=False,
                         torch_dtype=dtype, vocab_size=3)
    phi = O.get_spectral_filters(128, 8, dtype=dtype)
    torch.manual_seed(0)
    stu = STU(cfg, phi, 256)
    torch.nn.init.normal_(stu.M_phi_plus, std=0.05)
    torch.nn.init.normal_(stu.M_phi_minus, std=0.05)
    x = torch.randn(2, 100, 64).to(dtype)
    p = {"M_phi_plus": stu.M_phi_plus.detach().clone(), "M_phi_minus": stu.M_phi_minus.detach().clone()}
    ref = O.stu_forward(x, phi, p, 256, use_approx=False)
    y = stu.cuda()(x.cuda())
    tol = 1e-4 if dtype == torch.float32 else 3e-2
    assert float((y.float().cpu() - ref.float()).abs().max()) <= tol * float(ref.float().abs().max())


def test_save_and_load_pretrained_roundtrip(tmp_path):
    from flash_stu import FlashSTU
    ocfg, w, model = make_pair(seed=6, init="healthy", mlp_scale=2, n_embd=128, n_layers=2, n_heads=2, window_size=8,
                               num_eigh=8, seq_len=64, vocab_size=301)
    model.save_pretrained(str(tmp_path))
    again = FlashSTU.from_pretrained(str(tmp_path)).cuda().eval()
    assert again.tok_emb.weight is again.lm_head.weight
    ids = prompt(1, 9, 301, 7).cuda()
    assert torch.equal(model.generate(ids, max_length=30, do_sample=False),
                       again.generate(ids, max_length=30, do_sample=False))
    assert again.get_num_params() == model.get_num_params()


# ----------------------------------------------------------------- variants beyond the default configuration
def _variant_pair(seed, dtype=torch.float32, **kw):
    """Model with the given config variant + oracle-side restatement driven by the same state dict."""
    from flash_stu import FlashSTU, FlashSTUConfig
    base = dict(n_embd=128, n_layers=2, n_heads=2, window_size=16, num_eigh=8, seq_len=64, vocab_size=211,
                mlp_scale=2, torch_dtype=dtype, use_attn=True)
    base.update(kw)
    torch.manual_seed(seed)
    model = FlashSTU(FlashSTUConfig(**base))
    with torch.no_grad():
        for n_, p_ in model.named_parameters():
            if n_.endswith(".bias"):
                p_.copy_((0.1 * torch.randn(p_.shape)).to(dtype))
            elif "M_inputs" in n_ or "M_filters" in n_:
                p_.mul_(4.0)
    return model


def _ref_layer0_stu_sandwich(model, x):
    """Oracle-side restatement of stu_layer.py:78-97 with the sandwich, from the oracle's own pieces."""
    L = model.layers[0]
    sd = {k: v.detach().cpu() for k, v in L.state_dict().items()}
    cfg = model.config
    h = O.rms_norm(x, sd["stu_norm.weight"], cfg.rms_norm_eps)
    h = torch.nn.functional.linear(h, sd["stu_mlp_in_proj.weight"], sd.get("stu_mlp_in_proj.bias"))
    h = torch.nn.functional.silu(h)
    phi = model.phi.detach().cpu()
    h = O.stu_forward(h, phi, {"M_inputs": sd["stu.M_inputs"], "M_filters": sd["stu.M_filters"]}, model.n)
    h = torch.nn.functional.linear(h, sd["stu_mlp_out_proj.weight"], sd.get("stu_mlp_out_proj.bias"))
    x = x + h
    h2 = O.rms_norm(x, sd["mlp_norm.weight"], cfg.rms_norm_eps)
    g = torch.nn.functional.gelu(torch.nn.functional.linear(h2, sd["mlp.gate_proj.weight"], sd.get("mlp.gate_proj.bias")),
                                 approximate="tanh")
    u = torch.nn.functional.linear(h2, sd["mlp.up_proj.weight"], sd.get("mlp.up_proj.bias"))
    return x + torch.nn.functional.linear(g * u, sd["mlp.down_proj.weight"], sd.get("mlp.down_proj.bias"))


@pytest.mark.parametrize("bias", [False, True])
def test_stu_sandwich_layer_matches_restatement(bias):
    """stu_enable_mlp_sandwich (+ bias=True): the STU layer against the oracle's pieces, fp32."""
    model = _variant_pair(11, stu_enable_mlp_sandwich=True, stu_mlp_hidden_size=192, bias=bias)
    x = torch.randn(2, 40, 128, generator=torch.Generator().manual_seed(3))
    ref = _ref_layer0_stu_sandwich(model, x.clone())
    got = model.cuda().layers[0](x.cuda().clone()).cpu()
    assert float((got - ref).abs().max()) <= 2e-4 * float(ref.abs().max())


def test_sandwich_and_bias_generate_stateful_equals_recompute():
    """generate() of a variant the one-call step does not cover: the per-layer state loop returns the same ids
    as re-running the whole sequence every step."""
    model = _variant_pair(12, stu_enable_mlp_sandwich=True, stu_mlp_hidden_size=192, bias=True).cuda()
    ids = torch.randint(0, 211, (3, 9), generator=torch.Generator().manual_seed(5)).cuda()
    a = model.generate(ids, max_length=30, do_sample=False, use_cache=True)
    b = model.generate(ids, max_length=30, do_sample=False, use_cache=False)
    assert torch.equal(a, b)


def test_channel_tiling_is_the_block_diagonal_projection():
    """d_in_tile/d_out_tile (stu.py:123-191): per tile x[..., i:e] @ M_inputs[i:e, i:e] and the tile's filters,
    restated with the oracle's convolution tile by tile; decode through the engine matches recompute."""
    model = _variant_pair(13, d_in_tile=32, d_out_tile=32)
    stu = model.layers[0].stu
    x = torch.randn(2, 48, 128, generator=torch.Generator().manual_seed(4))
    phi = model.phi.detach().cpu()
    Mi, Mf = stu.M_inputs.detach().cpu(), stu.M_filters.detach().cpu()
    parts = []
    for i in range(0, 128, 32):
        plus, minus = O.convolve(x[..., i:i + 32] @ Mi[i:i + 32, i:i + 32], phi @ Mf[:, i:i + 32], model.n)
        parts.append(plus + minus)
    ref = torch.cat(parts, -1)
    model = model.cuda()
    got = model.layers[0].stu(x.cuda()).cpu()
    assert float((got - ref).abs().max()) <= 2e-5 * float(ref.abs().max())
    ids = torch.randint(0, 211, (2, 7), generator=torch.Generator().manual_seed(6)).cuda()
    assert torch.equal(model.generate(ids, max_length=24, do_sample=False),
                       model.generate(ids, max_length=24, do_sample=False, use_cache=False))


def test_all_stu_stack_and_exact_mode_generate():
    """use_attn=False (model.py:83-87) and use_approx=False decode: stateful loop == full recompute."""
    for kw in (dict(use_attn=False), dict(use_approx=False, n_embd=64, n_heads=2)):
        model = _variant_pair(14, **kw).cuda()
        ids = torch.randint(0, 211, (2, 6), generator=torch.Generator().manual_seed(7)).cuda()
        a = model.generate(ids, max_length=20, do_sample=False, use_cache=True)
        b = model.generate(ids, max_length=20, do_sample=False, use_cache=False)
        assert torch.equal(a, b), kw


def test_checkpoint_formats(tmp_path):
    """save_pretrained directory, a sharded directory with an index, and a bare training-style
    model_<step>.safetensors (training/distributed.py:140-148) all load to the same logits."""
    import json
    from safetensors.torch import save_file
    from flash_stu import FlashSTU
    model = _variant_pair(15).cuda()
    ids = torch.randint(0, 211, (2, 12), generator=torch.Generator().manual_seed(8)).cuda()
    ref = model(ids).logits
    d1 = tmp_path / "hf"
    model.save_pretrained(str(d1))
    assert torch.equal(FlashSTU.from_pretrained(str(d1)).cuda()(ids).logits, ref)
    # sharded: split the state dict over two files + index
    sd = {k: v.detach().cpu().contiguous() for k, v in model.state_dict().items() if k != "lm_head.weight"}
    keys = sorted(sd)
    d2 = tmp_path / "sharded"
    d2.mkdir()
    model.config.save_pretrained(str(d2))
    half = len(keys) // 2
    save_file({k: sd[k] for k in keys[:half]}, str(d2 / "model-00001-of-00002.safetensors"))
    save_file({k: sd[k] for k in keys[half:]}, str(d2 / "model-00002-of-00002.safetensors"))
    wm = {k: ("model-00001-of-00002.safetensors" if i < half else "model-00002-of-00002.safetensors") for i, k in enumerate(keys)}
    (d2 / "model.safetensors.index.json").write_text(json.dumps({"metadata": {}, "weight_map": wm}))
    assert torch.equal(FlashSTU.from_pretrained(str(d2)).cuda()(ids).logits, ref)
    # training checkpoint: one file, DDP-style prefix, config passed in
    f3 = tmp_path / "model_00100.safetensors"
    save_file({"module." + k: v for k, v in sd.items()}, str(f3))
    assert torch.equal(FlashSTU.from_pretrained(str(f3), config=model.config).cuda()(ids).logits, ref)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_exact_mode_decode_on_the_recurrence_state(dtype):
    """use_approx=False with stu_decode_mode='lds': one decode step per token on the bank state gives the logits of
    a full recompute to the fit's accuracy (fp32) / within the bf16 tolerance, and mostly the same greedy ids."""
    model = _variant_pair(16, dtype=dtype, use_approx=False, n_embd=64, n_heads=2, stu_decode_mode="lds").cuda()
    assert model.layers[0].stu._exact_lds_ok()
    ids = torch.randint(0, 211, (3, 10), generator=torch.Generator().manual_seed(9)).cuda()
    out = model(ids[:, :6], use_cache=True)
    past = out.past_key_values
    worst = 0.0
    for t in range(6, 10):
        step = model(ids[:, t:t + 1], past_key_values=past, use_cache=True)
        past = step.past_key_values
        full = model(ids[:, :t + 1]).logits[:, -1]
        rel = float((step.logits[:, -1].float() - full.float()).abs().max() / full.float().abs().max())
        worst = max(worst, rel)
    assert worst <= (2e-3 if dtype == torch.float32 else 2e-2), worst


