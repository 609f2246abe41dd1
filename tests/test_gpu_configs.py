"""BASELINE configs 3, 4 and 5 on the GPU: parity against the CPU oracle at sizes
the oracle finishes in seconds, plus size-independent properties at the full
BASELINE sizes (linearity, causality, delta response, state carry)."""
import functools
import math

import pytest
import torch

from oracle import flashstu_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from flash_stu import _hip
    _hip.load()
    return _hip


# ----------------------------------------------------------------- config 3
@functools.lru_cache(maxsize=4)
def _filters(L, K, dtype):
    """The Hankel filters, computed once per test session (the L=8192 eigendecomposition takes a while)."""
    return O.get_spectral_filters(L, K, dtype=dtype)


def _exact_stu(dtype, d, L, K, seed):
    from flash_stu import STU, FlashSTUConfig
    cfg = FlashSTUConfig(n_embd=d, n_heads=1, n_layers=1, seq_len=L, num_eigh=K, use_approx=False, torch_dtype=dtype,
                         vocab_size=3)
    phi = _filters(L, K, dtype)
    g = torch.Generator().manual_seed(seed)
    stu = STU(cfg, phi, O.nearest_power_of_two(2 * L - 1, True))
    with torch.no_grad():
        stu.M_phi_plus.copy_((torch.randn(K, d, d, generator=g) / math.sqrt(d)).to(dtype))
        stu.M_phi_minus.copy_((torch.randn(K, d, d, generator=g) / math.sqrt(d)).to(dtype))
    p = {"M_phi_plus": stu.M_phi_plus.detach().clone(), "M_phi_minus": stu.M_phi_minus.detach().clone()}
    return stu.cuda(), phi, p


@pytest.mark.parametrize("dtype,B,T,d", [(torch.bfloat16, 1, 4096, 256), (torch.bfloat16, 2, 2300, 128), (torch.float32, 1, 2304, 64)])
def test_stu_forward_of_a_few_long_sequences_goes_time_major(dtype, B, T, d):
    """Approx-mode STU.forward on a few long sequences (the shape class of the reference's own benchmark,
    tests/benchmark_tilling.py:157-165): without a cache the projected inputs are formed as time-major slabs by the
    prompt GEMM with swapped operands and convolved as such; with a cache they are transposed in front of the same
    convolution.  Both give the oracle's values, and the same bits as each other where the GEMM is the same."""
    from flash_stu import STU, FlashSTUConfig
    L, K = 4096, 8
    cfg = FlashSTUConfig(n_embd=d, n_heads=1, n_layers=1, seq_len=L, num_eigh=K, use_approx=True, torch_dtype=dtype,
                         vocab_size=3, stu_decode_mode="lds")
    phi = _filters(L, K, dtype)
    g = torch.Generator().manual_seed(11)
    stu = STU(cfg, phi, O.nearest_power_of_two(2 * L - 1, True))
    with torch.no_grad():
        stu.M_inputs.copy_((torch.randn(d, d, generator=g) / math.sqrt(d)).to(dtype))
        stu.M_filters.copy_((torch.randn(K, d, generator=g) / math.sqrt(K)).to(dtype))
    p = {"M_inputs": stu.M_inputs.detach().clone(), "M_filters": stu.M_filters.detach().clone()}
    stu = stu.cuda()
    x = torch.randn(B, T, d, generator=g).to(dtype)
    assert stu._few_long_sequences(B, T, d, x.element_size())
    y = stu(x.cuda())
    y2, _ = stu(x.cuda(), use_cache=True)
    ref = O.stu_forward(x, phi, p, 8192, use_approx=True).float()
    scale = float(ref.abs().max())
    for out in (y, y2):
        err = (out.float().cpu() - ref).abs()
        if dtype == torch.float32:
            assert float(err.max()) <= 2e-4 * scale
        else:
            assert float(err.max()) <= 3e-2 * scale and float(err.mean()) <= 3e-3 * scale
    assert float((y != y2).float().mean()) <= (0.0 if dtype == torch.float32 else 0.02)


@pytest.mark.parametrize("B,T,d", [(5, 2052, 96), (3, 4092, 160), (9, 2500, 128)])
def test_stu_forward_of_several_long_sequences_in_one_product(B, T, d):
    """Rows of the batch that lie next to each other in a channel's slab, of lengths that are no whole tile, to the same bounds."""
    test_stu_forward_of_a_few_long_sequences_goes_time_major(torch.bfloat16, B, T, d)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [200, 384, 20])
def test_c3_exact_mode_ragged_lengths_and_both_dtypes(dtype, T):
    """The exact-mode operator on sequences shorter than the filters and not a multiple of the contraction's
    128-position tiles (the slabs are padded to whole tiles and the padding's rows cut off again), in bf16 (matrix-core
    contraction over the time-major slabs) and fp32 (the general kernel on the slab as a strided operand), and below
    the shortest transform (time-domain filter bank, row-major U): all against the oracle on the same inputs."""
    stu, phi, p = _exact_stu(dtype, 64, 512, 8, 7)
    x = torch.randn(3, T, 64, generator=torch.Generator().manual_seed(8)).to(dtype)
    ref = O.stu_forward(x, phi, p, 1024, use_approx=False).float()
    y = stu(x.cuda()).float().cpu()
    assert y.shape == ref.shape and bool(torch.isfinite(y).all())
    scale = float(ref.abs().max())
    if dtype == torch.float32:
        assert float((y - ref).abs().max()) <= 2e-4 * scale
    else:
        assert float((y - ref).abs().max()) <= 3e-2 * scale
        assert float((y - ref).abs().mean()) <= 3e-3 * scale


def test_c3_exact_mode_prefill_parity_reduced():
    """Config 3's operator (use_approx=False, K=24, M_phi ~ N(0,1/sqrt(d))) at B=2, L=1024, d=128, bf16."""
    dtype = torch.bfloat16
    stu, phi, p = _exact_stu(dtype, 128, 1024, 24, 0)
    x = torch.randn(2, 1024, 128, generator=torch.Generator().manual_seed(1)).to(dtype)
    ref = O.stu_forward(x, phi, p, 2048, use_approx=False).float()
    y = stu(x.cuda()).float().cpu()
    scale = float(ref.abs().max())
    assert float((y - ref).abs().max()) <= 3e-2 * scale
    assert float((y - ref).abs().mean()) <= 3e-3 * scale


def test_c3_full_size_properties(hip):
    """B=4, L=8192, d=1024, K=24, bf16: the filter-bank kernel at the BASELINE shape.
    delta input returns the filters; the response is causal and shift-invariant; fp32 results
    are linear in the input."""
    B, L, d, K = 4, 8192, 1024, 24
    dtype = torch.bfloat16
    phi = _filters(L, K, dtype).cuda()
    x = torch.zeros(B, L, d, dtype=dtype, device="cuda")
    x[0, 0, :] = 1.0                      # delta at t=0
    x[1, 100, 5] = 2.0                    # delayed, scaled delta in one channel
    x[2] = torch.randn(L, d, generator=torch.Generator().manual_seed(2)).to(dtype).cuda()
    x[3, 4000:] = x[2, : L - 4000]        # batch 3 = batch 2 shifted by 4000
    Up = torch.empty(B, L, K, d, dtype=dtype, device="cuda")
    Um = torch.empty_like(Up)
    hip.stu_conv_bank(x, phi, Up, Um)
    torch.cuda.synchronize()
    sg = torch.ones(L, 1, device="cuda")
    sg[1::2] = -1
    assert torch.equal(Up[0, :, :, 7], phi)                                   # delta -> filter (exact in bf16)
    assert torch.equal(Um[0, :, :, 3].float(), (phi.float() * sg))
    assert float(Up[1, :100].abs().max()) == 0.0                               # causal
    assert torch.equal(Up[1, 100:, :, 5].float(), (2 * phi[: L - 100].float()).to(dtype).float())
    assert float(Up[1, :, :, 6].abs().max()) == 0.0                            # channels do not mix
    assert torch.equal(Up[3, 4000:], Up[2, : L - 4000])                        # shift invariance (same rounding)
    assert float(Up[3, :4000].abs().max()) == 0.0
    # spot-check one (b, t, k, channel) column against a float64 dot product
    t, k, c = 6000, 11, 321
    ref = (phi[: t + 1, k].double().flip(0) * x[2, : t + 1, c].double()).sum()
    assert abs(float(Up[2, t, k, c]) - float(ref)) <= 2.0 ** -7 * abs(float(ref)) + 1e-6


def test_c3_full_size_fft_bank_matches_time_domain(hip):
    """B=4, L=8192, d=1024, K=24, bf16: the FFT bank (transform length 16384, time-major outputs) against the
    time-domain bank kernel on the same input: at most one bf16 ulp apart, on few elements."""
    B, L, d, K = 4, 8192, 1024, 24
    dtype = torch.bfloat16
    phi = _filters(L, K, dtype).cuda()
    x = torch.randn(B, L, d, generator=torch.Generator().manual_seed(5)).to(dtype).cuda()
    Ud = torch.empty(B, L, K, d, dtype=dtype, device="cuda")
    hip.stu_conv_bank(x, phi, Ud, None)
    n = hip.fft_length(L)
    assert n == 16384
    Uf = torch.empty(B, K, d, L, dtype=dtype, device="cuda")
    hip.stu_conv_bank_fft(x, hip.stu_fft_filter(phi, n), Uf.permute(0, 3, 1, 2), None)
    torch.cuda.synchronize()
    for b in range(B):                                   # compare batch by batch to bound the fp32 temporaries
        a, r = Uf[b].permute(2, 0, 1).float(), Ud[b].float()
        diff = (a - r).abs()
        assert bool((diff <= r.abs() * 2.0 ** -7 + 1e-6).all())
        assert float((diff > 0).float().mean()) < 0.02


def test_c3_full_size_exact_mode_delta_response():
    """The whole exact-mode operator at the BASELINE shape (FFT bank + contraction): a unit impulse in channel i
    returns y[t] = T(T(phi[t] @ M+[:, i]) + T((-1)^t phi[t] @ M-[:, i])), and batch rows do not mix."""
    dtype = torch.bfloat16
    d, L, K = 1024, 8192, 24
    stu, phi, p = _exact_stu(dtype, d, L, K, 7)
    x = torch.zeros(4, L, d, dtype=dtype)
    x[1, 0, 17] = 1.0
    x[3, 5, 900] = 1.0
    y = stu(x.cuda()).float().cpu()
    sg = torch.ones(L, 1)
    sg[1::2] = -1
    for b, t0, i in ((1, 0, 17), (3, 5, 900)):
        plus = (phi.float() @ p["M_phi_plus"][:, i, :].float()).to(dtype).float()
        minus = ((phi.float() * sg) @ p["M_phi_minus"][:, i, :].float()).to(dtype).float()
        ref = (plus + minus).to(dtype).float()[: L - t0]
        got = y[b, t0:]
        scale = float(ref.abs().max())
        diff = (got - ref).abs()
        assert float(diff.max()) <= 2.0 ** -6 * scale
        assert float((diff > 0).float().mean()) < 0.05
        if t0:
            assert float(y[b, :t0].abs().max()) <= 1e-3 * scale
    assert float(y[0].abs().max()) == 0.0 and float(y[2].abs().max()) == 0.0


# ----------------------------------------------------------------- config 4
def _c4_tensors(T, Bt=64, d=1024, S=160, seed=3):
    g = torch.Generator().manual_seed(seed)
    A = (0.9 + 0.099 * torch.rand(S, generator=g)).float()
    Bm = (torch.randn(d, S, generator=g) / d).bfloat16()
    Cm = (torch.randn(S, d, generator=g) / S).bfloat16()
    x = torch.randn(T, Bt, d, generator=g).bfloat16()
    return A, Bm, Cm, x


def test_c4_lds_step_parity_at_full_width(hip):
    """Batch 64, d=1024, state 160, A~U(0.9,0.999) fp32, B~N(0,1/d), C~N(0,1/160) bf16, x~N(0,1):
    256 consecutive steps against the oracle's literal loop, state carried across two launches."""
    T = 256
    A, Bm, Cm, x = _c4_tensors(T)
    yref, href = O.lds_sequence(x, A, Bm, Cm)
    h = torch.zeros(64, 160, device="cuda")
    y1 = hip.lds_steps(h, x[:100].cuda(), A.cuda(), Bm.cuda(), Cm.cuda(), check_status=True)
    y2 = hip.lds_steps(h, x[100:].cuda(), A.cuda(), Bm.cuda(), Cm.cuda(), check_status=True)
    y = torch.cat([y1, y2]).float().cpu()
    diff = (y - yref.float()).abs()
    assert float(diff.max()) <= 2.0 ** -7 * float(yref.float().abs().max())
    assert float((diff > 0).float().mean()) < 0.05
    assert float((h.cpu() - href).abs().max()) <= 1e-4 * float(href.abs().max())


def test_c4_4096_steps_state_is_the_closed_form(hip):
    """The full 4096-step run: with a constant input the carried state converges to u/(1-A)
    and two launches of 2048 steps equal one launch of 4096."""
    T = 4096
    A, Bm, Cm, x = _c4_tensors(1)
    xs = x.expand(T, 64, 1024).contiguous().cuda()
    Ad, Bd, Cd = A.cuda(), Bm.cuda(), Cm.cuda()
    h1 = torch.zeros(64, 160, device="cuda")
    y_full = hip.lds_steps(h1, xs, Ad, Bd, Cd, check_status=True)
    h2 = torch.zeros(64, 160, device="cuda")
    ya = hip.lds_steps(h2, xs[:2048], Ad, Bd, Cd, check_status=True)
    yb = hip.lds_steps(h2, xs[2048:], Ad, Bd, Cd, check_status=True)
    torch.cuda.synchronize()
    assert torch.equal(torch.cat([ya, yb]), y_full) and torch.equal(h1, h2)
    u = x[0].float() @ Bm.float()                                   # (64,160)
    closed = u * (1 - A ** T) / (1 - A)
    assert float((h1.cpu() - closed).abs().max()) <= 2e-4 * float(closed.abs().max())
    ylast = (closed @ Cm.float())
    assert float((y_full[-1].float().cpu() - ylast).abs().max()) <= 2.0 ** -6 * float(ylast.abs().max())


# ----------------------------------------------------------------- config 5
def test_c5_shape_sampling_parity_reduced():
    """Config 5's structure (head dim 128, 24 filters, top-k 40 / temperature 0.8, seeded counter stream)
    on a model small enough for the CPU oracle; fp32 so that ids must be identical."""
    from test_gpu_model import make_pair, prompt
    ocfg, w, model = make_pair(seed=2, init="healthy", mlp_scale=2, n_embd=256, n_layers=4, n_heads=2, window_size=24,
                               num_eigh=24, seq_len=256, vocab_size=2003)
    ids = prompt(32, 20, ocfg.vocab_size, 4)          # batch 32 as in config 5: two row chunks of 16
    ref = O.generate(w, ocfg, ids, max_length=52, temperature=0.8, top_k=40, do_sample=True, mode="stateful", seed=2)
    got = model.generate(ids.cuda(), max_length=52, temperature=0.8, top_k=40, do_sample=True, seed=2)
    assert torch.equal(got.cpu(), ref)


@pytest.mark.parametrize("rows", [8, 32])
def test_c5_shape_bf16_sampling_spread_over_the_chip(hip, rows):
    """Config 5's sampling (top-k 40, temperature 0.8) in bf16 through the one-call step, where the head leaves its
    packed maxima and the sampler spreads every row over the chip: every generated id is the oracle's draw (and the
    one-workgroup-per-row kernel's) from the logits the step produced, eagerly and under graph replay."""
    from test_gpu_model import make_pair, prompt, replayed
    ocfg, w, model = make_pair(seed=2, init="healthy", dtype=torch.bfloat16, mlp_scale=2, n_embd=256, n_layers=4,
                               n_heads=2, window_size=24, num_eigh=24, seq_len=256, vocab_size=2003,
                               stu_decode_mode="lds")
    P, N = 20, 40
    ids = prompt(rows, P, ocfg.vocab_size, 4)
    got, gl = model.generate(ids.cuda(), max_length=P + N, temperature=0.8, top_k=40, do_sample=True, seed=2,
                             return_logits=True)
    how = dict(temperature=0.8, top_k=40, do_sample=True, seed=2)
    assert torch.equal(model.generate(ids.cuda(), max_length=P + N, **how), got)
    assert torch.equal(replayed(model, ids.cuda(), P + N, **how), got)
    miss = 0
    for t in range(N):
        lt = gl[:, t].contiguous()
        ref = torch.empty(rows, dtype=torch.int64, device="cuda")
        hip.sample(lt, ref, 0.8, 40, None, True, seed=2, step=t)
        assert torch.equal(got[:, P + t], ref), t
        o = O.next_token(lt.cpu(), 0.8, 40, None, True, seed=2, step=t)[:, 0]
        miss += int((got[:, P + t].cpu() != o).sum())
    assert miss <= 1, miss


@pytest.mark.parametrize("rows", [17, 20, 32])
def test_c5_shape_bf16_lds_teacher_forced(rows):
    """Same structure in bf16 with the recurrence state, logits within the bf16 tolerance.  17..32 rows step as one
    chunk: projections, MLP and head once over all rows on the packed-weight kernels (two row tiles per weight
    fragment), the state operators over all rows in one launch each."""
    from test_gpu_model import make_pair, prompt, _teacher_forced, replayed
    ocfg, w, model = make_pair(seed=2, init="healthy", dtype=torch.bfloat16, mlp_scale=2, n_embd=256, n_layers=4,
                               n_heads=2, window_size=24, num_eigh=24, seq_len=256, vocab_size=2003,
                               stu_decode_mode="lds")
    P, N = 20, 60
    ids = prompt(rows, P, ocfg.vocab_size, 4)
    got, gl = model.generate(ids.cuda(), max_length=P + N, do_sample=False, return_logits=True)
    assert torch.equal(model.generate(ids.cuda(), max_length=P + N, do_sample=False), got)
    assert torch.equal(replayed(model, ids.cuda(), P + N), got)
    ref = _teacher_forced(w, ocfg, got.cpu(), P).float()
    err = (gl.float().cpu() - ref).abs().amax(-1) / ref.abs().amax(-1)
    assert float(err.max()) <= 2e-2


@pytest.mark.parametrize("P", [1, 20])
def test_c5_shape_bf16_more_rows_than_one_chunk(P):
    """40 rows step as a chunk of 32 (packed-weight kernels over two row tiles, the recurrence step handing its
    odd-lag sum on, primed after a prompt of P positions) and a chunk of 8 (the 16-row kernels): every row's ids are
    those of its chunk generated alone, its logits agree with that run to rounding, and they meet the teacher-forced
    oracle."""
    from test_gpu_model import make_pair, prompt, _teacher_forced
    ocfg, w, model = make_pair(seed=2, init="healthy", dtype=torch.bfloat16, mlp_scale=2, n_embd=256, n_layers=4,
                               n_heads=2, window_size=24, num_eigh=24, seq_len=256, vocab_size=2003,
                               stu_decode_mode="lds")
    N = 30
    ids = prompt(40, P, ocfg.vocab_size, 4)
    got, gl = model.generate(ids.cuda(), max_length=P + N, do_sample=False, return_logits=True)
    assert torch.equal(model.generate(ids.cuda(), max_length=P + N, do_sample=False), got)        # graph replay
    for lo, hi in ((0, 32), (32, 40)):
        part, pl = model.generate(ids[lo:hi].cuda(), max_length=P + N, do_sample=False, return_logits=True)
        assert torch.equal(part, got[lo:hi])
        # (the prompt pass picks its GEMM tiles by the number of rows, so the logits agree to rounding, not bit for bit)
        assert float((pl.float() - gl[lo:hi].float()).abs().max()) <= 2e-2 * float(gl.float().abs().max())
    ref = _teacher_forced(w, ocfg, got.cpu(), P).float()
    err = (gl.float().cpu() - ref).abs().amax(-1) / ref.abs().amax(-1)
    assert float(err.max()) <= 2e-2


@pytest.mark.parametrize("d,heads,rows", [(1024, 8, 8), (2048, 16, 8), (2048, 16, 32), (1024, 8, 21)])
def test_c5_width_bf16_step_kernels(d, heads, rows):
    """Config 5's widths through the whole one-call step (head dim 128, d=2048 takes the 8-k-step variants of the
    balanced gate/up kernel and its norm prologue; 17..32 rows take the packed-weight kernels with two row tiles per
    weight fragment for the MLP, the small projections and the head): two layers, bf16, logits against the
    teacher-forced oracle."""
    from test_gpu_model import make_pair, prompt, _teacher_forced, replayed
    ocfg, w, model = make_pair(seed=4, init="healthy", dtype=torch.bfloat16, mlp_scale=4, n_embd=d, n_layers=2,
                               n_heads=heads, window_size=32, num_eigh=24, seq_len=128, vocab_size=1511,
                               stu_decode_mode="lds")
    P, N = 12, 28
    ids = prompt(rows, P, ocfg.vocab_size, 6)
    got, gl = model.generate(ids.cuda(), max_length=P + N, do_sample=False, return_logits=True)
    assert torch.equal(model.generate(ids.cuda(), max_length=P + N, do_sample=False), got)
    assert torch.equal(replayed(model, ids.cuda(), P + N), got)
    ref = _teacher_forced(w, ocfg, got.cpu(), P).float()
    err = (gl.float().cpu() - ref).abs().amax(-1) / ref.abs().amax(-1)
    assert float(err.max()) <= 2e-2


def test_c5_full_architecture_decode_against_full_sequence_recompute():
    """BASELINE config 5's full architecture (d=2048, 24 layers, 16 heads of 128, window 1024, L=8192, mlp_scale 12:
    3.98 B parameters) at batch 32 (one chunk of 32 rows that reads every weight once) with its sampler (top-k 40,
    temperature 0.8, seeded stream); the CPU oracle is out of reach at this size, so the checks are size-independent:
    graph replay equals the kernel-by-kernel loop token for token, a second run reproduces the ids, and the stateful
    logits equal those of a full-sequence forward over the same tokens within the bf16 tolerance.  The prompt is
    cut to 1100 tokens to keep the test short: longer than the 1025-slot ring, so the prompt pass fills a wrapped
    ring and every decode step reads the full window through the streamed head-dim-128 attention kernel."""
    from flash_stu import FlashSTU, FlashSTUConfig
    from test_gpu_model import prompt, replayed
    torch.manual_seed(2)
    cfg = FlashSTUConfig(n_embd=2048, n_layers=24, n_heads=16, window_size=1024, seq_len=8192, vocab_size=50257,
                         num_eigh=24, mlp_scale=12, torch_dtype=torch.bfloat16)
    with torch.device("cuda"):
        model = FlashSTU(cfg)
    model = model.cuda().eval()
    assert abs(model.get_num_params() - 3.98e9) < 0.05e9
    B, P, N = 32, 1100, 24
    ids = prompt(B, P, cfg.vocab_size, 2).cuda()
    kw = dict(max_length=P + N, do_sample=True, top_k=40, temperature=0.8, seed=2)
    eager, logits = model.generate(ids, return_logits=True, **kw)
    assert torch.equal(replayed(model, ids, **kw), eager)
    assert torch.equal(model.generate(ids, **kw), eager)
    worst = 0.0
    for s in (0, 5, N - 1):
        full = model(eager[:, :P + s].contiguous()).logits[:, -1, :].float()
        got = logits[:, s, :].float()
        worst = max(worst, float(((got - full).abs().amax(-1) / full.abs().amax(-1)).max()))
    assert worst <= 2e-2, worst
    del model
    torch.cuda.empty_cache()
