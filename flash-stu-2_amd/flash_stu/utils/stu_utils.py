"""Spectral filters of the STU: top eigenvectors of a fixed Hankel matrix.

Host-side, float64, run once per model (reference:
flash_stu/utils/stu_utils.py:18-31,33-143,146-193).  Unlike the reference this
needs no GPU: the eigen-decomposition runs in numpy on the host either way.
"""
from __future__ import annotations

import os
from typing import Optional

import numpy as np
import torch


def get_hankel(seq_len: int, use_hankel_L: bool = False) -> np.ndarray:
    idx = np.arange(1, seq_len + 1, dtype=np.float64)
    s = idx[:, None] + idx[None, :]
    if use_hankel_L:
        return ((-1.0) ** (s - 2.0) + 1.0) * (8.0 / ((s + 3.0) * (s - 1.0) * (s + 1.0)))
    return 2.0 / (s ** 3 - s)


def save_spectral_filters(phi: torch.Tensor, path: str, seq_len: Optional[int] = None, K: Optional[int] = None,
                          use_hankel_L: bool = False, **metadata) -> None:
    """Stores filters with the metadata keys the reference writes
    (stu_utils.py:33-82) so files are interchangeable."""
    os.makedirs(os.path.dirname(os.path.abspath(path)), exist_ok=True)
    L, k = phi.shape
    torch.save({"phi": phi.detach().cpu(), "seq_len": seq_len or L, "K": K or k, "use_hankel_L": use_hankel_L,
                "dtype": str(phi.dtype), **metadata}, path)


def load_spectral_filters(path: str, device=None, dtype: Optional[torch.dtype] = None,
                          verify_shape: Optional[tuple] = None) -> torch.Tensor:
    """Loads a filter file (tensor-only payload; nothing in it is executed)."""
    if not os.path.exists(path):
        raise FileNotFoundError(f"Filter file not found: {path}")
    blob = torch.load(path, map_location="cpu", weights_only=True)
    phi = blob["phi"] if isinstance(blob, dict) else blob
    if verify_shape is not None and tuple(phi.shape) != tuple(verify_shape):
        raise ValueError(f"Filter shape mismatch: expected {tuple(verify_shape)}, got {tuple(phi.shape)}")
    if dtype is not None:
        phi = phi.to(dtype)
    if device is None:
        device = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    return phi.to(device)


def get_spectral_filters(seq_len: int, K: int, use_hankel_L: bool = False, device=None,
                         dtype: torch.dtype = torch.bfloat16, load_from: Optional[str] = None) -> torch.Tensor:
    """(seq_len, K) filters: eigenvectors of the K largest eigenvalues (ascending
    order) scaled by eigenvalue**0.25, cast to `dtype`."""
    if load_from is not None:
        return load_spectral_filters(load_from, device=device, dtype=dtype, verify_shape=(seq_len, K))
    if device is None:
        device = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    sigma, vecs = np.linalg.eigh(get_hankel(seq_len, use_hankel_L))
    sigma, vecs = sigma[-K:], vecs[:, -K:]
    return torch.tensor(vecs * sigma ** 0.25, device=device, dtype=dtype)


# ---------------------------------------------------------------- the spectral convolution as an operator
def nearest_power_of_two(x: int, round_up: bool = False) -> int:
    """flash_stu/utils/numerics.py:3-6."""
    return 1 << (int(x) - 1).bit_length() if round_up else 1 << (int(x).bit_length() - 1)


def _alt_sign(L: int, like: torch.Tensor) -> torch.Tensor:
    s = torch.ones(L, 1, dtype=like.dtype, device=like.device)
    s[1::2] = -1
    return s


def _conv_length(T: int) -> int:
    """Transform length of the FFT kernels for T positions; 0 where the time-domain kernel runs instead (fewer than 32
    positions, or more than the in-LDS transform reaches)."""
    from .. import _hip
    return _hip.fft_length(T) if T >= 32 else 0


def _causal_conv(u: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    """u (B,T,d) with the per-channel filter v (L,d): out[b,t,c] = T(sum_{s<=t} v[s,c] u[b,t-s,c]), one branch."""
    from .. import _hip
    n = _conv_length(u.shape[1])
    if n == 0:
        return _hip.stu_conv_direct(u.contiguous(), v.contiguous(), single_branch=True)
    return _hip.stu_conv_fft(u.contiguous(), _hip.stu_fft_filter(v.contiguous(), n, single_branch=True), single_branch=True)


def _convolve_grads(ctx, u, v, spec, gp, gm, branches):
    """Gradients of the convolution in u and v, formed in fp32 whatever the input dtype (the reference differentiates
    through an fp32 FFT, stu_utils.py:226-228) and rounded once at the end.  branches 0: gp is the gradient of
    plus + minus; 1: of plus alone; 2: gp and gm are those of plus and minus.  One launch on the matrix cores (branches 0,
    bf16), or from the filters' spectra one launch of the transforms' gradient kernel; at the lengths of the time-domain kernel, and where the gradients are to be differentiated
    themselves (create_graph=True: the composition carries its graph), as convolutions: the minus branch
    sgn * conv(sgn * u, v) equals conv(u, v * (-1)^s), and
      d/du: correlation with the filter     = time-reversed convolution of the time-reversed gradient
      d/dv: correlation of gradient and u   = per batch row, convolution of the time-reversed gradient with that
            row's input as the filter, read backwards; summed over the batch in fp32."""
    from .. import _hip
    want_u, want_v = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
    graph = torch.is_grad_enabled()
    if branches == 0 and not graph and v.dtype == u.dtype == gp.dtype and _hip.stu_conv_mfma_grad_takes(*u.shape, v.shape[0], u.dtype):
        return _hip.stu_conv_mfma_grad(_aligned(gp), _aligned(u), _aligned(v), want_u, want_v)
    n = _conv_length(u.shape[1])
    if spec is None and n and not graph:
        spec = _hip.stu_fft_filter(v.contiguous(), n)            # the forward was a Toeplitz product of more than 2048 positions
    if spec is not None and not graph:
        return _hip.stu_conv_fft_grad(gp.contiguous(), gm.contiguous() if branches == 2 else None, u.contiguous(), spec,
                                      v.shape[0], branches, want_u, want_v)
    both = branches != 1
    gm = gp if branches == 0 else gm
    B, T, d = u.shape
    L = v.shape[0]
    uf, vf = u.float(), v.float()

    def conv(a, f):
        return _ApproxConvolve.apply(a, f, False)[0] if graph else _causal_conv(a, f)
    gpf = gp.float().flip(1).contiguous()
    gmf = gm.float().flip(1).contiguous() if both else None
    gu = gv = None
    if want_u:
        gu = conv(gpf, vf)
        if both:
            gu = gu + conv(gmf, vf * _alt_sign(L, vf))
        gu = gu.flip(1).to(u.dtype)
    if want_v:
        taps = min(L, T)
        acc_p = torch.zeros(T, d, dtype=torch.float32, device=u.device)
        acc_m = torch.zeros_like(acc_p) if both else None
        for b in range(B):
            ub = uf[b].contiguous()                              # (T,d): this row's input as the filter
            acc_p += conv(gpf[b:b + 1], ub)[0]
            if both:
                acc_m += conv(gmf[b:b + 1], ub)[0]
        gv = torch.zeros(L, d, dtype=torch.float32, device=u.device)
        gv[:taps] = acc_p.flip(0)[:taps]                         # lag s sits at position T-1-s
        if both:
            gv[:taps] += acc_m.flip(0)[:taps] * _alt_sign(taps, acc_m)
        gv = gv.to(v.dtype)
    return gu, gv


class _ApproxConvolve(torch.autograd.Function):
    """Both sign branches of the approx-mode convolution with their gradients."""

    @staticmethod
    def forward(ctx, u, v, both):
        from .. import _hip
        ctx.both = both
        n = _conv_length(u.shape[1])
        spec = _hip.stu_fft_filter(v.contiguous(), n) if n else None
        ctx.save_for_backward(u, v, spec)
        up = _hip.stu_conv_fft(u.contiguous(), spec, single_branch=True) if n else _causal_conv(u, v)
        if not both:
            return up, torch.zeros(0, dtype=u.dtype, device=u.device)
        return up, _causal_conv(u, v * _alt_sign(v.shape[0], v))

    @staticmethod
    def backward(ctx, gp, gm):
        u, v, spec = ctx.saved_tensors
        return (*_convolve_grads(ctx, u, v, spec, gp, gm, 2 if ctx.both else 1), None)


class ApproxConvolveSum(torch.autograd.Function):
    """y = T(T(plus) + T(minus)) of the approx-mode convolution, as the STU adds its branches (stu.py:120), with its
    gradients.  The odd lags cancel between the branches but for rounding, so they get none."""

    @staticmethod
    def forward(ctx, u, v):
        from .. import _hip
        # The form that the gradients will take, so that the filter is laid out once.  Beyond 2048 positions their only form are the
        # transforms, and a product in front of them pays for their spectra: GPU us of a step, 2 x 3000 x 2048 540 / 549 with
        # transforms in both directions, 1 x 4096 x 1536 337 / 347.
        B, T, d = u.shape
        if v.dtype == u.dtype and (_hip.stu_conv_mfma_grad_takes(B, T, d, v.shape[0], u.dtype) if T <= 2048 else
                                   _hip.stu_conv_mfma_takes(T, d, u.dtype)):
            ctx.save_for_backward(u, v, None)
            return _hip.stu_conv_mfma(_aligned(u), _hip.stu_conv_taps(_aligned(v), _hip.stu_conv_taps_len(u.shape[1])))
        n = _conv_length(u.shape[1])
        spec = _hip.stu_fft_filter(v.contiguous(), n) if n else None
        ctx.save_for_backward(u, v, spec)
        if n:
            return _hip.stu_conv_fft(u.contiguous(), spec)
        return _hip.stu_conv_direct(u.contiguous(), v.contiguous())

    @staticmethod
    def backward(ctx, gy):
        u, v, spec = ctx.saved_tensors
        return _convolve_grads(ctx, u, v, spec, gy, None, 0)


class ProjectInputs(torch.autograd.Function):
    """x (B,T,d_in) @ m (d_in,d_out) in bf16 with its gradients on the matrix-core kernels.  The gradient of m sums over all
    B*T positions: both operands are read as they lie (reduction index slowest), the long sum is taken in slices (8 x 2048
    positions of 768: 32 us; with the output's gradient transposed in front 50, the library product 94).
    Where the gradients are to be differentiated themselves (create_graph=True) they are plain products."""

    @staticmethod
    def takes(x, m) -> bool:
        if x.dim() != 3 or not x.is_cuda or x.dtype != torch.bfloat16 or m.dtype != torch.bfloat16 or m.device != x.device or torch.is_autocast_enabled():
            return False
        rows, d_in, d_out = x.shape[0] * x.shape[1], m.shape[0], m.shape[1]
        return (x.shape[2] == d_in and rows >= 128 and rows % 64 == 0 and d_in % 128 == 0 and d_out % 128 == 0 and m.is_contiguous()
                and m.data_ptr() % 16 == 0 and rows * d_in < 1 << 30 and rows * d_out < 1 << 30)

    @staticmethod
    def forward(ctx, x, m):
        from .. import _hip
        ctx.save_for_backward(x, m)
        x2 = _aligned(x.reshape(-1, x.shape[2]))
        return _hip.gemm(x2, _hip.transpose(m[None])[0]).view(*x.shape[:2], m.shape[1])

    @staticmethod
    def backward(ctx, g):
        from .. import _hip
        x, m = ctx.saved_tensors
        if torch.is_grad_enabled():
            return (g @ m.T if ctx.needs_input_grad[0] else None,
                    x.reshape(-1, x.shape[2]).T @ g.reshape(-1, g.shape[2]) if ctx.needs_input_grad[1] else None)
        g2 = _aligned(g.reshape(-1, g.shape[2]))
        gx = _hip.gemm(g2, m).view_as(x) if ctx.needs_input_grad[0] else None
        gm = None
        if ctx.needs_input_grad[1]:
            x2 = _aligned(x.reshape(-1, x.shape[2]))
            gm = _hip.gemm_tt(x2, g2)
        return gx, gm


class ApproxUnit(torch.autograd.Function):
    """The whole approx-mode STU, conv(x @ m_inputs, phi @ m_filters) with its branches added, in bf16 where its convolution and the
    gradients are products: five launches forward and seven backward, none of them a library's, and one node for the host to
    go through (8 x 2048 x 768: as four nodes, two of them library products, the host took longer than the GPU).  phi_e holds the even
    rows of phi as the gradient of m_filters reads them.  Where the gradients are to be differentiated themselves
    (create_graph=True) they are those of the composed operators.  No gradient needs the values of m_filters, which may therefore change
    before the backward pass, as they may behind phi @ m_filters."""

    @staticmethod
    def takes(x, phi, m_inputs, m_filters) -> bool:
        from .. import _hip
        if x.dim() != 3 or not x.is_cuda or torch.is_autocast_enabled() or phi.requires_grad:
            return False
        if any(t.dtype != torch.bfloat16 or t.device != x.device or not t.is_contiguous() or t.data_ptr() % 16 for t in (phi, m_inputs, m_filters)):
            return False
        (B, T, d_in), (L, K), d = x.shape, phi.shape, m_inputs.shape[1]
        return (x.dtype == torch.bfloat16 and m_inputs.shape[0] == d_in and m_filters.shape == (K, d) and T <= L and K <= 128
                and B * T >= 128 and d_in % 128 == 0 and d % 128 == 0 and B * T * d_in < 1 << 30 and B * T * d < 1 << 30
                and _hip.stu_conv_mfma_grad_takes(B, T, d, L, x.dtype))

    @staticmethod
    def forward(ctx, x, phi, phi_e, m_inputs, m_filters):
        from .. import _hip
        x2 = _aligned(x.reshape(-1, x.shape[2]))
        u = _hip.gemm(x2, _hip.transpose(m_inputs[None])[0]).view(*x.shape[:2], m_inputs.shape[1])
        v, taps = _hip.stu_conv_taps_project(phi, m_filters, x.shape[1])
        of_inputs, of_filters = any(ctx.needs_input_grad[i] for i in (0, 3)), ctx.needs_input_grad[4]
        ctx.save_for_backward(*((x, m_inputs) if of_inputs else (None, None)), *((phi, phi_e) if of_filters else (None, None)), u, v)
        ctx.m_filters = m_filters if ctx.needs_input_grad[4] else None
        ctx.version = m_filters._version if ctx.needs_input_grad[4] else 0
        return _hip.stu_conv_mfma(u, taps)

    @staticmethod
    def backward(ctx, gy):
        from .. import _hip
        x, m_inputs, phi, phi_e, u, v = ctx.saved_tensors        # (what the wanted ones need)
        want_x, _, _, want_i, want_f = ctx.needs_input_grad
        if torch.is_grad_enabled():
            filt, m_filters = v, ctx.m_filters
            if want_f:
                if m_filters._version != ctx.version and m_filters.grad_fn is not None:
                    raise RuntimeError("m_filters was modified in place by an operation that its gradient's own graph would run through")
                now = phi[:v.shape[0]] @ m_filters
                filt = v + (now - now.detach())          # the forward pass's values, on the way to m_filters
            wanted = [t for t, w in ((x, want_x), (m_inputs, want_i), (m_filters, want_f)) if w]
            proj = x @ m_inputs if want_x or want_i else u
            grads = iter(torch.autograd.grad(ApproxConvolveSum.apply(proj, filt), wanted, gy, create_graph=True))
            return next(grads) if want_x else None, None, None, next(grads) if want_i else None, next(grads) if want_f else None
        gy, gf = _aligned(gy), None
        if want_f:
            gu, gf = _hip.stu_conv_mfma_grad_project(gy, u, v, phi_e, phi.shape[1], want_x or want_i)
        else:
            gu, _ = _hip.stu_conv_mfma_grad(gy, u, v, True, False)
        if not (want_x or want_i):
            return None, None, None, None, gf
        gu = gu.view(-1, gu.shape[2])
        gx = _hip.gemm(gu, m_inputs).view_as(x) if want_x else None
        gi = _hip.gemm_tt(_aligned(x.reshape(-1, x.shape[2])), gu) if want_i else None
        return gx, None, None, gi, gf


def _aligned(t: torch.Tensor) -> torch.Tensor:
    """t with dense rows at a 16-byte address, as the matrix-core kernels read it."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def convolve(u: torch.Tensor, v: torch.Tensor, n: int, use_approx: bool = True, return_both: bool = True,
             sgn: Optional[torch.Tensor] = None, v_fft: Optional[torch.Tensor] = None):
    """The reference's causal convolution (flash_stu/utils/stu_utils.py:195-246), same arguments and results:
    u (B,T,d); approx mode v (L,d) per-channel filters -> (U_plus, U_minus) of shape (B,T,d); exact mode v (L,K) filter
    bank -> (B,T,K,d) each; U_minus is None with return_both=False.  Results are rounded to u's dtype.  `n` must cover
    the linear convolution (n >= 2T-1, as the reference chooses it); the kernels pick their own transform length, and
    `sgn` / `v_fft` (the reference's cached operands) are accepted and not needed.  Approx mode is differentiable in
    u and v (training-side use: flash_stu/modules/stu.py:89-98 under autograd); exact mode is forward only."""
    from .. import _hip
    if u.dim() != 3 or v.dim() != 2:
        raise ValueError("convolve: u must be (B,T,d) and v (L,d) or (L,K)")
    B, T, d = u.shape
    if n < 2 * T - 1:
        raise ValueError(f"convolve: n={n} is shorter than the linear convolution of {T} positions")
    if not u.is_cuda:
        raise _hip.FlashSTUHipError("tensor is not on the GPU: the HIP path has no CPU fallback")
    v = v.to(u.dtype)
    if use_approx:
        if v.shape[1] != d:
            raise ValueError(f"convolve: approx mode needs one filter per channel, got v {tuple(v.shape)} for d={d}")
        up, um = _ApproxConvolve.apply(u, v, bool(return_both))
        return up, (um if return_both else None)
    if u.requires_grad or v.requires_grad:
        raise NotImplementedError("convolve: exact mode (use_approx=False) is forward only")
    K = v.shape[1]
    up = torch.empty(B, T, K, d, dtype=u.dtype, device=u.device)
    um = torch.empty_like(up) if return_both else None
    nn_ = _hip.fft_length(T) if T >= 32 else 0
    if nn_ == 0:
        _hip.stu_conv_bank(u.contiguous(), v.contiguous(), up, um)
    else:
        spec = _hip.stu_fft_filter(v.contiguous(), nn_, single_branch=not return_both)
        ut = _hip.transpose(u.contiguous()).transpose(1, 2)        # time-major copy: coalesced column loads
        slabs = None
        if nn_ == 16384:
            # A workgroup has one channel: into (T,K,d) it would store one element of a line at a time, and with two of them to
            # a compute unit more lines are open than the L2s hold.  Time-major slabs of one row, transposed instead: 24
            # filters, both branches, us, into (T,K,d) / slabs, 1 x 8000 x 1024 bf16 4118 / 1074, fp32 5453 / 1604 (one
            # workgroup to a compute unit 2651 and 4123), 1 x 8000 x 256 bf16 666 / 331, 4 x 5000 x 768 5028 / 2690.
            try:
                slabs = torch.empty(1 + bool(return_both), K, d, T, dtype=u.dtype, device=u.device)
            except torch.OutOfMemoryError:
                pass                                               # results that leave no room for them
        if slabs is None:
            _hip.stu_conv_bank_fft(ut, spec, up, um)
        else:
            views = [t[None].permute(0, 3, 1, 2) for t in slabs] + [None]
            for b in range(B):
                _hip.stu_conv_bank_fft(ut[b:b + 1], spec, views[0], views[1])
                for slab, out in zip(slabs, (up, um)):
                    _hip.transpose(slab.view(1, K * d, T), out[b].view(1, T, K * d))
    return up, um
