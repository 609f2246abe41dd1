"""Decode engine behind FlashSTU.generate(): prefill through the module path,
then one C-ABI call (fstu_decode_steps) that launches the fused kernel sequence
of every token for the whole layer stack against preallocated state and workspaces,
or, for several row chunks, the same steps captured as a HIP graph per chunk.

The token buffer (B, max_length) lives on the GPU for the whole loop; each step
reads column pos and writes column pos+1, so the host never sees a token until
generate() returns (reference loop: flash_stu/model.py:245-302, which re-allocates
the sequence with torch.cat every step).

The decode kernels take at most 16 activation rows; a larger batch runs as
consecutive row chunks of 16 against the same weights and batch-first state.
"""
from __future__ import annotations

import array
import ctypes
from typing import List, Optional

import torch

from . import _hip
from .layers.attention_layer import AttentionLayer
from .layers.stu_layer import STULayer
from .modules.attention import Attention
from .modules.norm import RMSNorm
from .modules.stu import STU
from .modules.swiglu import MLP

_vp, _i, _f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float


class LayerDesc(ctypes.Structure):
    _fields_ = [("kind", _i), ("norm1_w", _vp), ("mlp_norm_w", _vp), ("w_gate", _vp), ("w_up", _vp), ("w_down", _vp),
                ("m_inputs_t", _vp), ("filt", _vp), ("hist", _vp), ("lds_a", _vp), ("lds_ce", _vp), ("lds_co", _vp), ("lds_state", _vp), ("lds_ring", _vp), ("lds_fir", _vp), ("lds_ocache", _vp),
                ("w_qkv", _vp), ("w_proj", _vp), ("kring", _vp), ("vring", _vp), ("slopes", _vp),
                ("wp_gate", _vp), ("wp_up", _vp), ("wp_down", _vp), ("wp_m_inputs", _vp), ("wp_qkv", _vp),
                ("wp_proj", _vp)]


class ModelDesc(ctypes.Structure):
    _fields_ = [("dtype", _i), ("B", _i), ("d", _i), ("I", _i), ("V", _i), ("n_layers", _i), ("n_heads", _i),
                ("head_dim", _i), ("window", _i), ("kv_cap", _i), ("L", _i), ("hist_cap", _i), ("stu_mode", _i),
                ("lds_S", _i), ("lds_fir_taps", _i), ("single_branch", _i), ("ksplit_down", _i), ("hist_nsplit_max", _i), ("row0", _i),
                ("eps", _f), ("softcap", _f), ("emb", _vp), ("final_norm_w", _vp), ("layers", ctypes.POINTER(LayerDesc)),
                ("x", _vp), ("h", _vp), ("qkv", _vp), ("attn", _vp), ("act", _vp), ("xp", _vp), ("y", _vp),
                ("partial", _vp), ("eo", _vp), ("logits", _vp), ("best", _vp), ("samp_ws", _vp),
                ("wp_emb", _vp), ("x2", _vp), ("glu_packed", _i), ("down_packed", _i), ("merge_norm", _i),
                ("row_major", _i)]


def pick_ksplit_down(I: int) -> int:
    """K split of the down projection: enough waves to fill 256 CUs while every
    slice still divides into the 64-wide k steps of the MFMA kernel."""
    for ks in (12, 16, 8, 6, 4, 3, 2):
        if I % (ks * 256) == 0:
            return ks
    for ks in (8, 4, 2):
        if I % (ks * 64) == 0:
            return ks
    return 1


# What the layers' own calls run, as defined when the package was imported
_AS_DEFINED = [(cls, name, cls.__dict__[name]) for cls, names in (
    (torch.nn.Module, ("__call__", "_call_impl")), (RMSNorm, ("forward", "add_then_norm")), (MLP, ("forward",)),
    (Attention, ("forward",)), (STU, ("forward", "_step")), (STULayer, ("forward",)), (AttentionLayer, ("forward",)))
    for name in names]
_OWN_NAMES = {name for _, name, _ in _AS_DEFINED}


def _as_written(m, cls) -> bool:
    """The module is of this class and calling it runs this class's methods and nothing else."""
    return type(m) is cls and not m._forward_hooks and not m._forward_pre_hooks and _OWN_NAMES.isdisjoint(m.__dict__)


# LayerDesc as words of 8 bytes: every field is a pointer but the first, an int in a word of its own
_LAYER_WORDS = [name for name, _ in LayerDesc._fields_]
_AT = {name: i for i, name in enumerate(_LAYER_WORDS)}
assert ctypes.sizeof(LayerDesc) == 8 * len(_LAYER_WORDS) and all(getattr(LayerDesc, name).offset == 8 * i for name, i in _AT.items())


def _weight(m):
    """The weight of a norm or a linear layer; past the module's attribute lookup where its class is the plain one (a
    parametrized module has a class of its own, and forms a temporary on each access)."""
    w = m._parameters.get("weight") if type(m) in (torch.nn.Linear, RMSNorm) else None
    return m.weight if w is None else w


@_hip.inference
def step_on_caches(model, ids: torch.Tensor, past):
    """One position of each row, ids (B,1), against the caches that model(..., use_cache=True) returned: (logits (B,1,V),
    caches one position on) through the one-call step, the state in the caches advanced in place, or None where a row
    count, a configuration, a cache or a module is not what that step takes (the layers' own forward calls then run).

    Everything is read from the model and the caches of this call: no pointer or check outlives it, and the weights are
    the parameters themselves, not packed copies.  Every tensor whose address is taken is held until the launches are
    enqueued: a parametrized weight is a temporary that its module forms on each access."""
    cfg = model.config
    mod = torch.nn.modules.module
    if not (ids.dim() == 2 and ids.shape[1] == 1 and 1 <= ids.shape[0] <= _hip.MAX_DECODE_ROWS and ids.dtype == torch.int64
            and DecodeEngine.supports(cfg) and isinstance(past, (tuple, list)) and len(past) == len(model.layers) > 0
            and not mod._global_forward_hooks and not mod._global_forward_pre_hooks and _as_written(model.norm, RMSNorm)
            and all(cls.__dict__.get(name) is f for cls, name, f in _AS_DEFINED)):
        return None
    emb = model.lm_head.weight
    dt, dev, B, (V, d) = emb.dtype, emb.device, ids.shape[0], emb.shape
    H, W, eps, cap0 = cfg.n_heads, cfg.window_left, cfg.rms_norm_eps, float(cfg.softcap or 0.0)
    n, lds = len(model.layers), cfg.resolved_stu_decode_mode() == "lds"
    if (dt not in (torch.bfloat16, torch.float32) or not emb.is_cuda or ids.device != dev or model.tok_emb.weight is not emb
            or model.lm_head.bias is not None or d != cfg.n_embd or d % H != 0 or model.norm.eps != eps):
        return None
    I, hd = d * cfg.mlp_scale, d // H
    # What every launch reads or writes, its shape and the descriptor field it goes to, layer behind layer: checked below all
    # together, since a check of its own for each of some 130 tensors took the host longer than the GPU takes for the step (a step's host
    # side at 12 layers 430 us, 390 so; of both the launches are 140).
    tensors, shapes, places = [], [], []     # of the model's dtype
    tensors32, shapes32, places32 = [], [], []
    vec, mat_id, mat_di, mat_dd, mat_3d = (d,), (I, d), (d, I), (d, d), (3 * d, d)
    ring = (B, H, W + 1, hd)
    out = []
    pos = hist_cap = fir_taps = None
    S = 0
    for i, (layer, entry) in enumerate(zip(model.layers, past)):
        stu_layer = type(layer) is STULayer
        if not _as_written(layer, STULayer if stu_layer else AttentionLayer) or not isinstance(entry, tuple) or len(entry) != 3:
            return None
        sub = layer._modules                 # (of exactly these classes: what the attributes of the layer are)
        op, norm1 = (sub["stu"], sub["stu_norm"]) if stu_layer else (sub["attn"], sub["attn_norm"])
        mlp, norm2 = sub["mlp"], sub["mlp_norm"]
        if not (_as_written(op, STU if stu_layer else Attention) and _as_written(norm1, RMSNorm) and type(norm2) is RMSNorm
                and _OWN_NAMES.isdisjoint(norm2.__dict__) and _as_written(mlp, MLP) and norm1.eps == eps and norm2.eps == eps):
            return None
        proj = mlp._modules
        gate, up, down = proj["gate_proj"], proj["up_proj"], proj["down_proj"]
        a0, a1, pos_t = entry
        if gate.bias is not None or pos_t.is_cuda or pos_t.dim() != 1 or pos_t.numel() < 1:
            return None
        p = int(pos_t.tolist()[0])           # (any dtype that holds it)
        if pos is not None and p != pos:
            return None
        pos = p
        at = i * len(_LAYER_WORDS)
        tensors += (_weight(norm1), _weight(norm2), _weight(gate), _weight(up), _weight(down))
        shapes += (vec, vec, mat_id, mat_id, mat_di)
        places += (at + _AT["norm1_w"], at + _AT["mlp_norm_w"], at + _AT["w_gate"], at + _AT["w_up"], at + _AT["w_down"])
        if not stu_layer:
            if op.n_heads != H or op.window_size != W or op.softcap != cap0 or op.c_attn.bias is not None or op.c_proj.bias is not None:
                return None
            tensors += (_weight(op.c_attn), _weight(op.c_proj), a0, a1)
            shapes += (mat_3d, mat_dd, ring, ring)
            places += (at + _AT["w_qkv"], at + _AT["w_proj"], at + _AT["kring"], at + _AT["vring"])
            tensors32.append(op.alibi_slopes)
            shapes32.append((H,))
            places32.append(at + _AT["slopes"])
        else:
            if op.M_inputs.device != dev or op.d_in != d or op.config is not cfg:
                return None
            tensors.append(op.m_inputs_t())
            shapes.append(mat_dd)
            places.append(at + _AT["m_inputs_t"])
            if lds:
                a, ce, co = op.lds_params()
                fir = op.lds_fir()
                taps = fir.shape[0] if fir is not None and a0.shape[1] == fir.shape[0] else 0
                if fir_taps not in (None, taps) or S not in (0, a.numel()) or (taps == 0 and a0.numel() != 0):
                    return None
                fir_taps, S = taps, a.numel()
                tensors32 += (a, ce, co, a1)
                shapes32 += ((S,), (S, d), (S, d), (B, 2, S, d))
                places32 += (at + _AT["lds_a"], at + _AT["lds_ce"], at + _AT["lds_co"], at + _AT["lds_state"])
                if taps:
                    tensors.append(a0)
                    shapes.append((B, taps, d))
                    places.append(at + _AT["lds_ring"])
                    tensors32.append(fir)
                    shapes32.append((taps, d))
                    places32.append(at + _AT["lds_fir"])
            else:
                filt = op.effective_filter()
                if a0.dim() != 3 or hist_cap not in (None, a0.shape[1]) or a1.numel() != 0 or pos >= a0.shape[1] or pos >= filt.shape[0]:
                    return None
                hist_cap = a0.shape[1]
                S = filt.shape[0]
                tensors += (filt, a0)
                shapes += ((S, d), (B, hist_cap, d))
                places += (at + _AT["filt"], at + _AT["hist"])
        out.append(entry)
    tensors += (emb, _weight(model.norm))
    shapes += ((V, d), vec)
    every = tensors + tensors32
    if (pos < 0 or any(t is None for t in every) or [t.shape for t in tensors] != shapes
            or [t.shape for t in tensors32] != shapes32 or {t.dtype for t in tensors} != {dt} or {t.dtype for t in tensors32} - {torch.float32}
            or {t.device for t in every} != {dev} or not all(map(torch.Tensor.is_contiguous, every))):
        return None
    ptrs = list(map(torch.Tensor.data_ptr, every))
    aligned = not any(q % 16 for q in ptrs)
    words = array.array("Q", bytes(8 * n * len(_LAYER_WORDS)))
    for place, q in zip(places + places32, ptrs[:len(places)] + ptrs[len(tensors):]):
        words[place] = q
    for i, layer in enumerate(model.layers):
        if type(layer) is not STULayer:
            words[i * len(_LAYER_WORDS)] = 1          # kind, the low half of its word
    m = ModelDesc()
    m.dtype = _hip.FSTU_BF16 if dt == torch.bfloat16 else _hip.FSTU_F32
    m.B, m.d, m.I, m.V, m.n_layers = B, d, I, V, n
    m.n_heads, m.head_dim, m.window, m.kv_cap = H, hd, W, W + 1
    m.L, m.hist_cap, m.stu_mode, m.lds_S = (cfg.seq_len if lds else S), hist_cap or 0, int(lds), (S if lds else 0)
    m.lds_fir_taps, m.single_branch = fir_taps or 0, int(cfg.use_hankel_L)
    m.ksplit_down = pick_ksplit_down(I) if dt == torch.bfloat16 else min(8, max(1, I // 512))
    m.hist_nsplit_max = DecodeEngine.HIST_NSPLIT_MAX
    m.eps, m.softcap = float(eps), cap0
    m.emb, m.final_norm_w = ptrs[len(places)], ptrs[len(places) + 1]
    m.layers = ctypes.cast(words.buffer_info()[0], ctypes.POINTER(LayerDesc))
    logits = torch.empty(B, 1, V, dtype=dt, device=dev)
    m.logits = logits.data_ptr()
    esz = emb.element_size()
    if aligned and dt == torch.bfloat16 and d <= 1024:
        # The launches of the packed step (norms as prologues, down projection in a few slices) on the parameters themselves.
        # 24 positions behind a prompt of 600, ms so / through the row-major kernels and launches of their own: 12 layers of 768,
        # 4 rows 11.8 / 13.1, 16 rows 16.7 / 17.9; 8 layers of 1024, 4 rows 8.9 / 9.4; but of 2048, where the bytes decide and one
        # workgroup to a compute unit fetches rows in halves of a line, 25.2 / 24.1.
        m.glu_packed = m.row_major = 1
        m.down_packed = m.merge_norm = int(I % 512 == 0)
    sizes = dict(x=B * d * esz, x2=B * d * esz, h=B * d * esz, y=B * d * esz, xp=B * d * esz, attn=B * d * esz, qkv=3 * B * d * esz,
                 act=B * I * esz, partial=max(m.ksplit_down, 16) * B * d * 4,
                 eo=0 if lds else DecodeEngine.HIST_NSPLIT_MAX * 2 * B * d * 4)
    ws = torch.empty(sum((v + 255) // 256 * 256 for v in sizes.values()), dtype=torch.uint8, device=dev)
    at = ws.data_ptr()
    for name, size in sizes.items():
        setattr(m, name, at)
        at += (size + 255) // 256 * 256
    ids = ids.contiguous()       # one token expanded over the rows has a row stride of 0
    _hip._check(_hip.load().fstu_decode_logits(ctypes.byref(m), ids.data_ptr(), 1, pos, _hip._stream()),
                "fstu_decode_logits")
    return logits, tuple((a0, a1, pos_t + 1) for a0, a1, pos_t in out)


class _Chunk:
    """Descriptor, workspaces and graph handle of one chunk of at most 16 batch rows."""

    def __init__(self, b0: int, b1: int):
        self.b0, self.b1 = b0, b1
        self.keep: List[torch.Tensor] = []
        self.arr = None
        self.desc: Optional[ModelDesc] = None
        self.logits: Optional[torch.Tensor] = None
        self.graphs = {}            # steps per graph -> handle
        self.dyn: Optional[torch.Tensor] = None
        self.stream = None


class DecodeEngine:
    HIST_NSPLIT_MAX = 16

    @staticmethod
    def supports(cfg) -> bool:
        """The one-call decode step covers approx-mode STU layers without the sandwich and bias-free linears;
        other variants decode through the layers' own state (FlashSTU.generate picks the loop)."""
        if cfg.use_hankel_L and cfg.resolved_stu_decode_mode() == "lds":
            return False     # single-branch filters on the recurrence state: the odd lags read the other bank
        return bool(cfg.use_approx) and not cfg.stu_enable_mlp_sandwich and not cfg.bias

    def __init__(self, model):
        cfg = model.config
        if not self.supports(cfg):
            raise NotImplementedError("the fused decode engine covers use_approx=True without the STU sandwich and "
                                      "without biases; FlashSTU.generate falls back to the per-layer state loop")
        self.model = model
        self.cfg = cfg
        self.lib = _hip.load()
        self.chunks: List[_Chunk] = []
        self._packed = {}
        self._unfinished = False    # packed copies whose kernels may still run
        self._gstream = None
        self._gstreams = []

    # ------------------------------------------------------------------
    def _pack(self, w: torch.Tensor, place, derived: bool = False) -> torch.Tensor:
        """MFMA-fragment-ordered copy of the (N,K) bf16 weight at `place` in the model, rebuilt only when the weight changes.
        The entry holds the storage that it was made from: while it is there no other tensor can come to lie at the address
        it is recognised by.  derived: w is itself a copy that its module forms anew when the parameter changes and that
        nothing writes to afterwards, so its address alone tells it (one formed under torch.inference_mode() has no counter of
        its changes)."""
        hit, made_from = self._packed.get(place), (0 if derived else w._version, w.data_ptr())
        if hit is None or hit[0] != made_from:
            hit = (made_from, _hip.pack_rows(w), w.detach())
            self._packed[place] = hit
            self._unfinished = True
        return hit[1]

    @property
    def desc(self) -> ModelDesc:
        """Descriptor of the first row chunk (the whole batch when B <= 16)."""
        return self.chunks[0].desc

    @property
    def logits(self) -> torch.Tensor:
        """(B,V) logits of the last eager step."""
        return self.chunks[0].logits if len(self.chunks) == 1 else torch.cat([c.logits for c in self.chunks], 0)

    def _build(self, caches, B: int, total_len: int):
        cfg = self.cfg
        d = cfg.n_embd
        mode = cfg.resolved_stu_decode_mode()
        caches = list(caches)
        if mode != "lds":                      # history buffers must hold the whole generation
            for i, layer in enumerate(self.model.layers):
                if isinstance(layer, STULayer):
                    hist, state, pos = caches[i]
                    if hist.shape[1] < total_len:
                        bigger = hist.new_zeros(B, total_len, d)
                        bigger[:, : hist.shape[1]] = hist
                        caches[i] = (bigger, state, pos)
        self.graph_end()
        self.chunks = []
        R = _hip.MAX_DECODE_ROWS
        # Rows are stepped in chunks of up to 16 (the width of the skinny decode kernels), each chunk re-reading the
        # weights.  A chunk of 17..32 rows instead runs its MLP, nearly all of the weight bytes, once over all rows on the
        # tiled GEMM kernel (bf16, recurrence STU state).
        wide = (cfg.torch_dtype == torch.bfloat16 and mode == "lds" and d % 256 == 0 and (d * cfg.mlp_scale) % 64 == 0)
        b0 = 0
        while b0 < B:
            rows = min(B - b0, 2 * R if (wide and B - b0 > R) else R)
            ch = _Chunk(b0, b0 + rows)
            self._build_chunk(ch, caches)
            self.chunks.append(ch)
            b0 += rows
        if self._unfinished:        # the copies outlive this call: a later one may read them on another stream
            torch.cuda.current_stream().synchronize()
            self._unfinished = False
        return tuple(caches)

    def _build_chunk(self, ch: _Chunk, caches):
        model, cfg = self.model, self.cfg
        dev = model.lm_head.weight.device
        dt = cfg.torch_dtype
        d, I, V = cfg.n_embd, cfg.n_embd * cfg.mlp_scale, cfg.vocab_size
        mode = cfg.resolved_stu_decode_mode()
        b0, b1 = ch.b0, ch.b1
        B = b1 - b0
        n = len(model.layers)

        def keep(t):
            ch.keep.append(t)
            return t

        def ptr(t):      # held as long as the descriptor: a parametrized weight is a temporary of this access
            return keep(t).data_ptr()
        arr = (LayerDesc * n)()
        hist_cap = 0
        fir_taps = 0
        weights = []        # the projections of each layer, read once
        for i, layer in enumerate(model.layers):
            ld = arr[i]
            gate, up, down = (keep(p.weight) for p in (layer.mlp.gate_proj, layer.mlp.up_proj, layer.mlp.down_proj))
            weights.append(dict(gate=gate, up=up, down=down))
            ld.w_gate, ld.w_up, ld.w_down = gate.data_ptr(), up.data_ptr(), down.data_ptr()
            ld.mlp_norm_w = ptr(layer.mlp_norm.weight)
            if isinstance(layer, STULayer):
                stu = layer.stu
                ld.kind = 0
                ld.norm1_w = ptr(layer.stu_norm.weight)
                mit = keep(stu.m_inputs_t())
                weights[i]["m_inputs"] = mit
                ld.m_inputs_t = mit.data_ptr()
                hist, state, pos = caches[i]
                if mode == "lds":
                    a, ce, co = stu.lds_params()
                    st = state[b0:b1]
                    keep(a), keep(ce), keep(co), keep(st)
                    ld.lds_a, ld.lds_ce, ld.lds_co, ld.lds_state = a.data_ptr(), ce.data_ptr(), co.data_ptr(), st.data_ptr()
                    fir = stu.lds_fir()
                    if fir is not None and hist.shape[1] == fir.shape[0]:
                        ring = hist[b0:b1]       # in lds mode the history slot of the cache entry is the ring of the last inputs
                        keep(fir), keep(ring)
                        ld.lds_ring, ld.lds_fir = ring.data_ptr(), fir.data_ptr()
                        fir_taps = fir.shape[0]
                    if B > _hip.MAX_DECODE_ROWS and dt == torch.bfloat16 and not cfg.use_hankel_L:
                        # 17..32 rows: the odd-lag sum is handed from step to step, so a step reads one bank only;
                        # primed here for the first decode position from the state and ring the prompt left
                        oc = _hip.stu_step_lds_prime(st, a, co, int(pos[0]) - 1, dt,
                                                     ring=hist[b0:b1] if ld.lds_ring else None, fir=fir if ld.lds_ring else None)
                        keep(oc)
                        ld.lds_ocache = oc.data_ptr()
                else:
                    hs = hist[b0:b1]
                    if hist_cap and hs.shape[1] != hist_cap:
                        raise RuntimeError("STU histories must share one capacity")
                    hist_cap = hs.shape[1]
                    filt = stu.effective_filter()
                    keep(filt), keep(hs)
                    ld.filt, ld.hist = filt.data_ptr(), hs.data_ptr()
            elif isinstance(layer, AttentionLayer):
                att = layer.attn
                ld.kind = 1
                ld.norm1_w = ptr(layer.attn_norm.weight)
                qkv, proj = keep(att.c_attn.weight), keep(att.c_proj.weight)
                weights[i].update(qkv=qkv, proj=proj)
                ld.w_qkv, ld.w_proj = qkv.data_ptr(), proj.data_ptr()
                kr, vr, pos = caches[i]
                kr, vr = kr[b0:b1], vr[b0:b1]
                keep(kr), keep(vr)
                ld.kring, ld.vring = kr.data_ptr(), vr.data_ptr()
                ld.slopes = ptr(att.alibi_slopes)
            else:
                raise TypeError(type(layer))
        m = ModelDesc()
        m.dtype = _hip.FSTU_BF16 if dt == torch.bfloat16 else _hip.FSTU_F32
        m.B, m.d, m.I, m.V, m.n_layers = B, d, I, V, n
        m.n_heads, m.head_dim = cfg.n_heads, d // cfg.n_heads
        m.window, m.kv_cap = cfg.window_left, cfg.window_left + 1
        m.L, m.hist_cap = cfg.seq_len, hist_cap
        m.stu_mode = 1 if mode == "lds" else 0
        m.lds_S = cfg.stu_lds_state_dim
        m.lds_fir_taps = fir_taps
        m.single_branch = int(cfg.use_hankel_L)
        m.ksplit_down = pick_ksplit_down(I) if dt == torch.bfloat16 else min(8, max(1, I // 512))
        m.hist_nsplit_max = self.HIST_NSPLIT_MAX
        m.row0 = b0
        m.eps, m.softcap = float(cfg.rms_norm_eps), float(cfg.softcap or 0.0)
        emb = keep(model.lm_head.weight)
        m.emb, m.final_norm_w = emb.data_ptr(), ptr(model.norm.weight)
        m.layers = ctypes.cast(arr, ctypes.POINTER(LayerDesc))

        ch.logits = keep(torch.zeros(B, V, dtype=dt, device=dev))
        m.logits = ch.logits.data_ptr()
        # the other workspaces in one piece, cleared by one launch: rows of d in the model's dtype, the others by their bytes
        esz = ch.logits.element_size()
        sizes = dict(x=B * d * esz, h=B * d * esz, qkv=3 * B * d * esz, attn=B * d * esz, act=B * I * esz, xp=B * d * esz, y=B * d * esz,
                     x2=B * d * esz,             # the stream behind the norms that a projection forms itself
                     partial=max(m.ksplit_down, 16) * B * d * 4, eo=self.HIST_NSPLIT_MAX * 2 * B * d * 4, best=32 * 64 * 8,
                     samp_ws=int(self.lib.fstu_sample_ws_bytes()))
        at = keep(torch.zeros(sum(-(-n // 256) * 256 for n in sizes.values()), dtype=torch.uint8, device=dev)).data_ptr()
        place = {}
        for name, size in sizes.items():
            place[name] = at
            at += -(-size // 256) * 256
        for name in sizes:
            if name != "x2" or dt == torch.float32:
                setattr(m, name, place[name])
        if dt == torch.bfloat16 and self.lib.fstu_glu_packed_supported(B, d, I):
            # gate/up projection over packed weights, one workgroup per CU with equal bytes each
            for i, (ld, w) in enumerate(zip(arr, weights)):
                ld.wp_gate, ld.wp_up = ptr(self._pack(w["gate"], (i, "gate"))), ptr(self._pack(w["up"], (i, "up")))
            m.glu_packed = 1
            if I % 512 == 0 and d % 16 == 0:
                for i, (ld, w) in enumerate(zip(arr, weights)):
                    ld.wp_down = ptr(self._pack(w["down"], (i, "down")))
                m.down_packed = 1
            if B * (d + 8) * 2 <= 96 * 1024:
                m.x2 = place["x2"]              # second residual buffer: the MLP norm runs as the gate/up prologue
                if mode == "lds" and d % 256 == 0 and m.down_packed and B * (d // 8) <= 1024 and I % 128 == 0:
                    # the add+norm between two layers runs as the prologue of the next layer's first projection
                    # (the down projection leaves 4 split-K slices for it): one launch less per layer
                    for i, (ld, w) in enumerate(zip(arr, weights)):
                        if "qkv" in w:
                            ld.wp_qkv = ptr(self._pack(w["qkv"], (i, "qkv")))
                    m.merge_norm = 1
        if dt == torch.bfloat16 and self.lib.fstu_mlp_packed_rows32_supported(B, d, I):
            # 17..32 rows: the MLP streams packed weights as two row tiles per weight fragment
            for i, (ld, w) in enumerate(zip(arr, weights)):
                ld.wp_gate, ld.wp_up, ld.wp_down = (ptr(self._pack(w[k], (i, k))) for k in ("gate", "up", "down"))
                if "qkv" in w:
                    ld.wp_qkv, ld.wp_proj = ptr(self._pack(w["qkv"], (i, "qkv"))), ptr(self._pack(w["proj"], (i, "proj")))
                elif mode == "lds":
                    ld.wp_m_inputs = ptr(self._pack(w["m_inputs"], (i, "m_inputs"), derived=True))
        if dt == torch.bfloat16 and self.lib.fstu_glu_packed_supported(min(B, _hip.MAX_DECODE_ROWS), d, V):
            m.wp_emb = ptr(self._pack(emb, "emb"))      # the head streams a packed copy of the embedding
        ch.arr, ch.desc = arr, m
        if B > _hip.MAX_DECODE_ROWS:
            # first use of the tiled kernels outside any graph capture (their launch set-up raises an LDS limit once)
            wx = torch.zeros(B, 64, dtype=dt, device=dev)
            ww = torch.zeros(8, 64, dtype=dt, device=dev)
            _hip.gemm(wx, ww, up_weight=ww)
            _hip.gemm_splitk(wx, ww, 1)

    # ------------------------------------------------------------------ eager steps
    def steps(self, tokens: torch.Tensor, pos: int, n: int, temperature, top_k, top_p, do_sample, seed, step_idx):
        """n steps of every chunk: the first feeds tokens[:, pos], each writes the token that the next one feeds."""
        stride = tokens.stride(0)
        for ch in self.chunks:
            rc = self.lib.fstu_decode_steps(ctypes.byref(ch.desc), tokens.data_ptr() + 8 * (ch.b0 * stride + pos), stride, pos, int(n),
                                            float(temperature), int(top_k) if top_k else 0, float(top_p) if top_p else 0.0,
                                            int(bool(do_sample)), int(seed) & ((1 << 64) - 1), int(step_idx),
                                            torch.cuda.current_stream().cuda_stream)
            _hip._check(rc, "fstu_decode_steps")

    def step(self, tokens: torch.Tensor, pos: int, temperature, top_k, top_p, do_sample, seed, step_idx):
        """Feeds tokens[:, pos], writes the sampled id to tokens[:, pos+1]."""
        stride = tokens.stride(0)
        for ch in self.chunks:
            base = tokens.data_ptr() + 8 * (ch.b0 * stride + pos)
            rc = self.lib.fstu_decode_step(ctypes.byref(ch.desc), base, base + 8, stride, pos, float(temperature),
                                           int(top_k) if top_k else 0, float(top_p) if top_p else 0.0,
                                           int(bool(do_sample)), int(seed) & ((1 << 64) - 1), int(step_idx),
                                           torch.cuda.current_stream().cuda_stream)
            _hip._check(rc, "fstu_decode_step")

    # ------------------------------------------------------------------ graph replay
    def graph_supported(self) -> bool:
        return self.cfg.resolved_stu_decode_mode() == "lds"

    GRAPH_STEPS = 8     # decode steps per graph launch in generate() (the launch of a graph costs several microseconds)

    def graph_begin(self, tokens: torch.Tensor, pos: int, step_idx: int, temperature, top_k, top_p, do_sample, seed,
                    steps_per_graph: int = 1, keep: bool = False):
        """Captures steps_per_graph decode steps per row chunk as a HIP graph, each chunk on a side stream of its own: the
        chunks are independent (own workspaces, state rows and device-side position), so their graphs run concurrently
        and the second chunk finds the layer's weights, which the first has just streamed, in the Infinity Cache.  Each
        graph_step() then runs steps_per_graph decode steps: each feeds tokens[:, pos], writes tokens[:, pos+1] and
        advances pos on the device.  `pos` is the position the first launch of THIS graph will process.  keep=True adds
        the graph to those already captured (same tokens, sampling arguments and device-side counters) instead of
        replacing them: a run can then mix long graphs with single-step ones (graph_step(n), graph_seek)."""
        if not keep:
            self.graph_end()
        n = int(steps_per_graph)
        self.graph_steps = n
        n_streams = len(self.chunks)
        if not self._gstreams:
            self._gstreams = [torch.cuda.Stream(device=tokens.device) for _ in range(n_streams)]
        stride = tokens.stride(0)
        for ch in self.chunks:
            if ch.dyn is None:
                # filled by kernels: a copy from the host would wait for everything launched so far
                ch.dyn = torch.full((2,), pos, dtype=torch.int32, device=tokens.device)
                ch.dyn[1:].fill_(step_idx)
        for st in self._gstreams:
            st.wait_stream(torch.cuda.current_stream())
        for i, ch in enumerate(self.chunks):
            handle = _vp()
            ch.stream = self._gstreams[i % len(self._gstreams)]
            rc = self.lib.fstu_decode_graph_create(ctypes.byref(ch.desc), tokens.data_ptr() + 8 * ch.b0 * stride, stride,
                                                   ch.dyn.data_ptr(), int(pos), n, float(temperature),
                                                   int(top_k) if top_k else 0,
                                                   float(top_p) if top_p else 0.0, int(bool(do_sample)),
                                                   int(seed) & ((1 << 64) - 1), ch.stream.cuda_stream,
                                                   ctypes.byref(handle))
            _hip._check(rc, "fstu_decode_graph_create")
            ch.graphs[n] = handle
        self._graph_tokens = tokens

    def graph_step(self, steps_per_graph: Optional[int] = None):
        n = self.graph_steps if steps_per_graph is None else int(steps_per_graph)
        for ch in self.chunks:
            _hip._check(self.lib.fstu_decode_graph_launch(ch.graphs[n], ch.stream.cuda_stream), "fstu_decode_graph_launch")

    def graph_seek(self, steps_per_graph: int, pos: int):
        """Tells the graph of that length which position its next launch will process (needed after graphs of another
        length have advanced the device-side position in between)."""
        for ch in self.chunks:
            _hip._check(self.lib.fstu_decode_graph_seek(ch.graphs[int(steps_per_graph)], int(pos)), "fstu_decode_graph_seek")

    def graph_sync(self):
        """Blocks until every chunk's replay stream has drained."""
        for st in self._gstreams:
            st.synchronize()

    def graph_end(self):
        live = [ch for ch in self.chunks if ch.graphs]
        if live:
            for st in self._gstreams:
                torch.cuda.current_stream().wait_stream(st)
                st.synchronize()
            for ch in live:
                for handle in ch.graphs.values():
                    self.lib.fstu_decode_graph_destroy(handle)
                ch.graphs = {}
        for ch in self.chunks:
            ch.dyn = None
        self._gstreams = []

    # ------------------------------------------------------------------
    @_hip.inference
    def prefill(self, input_ids: torch.Tensor, total_len: int):
        """Runs the prompt through the module path with caches, returns the
        logits of the last position (B,V) and prepares the step descriptors."""
        model = self.model
        B, P = input_ids.shape
        x = model._embed(input_ids.contiguous())
        x, caches = model._run_layers(x, None, True, None)
        xn = model.norm(x[:, -1:, :].contiguous())
        logits = model._head(xn)[:, 0, :].contiguous()
        self.caches = self._build(caches, B, total_len)
        return logits

    @_hip.inference
    def generate(self, input_ids: torch.Tensor, n_new: int, temperature=1.0, top_k=None, top_p=None, do_sample=True,
                 seed: int = 0, return_logits: bool = False, use_graph: bool = True):
        if not input_ids.is_cuda:
            raise _hip.FlashSTUHipError("input_ids must be on the GPU: this model has no CPU path")
        B, P = input_ids.shape
        total = P + n_new
        if total > self.cfg.seq_len:
            # the history ends there, and the recurrence state would carry a tail the filters (zero from lag seq_len
            # on) do not have; FlashSTU.generate routes such calls to the recompute loop
            raise ValueError(f"stateful decode needs prompt+new tokens ({total}) <= seq_len ({self.cfg.seq_len})")
        tokens = torch.zeros(B, total, dtype=torch.int64, device=input_ids.device)
        tokens[:, :P] = input_ids
        logits = self.prefill(input_ids, total)
        _hip.sample(logits, tokens[:, P], temperature, top_k, top_p, do_sample, seed, 0)
        all_logits = [logits.clone()] if return_logits else None
        # One chunk of rows: the steps are launched one by one.  The host enqueues a step (50 launches) in 0.15 ms, the GPU
        # takes 0.3 ms for it, so nothing waits, and a graph gives nothing back for its capture and the gaps between its
        # replays.  ms for the whole call, graphs of 8 steps / step by step: 768-d, 128 tokens, 8 rows 48.9 / 41.7, 16 rows
        # with top-k 53.1 / 44.9, 64 tokens, 1 row 23.0 / 19.3, 32 rows 33.5 / 28.9; 2048-d 32 rows 57.5 / 54.5; 128-d, 2
        # layers 8.4 / 7.6.  Several chunks replay graphs on a stream each, side by side, from the first step on: 768-d, 64
        # rows, 24 tokens 18.3 / 21.4, 96 rows, 32 tokens 29.1 / 41.8, 33 rows, 3 tokens 4.8 either way.
        if use_graph and not return_logits and self.graph_supported() and len(self.chunks) > 1 and n_new > 2:
            todo, pos, S = n_new - 1, P, self.GRAPH_STEPS
            try:
                if todo >= 4 * S:       # long runs: S steps per graph launch, the remainder one by one
                    self.graph_begin(tokens, pos, pos - P + 1, temperature, top_k, top_p, do_sample, seed, steps_per_graph=S)
                    for _ in range(todo // S):
                        self.graph_step()
                    pos += (todo // S) * S
                    todo -= (todo // S) * S
                if todo > 0:
                    self.graph_begin(tokens, pos, pos - P + 1, temperature, top_k, top_p, do_sample, seed)
                    for _ in range(todo):
                        self.graph_step()
            finally:
                self.graph_end()
            return tokens
        if not return_logits:
            self.steps(tokens, P, n_new - 1, temperature, top_k, top_p, do_sample, seed, 1)
            return tokens
        for s in range(1, n_new):
            self.step(tokens, P + s - 1, temperature, top_k, top_p, do_sample, seed, s)
            all_logits.append(self.logits.clone())
        return tokens, torch.stack(all_logits, 1)
