"""Monarch attention operators with the reference's call signatures.

    monarch_attn_with_kv_cache  <->  wan/modules/monarch_attn.py:1778-1796
    monarch_attn                <->  wan/modules/monarch_attn.py:1753-1776

Inputs are [B, S, H, D] CUDA tensors (bf16 / fp16 / fp32, head_dim contiguous) in token order;
the KV cache holds rows in Monarch block order and is updated in place.  Under autograd the operators
are torch.autograd.Functions whose backward runs the library's backward kernels (num_iters == 1).
num_iters > 1 runs the alternating refinement the reference implements in pure torch
(monarch_attn_slow, wan/modules/monarch_attn.py:1705-1751) as HIP kernels; under autograd its forward is still the HIP
kernels and its backward differentiates a torch restatement of the passes on the GPU (the reference's own refinement is
differentiable torch and has no backward kernels either).
"""
import contextlib
import ctypes as C
import threading
import weakref

import torch

from . import lib as _l

_DT = {torch.bfloat16: _l.SFM_BF16, torch.float16: _l.SFM_F16, torch.float32: _l.SFM_F32}


def _check4(name, t, dtype=None, device=None):
    if not isinstance(t, torch.Tensor) or t.dim() != 4:
        raise ValueError(f"{name} must be a [B, S, H, D] tensor")
    if not t.is_cuda:
        raise ValueError(f"{name} must live on the GPU")
    if t.stride(3) != 1:
        raise ValueError(f"{name}: head_dim must be contiguous")
    if dtype is not None and t.dtype != dtype:
        raise ValueError(f"{name}: dtype {t.dtype} differs from q's {dtype}")
    if device is not None and t.device != device:
        raise ValueError(f"{name}: device {t.device} differs from q's {device}")


def _desc(q, k, v, out, f_tied, h_reduce, w_reduce, h, w, sm_scale, kv_block_order, causal_block_frames, num_iters=1,
          one_kernel=False):
    if q.dtype not in _DT:
        raise ValueError(f"unsupported dtype {q.dtype}")
    B, q_tokens, H, D = q.shape
    # all fields in one call: one by one they take twice as long, a seventh of a small call's host time
    return _l.MonarchDesc(_DT[q.dtype], B, H, D, q_tokens, k.shape[1], (f_tied, h_reduce, w_reduce, h, w), kv_block_order,
                          causal_block_frames, float(sm_scale), int(num_iters), _l.SFM_MONARCH_ONE_KERNEL if one_kernel else 0,
                          q.stride()[:3], k.stride()[:3], v.stride()[:3], out.stride()[:3])


_raw_stream = torch._C._cuda_getCurrentRawStream      # torch.cuda.current_stream(device).cuda_stream without the Stream object
_HERE = contextlib.nullcontext()


def _on_device(device):
    """torch.cuda.device(device), or nothing where it is the current device already."""
    return _HERE if torch.cuda.current_device() == device.index else torch.cuda.device(device)


_SCRATCH = {}


def scratch(nbytes, device):
    """The library's workspace for a call on `device`'s current stream: one grow-only byte buffer per (device, stream),
    so that steady-state calls allocate nothing (a caller recording a HIP graph warms the buffer up with one eager
    call first).  Calls on one stream are ordered, so they can share it; `release_scratch()` gives the memory back."""
    index = device.index if device.index is not None else torch.cuda.current_device()
    key = (index, _raw_stream(index))
    buf = _SCRATCH.get(key)
    if buf is None or buf.numel() < nbytes:
        _drop_kept(index)
        buf = _SCRATCH[key] = torch.empty(max(int(nbytes), 1), dtype=torch.uint8, device=device)
    return buf


def release_scratch():
    _SCRATCH.clear()


class _Kept:
    """What one forward left for its backward, until that takes it, another call has it dropped or its graph dies."""
    __slots__ = ("buf", "budget", "__weakref__")

    def __init__(self, buf, budget):
        self.buf, self.budget = buf, budget

    def __del__(self):
        if self.buf is not None:
            self.budget.graph_died(self)


class _KeptBudget:
    """What the forwards of one device hold for backwards to come: the newest one's intermediates, 2 GiB at most.  The workspace of a
    backward that finds them is smaller by as much, so a program that calls forward and backward in turn has no more memory
    in use than if every backward formed them again (12 heads at 480p, three frames against 21: 769 + 760 MB, else 1500 and 29
    of dq in float32).  They are dropped, and their backward forms them again, for the next forward's, for a backward that has
    none and needs the larger workspace, and where a workspace grows.

    To leave them costs a forward 10 % (12 heads at 480p, 21 frames: 291 us without, 320), lost where no backward takes them: an
    evaluation with gradients on, several layers in front of their backwards.  After two in a row that nothing took, forwards
    leave nothing until a backward comes that would have found its own."""

    def __init__(self):
        self.left = 2 << 30                      # sfm_monarch_kept_bytes never asks for more
        self.lock = threading.RLock()            # a _Kept may die inside any of these, in the garbage collector
        self.pending = None                      # the one _Kept with a buffer, weakly: it dies with its graph
        self.unused = 0                          # that no backward took, since one did
        self.turn = 0                            # what a forward leaves, or would have left, is there until the next turn

    def take(self, nbytes, device):
        if nbytes > self.left:
            return None
        try:
            return torch.empty(nbytes, dtype=torch.uint8, device=device)
        except torch.OutOfMemoryError:
            return None

    def hold(self, buf):
        kept = _Kept(buf, self)
        with self.lock:
            if self.pending is not None:         # of another thread, since this one's forward began
                self.drop()
            self.left -= buf.numel()
            self.pending = weakref.ref(kept)
        return kept

    def _release(self, kept):
        """The buffer that `kept` no longer holds (with the lock)."""
        buf, kept.buf = kept.buf, None
        if buf is not None:
            self.left += buf.numel()
            self.pending = None
        return buf

    def claim(self, kept):
        """The buffer, for one backward: from here on nobody drops it, and it dies with its last use."""
        with self.lock:
            buf = self._release(kept)
            if buf is not None:
                self.unused = 0
        return buf

    def graph_died(self, kept):
        with self.lock:
            if self._release(kept) is not None:
                self.unused += 1

    def missed(self, turn):
        """A backward whose forward left nothing: would it be there?"""
        if turn == self.turn:
            self.unused = 0

    def drop(self):
        self.turn += 1                           # one lost to another thread costs a forward that leaves something for nobody
        if self.pending is None:
            return
        with self.lock:
            kept = self.pending and self.pending()
            if kept is not None and self._release(kept) is not None:
                self.unused += 1


_KEPT = {}
_top_hooks = getattr(torch._C._autograd, "_top_saved_tensors_default_hooks", None)


def _kept_buffer(desc, device):
    """A buffer for the intermediates of a forward under autograd, or None.  None too while hooks on saved tensors are set: their
    program wants little memory between forward and backward (activation checkpointing, save_on_cpu)."""
    budget = _KEPT.get(device.index)
    if budget is None:
        budget = _KEPT.setdefault(device.index, _KeptBudget())
    budget.drop()
    if budget.unused > 1 or _top_hooks is None or _top_hooks(False) is not None:
        return None
    n = C.c_size_t(0)
    _l.check(_l.load().sfm_monarch_kept_bytes(C.byref(desc), C.byref(n)))
    return budget.take(n.value, device) if n.value else None


def _drop_kept(index):
    """Every call that writes cache rows makes this one too (where anything was ever kept: its cost is 0.3 of the smallest call's 18 us): a backward takes K and V from the caches as it finds them, and with rows
    written since its forward it has to form the right factor from those too, not from the ones that the forward saw.  (A replayed
    graph makes no call: rows that it writes reach K and V alone.)"""
    if index in _KEPT:
        _KEPT[index].drop()


def monarch_workspace_bytes(desc, heads_per_pass=0):
    n = C.c_size_t(0)
    _l.check(_l.load().sfm_monarch_workspace_bytes(C.byref(desc), heads_per_pass, C.byref(n)))
    return n.value


def _stream(t):
    return C.c_void_p(_raw_stream(t.device.index))


def _from_block_order(x, f_tied, h_reduce, w_reduce, h, w):
    """Inverse of the reference's rearrangement (monarch_attn.py:1696-1703) on a [B, n, H, D] tensor."""
    if f_tied == 1 and h_reduce == 1 and w_reduce == 1:
        return x
    B, n, H, D = x.shape
    x = x.reshape(B, -1, h_reduce, w_reduce, f_tied, h // h_reduce, w // w_reduce, H, D)
    return x.permute(0, 1, 4, 2, 5, 3, 6, 7, 8).reshape(B, n, H, D)


def _causal_block_frames(q, k, tiling, block_causal_size, num_iters=1):
    """Block-causal size in tokens -> block-frames, with the reference's checks (monarch_attn.py:1485-1491)."""
    if block_causal_size is None:
        return 0
    f_tied, h_reduce, w_reduce, h, w = tiling
    per_block = f_tied * (h // h_reduce) * (w // w_reduce)
    if q.shape[1] % block_causal_size:
        raise ValueError(f"block_causal_size ({block_causal_size}) must divide sequence length ({q.shape[1]})")
    if k.shape[1] != q.shape[1]:
        raise ValueError("causal attention needs kv length equal to q length")
    if block_causal_size % per_block:
        raise ValueError("block_causal_size must align with Monarch block sizes")
    if num_iters != 1:
        raise ValueError("causal currently only supported for num_iters=1")
    return block_causal_size // per_block


def kv_cache_write(new_k, new_v, k_cache, v_cache, start_idx, end_idx, f_tied, h_reduce, w_reduce, h, w):
    """new_k / new_v (token order) into k_cache / v_cache[:, start_idx:end_idx] in Monarch block order
    (monarch_attn.py:1784-1785, 1230-1231)."""
    if new_k.stride() != new_v.stride():
        new_k, new_v = new_k.contiguous(), new_v.contiguous()
    if k_cache.stride() != v_cache.stride():
        raise ValueError("k_cache and v_cache must share their strides")
    B, _, H, D = new_k.shape
    if B > k_cache.shape[0] or H > k_cache.shape[2] or D > k_cache.shape[3]:
        raise ValueError(f"new_k {tuple(new_k.shape)} holds more batches, heads or channels than the cache {tuple(k_cache.shape)}")
    if _KEPT:
        _drop_kept(k_cache.device.index)
    with _on_device(new_k.device):
        _l.check(_l.load().sfm_kv_cache_write(_DT[new_k.dtype], B, H, D, C.byref(_l.Tiling(f_tied, h_reduce, w_reduce, h, w)),
                                              new_k.data_ptr(), new_v.data_ptr(), _l.strides3(new_k), k_cache.data_ptr(),
                                              v_cache.data_ptr(), _l.strides3(k_cache), k_cache.shape[1], start_idx, end_idx,
                                              _stream(new_k)))


def _like_q(q, new_k):
    """The operators with a cache write take the new chunk's batches, heads and head_dim from q.  A chunk of other sizes is
    written by itself (kv_cache_write takes them from the chunk)."""
    n, s = new_k.shape, q.shape
    return n[0] == s[0] and n[2] == s[2] and n[3] == s[3]


def _monarch_fwd_stats(q, k, v, tiling, sm_scale, kv_block_order, cbf, heads_per_pass=0, new=None):
    """Forward for autograd, with new = (new_k, new_v, start_idx, end_idx) of the KV-cache operator: returns (out, stats)
    where stats is the opaque row-statistics tensor that sfm_monarch_bwd_saved takes, or None when the forward that runs for
    these tensors produces none (the reference's forward keeps z and z_lse the same way, monarch_attn.py:1309-1317)."""
    return _monarch_fwd_kept(q, k, v, tiling, sm_scale, kv_block_order, cbf, heads_per_pass, new, keep=False)[:2]


def _monarch_fwd_kept(q, k, v, tiling, sm_scale, kv_block_order, cbf, heads_per_pass=0, new=None, keep=True):
    """_monarch_fwd_stats that returns (out, stats, kept): kept is the scratch of a forward whose intermediates
    sfm_monarch_bwd_kept takes, or None (a bound on the heads of a pass bounds the scratch, which is then not held).  Forward and
    backward of 12 heads at 480p, three frames against 21 (766 MB kept): 1159 us with step 1 run again by the backward, 976 so; a
    block-causal clip of nine frames, three tied, 620 and 534."""
    out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
    d = _desc(q, k, v, out, *tiling, sm_scale, kv_block_order, cbf, 1)
    lib, n = _l.load(), C.c_size_t(0)
    _l.check(lib.sfm_monarch_stats_bytes(C.byref(d), C.byref(n)))
    stats = torch.empty(n.value // 4, dtype=torch.float32, device=q.device) if n.value else None
    kept = None
    if keep and stats is not None and not heads_per_pass:
        kept = _kept_buffer(d, q.device)
    elif new is not None and _KEPT:
        _drop_kept(q.device.index)
    if kept is not None:
        nbytes, ws = kept.numel(), kept
    else:
        nbytes = monarch_workspace_bytes(d, heads_per_pass)
        ws = scratch(nbytes, q.device)
    if new is not None and (stats is None or not _like_q(q, new[0])):
        kv_cache_write(*new[:2], k, v, *new[2:], *tiling)
        new = None
    with _on_device(q.device):
        if new is not None:
            new_k, new_v, start_idx, end_idx = new
            if new_k.stride() != new_v.stride():
                new_k, new_v = new_k.contiguous(), new_v.contiguous()
            if k.stride() != v.stride():
                raise ValueError("k_cache and v_cache must share their strides")
            fn = lib.sfm_monarch_attn_with_kv_cache_stats if kept is None else lib.sfm_monarch_attn_with_kv_cache_kept
            _l.check(fn(
                C.byref(d), q.data_ptr(), k.data_ptr(), v.data_ptr(), new_k.data_ptr(), new_v.data_ptr(), _l.strides3(new_k),
                start_idx, end_idx, out.data_ptr(), stats.data_ptr(), ws.data_ptr(), nbytes, _stream(q)))
        elif stats is None:
            _l.check(lib.sfm_monarch_fwd(C.byref(d), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                                         ws.data_ptr(), nbytes, _stream(q)))
        else:
            fn = lib.sfm_monarch_fwd_stats if kept is None else lib.sfm_monarch_fwd_kept
            _l.check(fn(C.byref(d), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), stats.data_ptr(), ws.data_ptr(), nbytes,
                        _stream(q)))
    return out, stats, kept


def _monarch_bwd(q, k, v, dout, tiling, sm_scale, kv_block_order, cbf, kv_f0=0, kv_f1=None, heads_per_pass=0, out=None,
                 stats=None, kept=None):
    """Raw call of sfm_monarch_bwd (or sfm_monarch_bwd_saved when the forward's `out` and `stats` are given, sfm_monarch_bwd_kept
    when its `kept` is too): returns (dq float32, with `kept` in q's dtype, dk, dv); dk, dv cover kv
    block-frames [kv_f0, kv_f1) in the row order of k."""
    f_tied, h_reduce, w_reduce, h, w = tiling
    per_frame = f_tied * (h // h_reduce) * (w // w_reduce)
    nf = k.shape[1] // per_frame
    if kv_f1 is None:
        kv_f1 = nf
    if dout.stride(3) != 1 or (out is not None and dout.stride() != out.stride()):
        dout = dout.contiguous()
    if out is not None and out.stride() != dout.stride():
        out = out.contiguous()
    dk = torch.empty((k.shape[0], (kv_f1 - kv_f0) * per_frame, k.shape[2], k.shape[3]), dtype=k.dtype, device=k.device)
    dv = torch.empty_like(dk)
    bd = _l.MonarchBwdDesc()
    bd.fwd = _desc(q, k, v, dout, f_tied, h_reduce, w_reduce, h, w, sm_scale, kv_block_order, cbf)
    bd.dkv_stride = _l.strides3(dk)
    bd.kv_grad_frame_start, bd.kv_grad_frame_end = kv_f0, kv_f1
    lib, n = _l.load(), C.c_size_t(0)
    if kept is not None:
        dq = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        bd.dq_stride = _l.strides3(dq)
        rc = lib.sfm_monarch_bwd_kept_workspace_bytes(C.byref(bd), C.byref(n))
        if rc == _l.SFM_ERR_UNSUPPORTED:         # the implementation switches were changed since the forward
            kept = None
        else:
            _l.check(rc)
    if kept is None:
        dq = torch.empty(q.shape, dtype=torch.float32, device=q.device)
        bd.dq_stride = _l.strides3(dq)
        _l.check(lib.sfm_monarch_bwd_workspace_bytes(C.byref(bd), heads_per_pass, C.byref(n)))
    ws = scratch(n.value, q.device)
    with _on_device(q.device):
        if kept is not None:
            _l.check(lib.sfm_monarch_bwd_kept(C.byref(bd), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                                              stats.data_ptr(), kept.data_ptr(), kept.numel(), dout.data_ptr(), dq.data_ptr(),
                                              dk.data_ptr(), dv.data_ptr(), ws.data_ptr(), n.value, _stream(q)))
        elif out is None or stats is None:
            _l.check(lib.sfm_monarch_bwd(C.byref(bd), q.data_ptr(), k.data_ptr(), v.data_ptr(), dout.data_ptr(), dq.data_ptr(),
                                         dk.data_ptr(), dv.data_ptr(), ws.data_ptr(), n.value, _stream(q)))
        else:
            _l.check(lib.sfm_monarch_bwd_saved(C.byref(bd), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                                               stats.data_ptr(), dout.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                                               ws.data_ptr(), n.value, _stream(q)))
    return dq, dk, dv


def _save(ctx, inputs, out, stats, kept):
    """The forward's tensors for the backward: the inputs, then the output and its row statistics if it left any.  `kept` is no saved
    tensor: it may be dropped before."""
    if stats is None:
        ctx.save_for_backward(*inputs)
    else:
        ctx.save_for_backward(*inputs, out, stats)
    budget = _KEPT.get(out.device.index)
    ctx.kept = None if kept is None else budget.hold(kept)
    ctx.turn = -1 if budget is None else budget.turn


def _saved(ctx):
    """(inputs, what _monarch_bwd takes of the forward's)."""
    q, k, v, *left = ctx.saved_tensors
    out, stats = left or (None, None)
    budget, kept = _KEPT.get(q.device.index), None
    if ctx.kept is not None:
        kept = ctx.kept.budget.claim(ctx.kept)
    elif budget is not None:
        budget.missed(ctx.turn)
    if kept is None and budget is not None:
        budget.drop()
    return (q, k, v), {"out": out, "stats": stats, "kept": kept}


class _MonarchFn(torch.autograd.Function):
    """monarch_attn under autograd (_attention_no_cache, monarch_attn.py:1472-1693)."""

    @staticmethod
    def forward(ctx, q, k, v, tiling, sm_scale, block_causal_size, heads_per_pass, kv_block_order):
        cbf = _causal_block_frames(q, k, tiling, block_causal_size)
        _check4("q", q)
        _check4("k", k, q.dtype, q.device)
        _check4("v", v, q.dtype, q.device)
        if k.stride() != v.stride():
            k, v = k.contiguous(), v.contiguous()
        out, *kept = _monarch_fwd_kept(q, k, v, tiling, sm_scale, 1 if kv_block_order else 0, cbf, heads_per_pass)
        _save(ctx, (q, k, v), out, *kept)
        ctx.cfg = (tiling, sm_scale, cbf, kv_block_order)
        return out

    @staticmethod
    def backward(ctx, dout):
        (q, k, v), left = _saved(ctx)
        tiling, sm_scale, cbf, kv_block_order = ctx.cfg
        dq, dk, dv = _monarch_bwd(q, k, v, dout, tiling, sm_scale, 1 if kv_block_order else 0, cbf, **left)
        return dq.to(q.dtype), dk, dv, None, None, None, None, None


class _MonarchCacheFn(torch.autograd.Function):
    """monarch_attn_with_kv_cache under autograd (_attention_with_cache, monarch_attn.py:1225-1470): the caches
    are written in place in the forward and saved by reference, as the reference does; with grad_only_new_kv
    only the block-frames written by this call get K/V gradients (:1364-1374).  Rows that another call writes before the
    backward are what it computes with, right factor included (_drop_kept); the output and its statistics are the forward's."""

    @staticmethod
    def forward(ctx, q, k_cache, v_cache, new_k, new_v, start_idx, end_idx, tiling, sm_scale, grad_only_new_kv,
                heads_per_pass):
        _check4("q", q)
        for name, t in (("k_cache", k_cache), ("v_cache", v_cache), ("new_k", new_k), ("new_v", new_v)):
            _check4(name, t, q.dtype, q.device)
        if k_cache.shape != v_cache.shape or new_k.shape != new_v.shape:
            raise ValueError("k/v shapes differ")
        if new_k.shape[1] != end_idx - start_idx:
            raise ValueError(f"new_k holds {new_k.shape[1]} tokens but end_idx - start_idx = {end_idx - start_idx}")
        out, *kept = _monarch_fwd_kept(q, k_cache, v_cache, tiling, sm_scale, 1, 0, heads_per_pass,
                                       new=(new_k, new_v, start_idx, end_idx))
        _save(ctx, (q, k_cache, v_cache), out, *kept)
        ctx.cfg = (start_idx, end_idx, tiling, sm_scale, grad_only_new_kv)
        return out

    @staticmethod
    def backward(ctx, dout):
        (q, k_cache, v_cache), left = _saved(ctx)
        start_idx, end_idx, tiling, sm_scale, grad_only_new_kv = ctx.cfg
        f_tied, h_reduce, w_reduce, h, w = tiling
        per_frame = f_tied * (h // h_reduce) * (w // w_reduce)
        if grad_only_new_kv:
            dq, dk, dv = _monarch_bwd(q, k_cache, v_cache, dout, tiling, sm_scale, 1, 0, start_idx // per_frame,
                                      end_idx // per_frame, **left)
            dk_cache = dv_cache = None
            dk_new, dv_new = dk, dv
        else:
            dq, dk_cache, dv_cache = _monarch_bwd(q, k_cache, v_cache, dout, tiling, sm_scale, 1, 0, **left)
            dk_new, dv_new = dk_cache[:, start_idx:end_idx], dv_cache[:, start_idx:end_idx]
        dk_new = _from_block_order(dk_new, *tiling)
        dv_new = _from_block_order(dv_new, *tiling)
        return dq.to(q.dtype), dk_cache, dv_cache, dk_new, dv_new, None, None, None, None, None, None


def _to_block_order(x, f_tied, h_reduce, w_reduce, h, w):
    """The reference's rearrangement (monarch_attn.py:1696-1703) of a token-order [B, n, H, D] tensor: rows in Monarch
    block order."""
    if f_tied == 1 and h_reduce == 1 and w_reduce == 1:
        return x
    B, n, H, D = x.shape
    x = x.reshape(B, -1, f_tied, h_reduce, h // h_reduce, w_reduce, w // w_reduce, H, D)
    return x.permute(0, 1, 3, 5, 2, 4, 6, 7, 8).reshape(B, n, H, D)


def _refinement_torch(qb, kb, vb, sm_scale, num_iters):
    """The refinement passes (monarch_attn.py:1705-1751) as differentiable torch ops on block-ordered tensors
    qb [B, a, b1, b2, H, D], kb / vb [B, f, b1, b2, H, D]; used for gradients only.  Pass p forms the right factor R from
    the per-block query representatives of pass p - 1 (first pass: the queries themselves, weight 1), then the left
    factor L; the last pass's factors are applied to V."""
    rs = float(sm_scale) ** 0.5
    q = qb.permute(0, 4, 1, 2, 3, 5) * rs                 # [B, H, a, i, j, D]
    k = kb.permute(0, 4, 1, 2, 3, 5) * rs                 # [B, H, f, k, l, D]
    v = vb.permute(0, 4, 1, 2, 3, 5)
    nf = k.shape[2]
    rep = q.unsqueeze(3).expand(-1, -1, -1, nf, -1, -1, -1)          # [B, H, a, f, k, j, D]: block row k of the queries
    inv_w = q.new_full((), 1.0 / (1.0 + 1e-6))
    for it in range(num_iters):
        z = torch.einsum("bhafkjd,bhfkld->bhafkjl", rep, k) * inv_w
        log_r = torch.log_softmax(z, -1)
        r = log_r.exp()
        kbar = torch.einsum("bhafkjl,bhfkld->bhafkjd", r, k)
        neg_h = (r * log_r).sum(-1)                                   # [B, H, a, f, k, j]
        s2 = torch.einsum("bhaijd,bhafkjd->bhaijfk", q, kbar) - neg_h.permute(0, 1, 2, 5, 3, 4).unsqueeze(3)
        left = torch.softmax(s2.flatten(5), -1).reshape(s2.shape)    # [B, H, a, i, j, f, k]
        if it + 1 < num_iters:
            rep = torch.einsum("bhaijfk,bhaijd->bhafkjd", left, q)
            inv_w = torch.clamp(1.0 / (left.sum(3).permute(0, 1, 2, 4, 5, 3) + 1e-6), max=1e4).unsqueeze(-1)
    y = torch.einsum("bhafkjl,bhfkld->bhafkjd", r, v)
    return torch.einsum("bhaijfk,bhafkjd->bhaijd", left, y).permute(0, 2, 3, 4, 1, 5)


def _refinement_grads(q, k, v, dout, tiling, sm_scale, num_iters, kv_block_order):
    """(dq, dk, dv) of the refinement for token-order q / dout and k, v in token order or (kv_block_order) block order;
    gradients come back in the same orders, float32."""
    f_tied, h_reduce, w_reduce, h, w = tiling
    b1, b2 = f_tied * (h // h_reduce), w // w_reduce
    with torch.enable_grad():
        q_, k_, v_ = (t.detach().float().requires_grad_(True) for t in (q, k, v))
        B, _, H, D = q.shape
        qb = _to_block_order(q_, *tiling).reshape(B, -1, b1, b2, H, D)
        kb = (k_ if kv_block_order else _to_block_order(k_, *tiling)).reshape(B, -1, b1, b2, H, D)
        vb = (v_ if kv_block_order else _to_block_order(v_, *tiling)).reshape(B, -1, b1, b2, H, D)
        ob = _refinement_torch(qb, kb, vb, sm_scale, num_iters)
        out = _from_block_order(ob.reshape(B, -1, H, D), *tiling)
        return torch.autograd.grad(out, (q_, k_, v_), dout.float())


class _MonarchIterFn(torch.autograd.Function):
    """monarch_attn with num_iters > 1 under autograd: HIP kernels forward, torch restatement for the gradients."""

    @staticmethod
    def forward(ctx, q, k, v, tiling, sm_scale, num_iters, heads_per_pass, kv_block_order):
        with torch.no_grad():
            out = monarch_attn(q, k, v, *tiling, sm_scale=sm_scale, num_iters=num_iters, heads_per_pass=heads_per_pass,
                               kv_block_order=kv_block_order)
        ctx.save_for_backward(q, k, v)
        ctx.cfg = (tiling, sm_scale, num_iters, kv_block_order)
        return out

    @staticmethod
    def backward(ctx, dout):
        q, k, v = ctx.saved_tensors
        tiling, sm_scale, num_iters, kv_block_order = ctx.cfg
        dq, dk, dv = _refinement_grads(q, k, v, dout, tiling, sm_scale, num_iters, kv_block_order)
        return dq.to(q.dtype), dk.to(k.dtype), dv.to(v.dtype), None, None, None, None, None


class _MonarchCacheIterFn(torch.autograd.Function):
    """monarch_attn_with_kv_cache with num_iters > 1 under autograd (cache written in place in the forward)."""

    @staticmethod
    def forward(ctx, q, k_cache, v_cache, new_k, new_v, start_idx, end_idx, tiling, sm_scale, num_iters, grad_only_new_kv,
                heads_per_pass):
        with torch.no_grad():
            out = monarch_attn_with_kv_cache(q, k_cache, v_cache, new_k, new_v, start_idx, end_idx, *tiling, sm_scale=sm_scale,
                                             num_iters=num_iters, heads_per_pass=heads_per_pass)
        ctx.save_for_backward(q, k_cache, v_cache)
        ctx.cfg = (start_idx, end_idx, tiling, sm_scale, num_iters, grad_only_new_kv)
        return out

    @staticmethod
    def backward(ctx, dout):
        q, k_cache, v_cache = ctx.saved_tensors
        start_idx, end_idx, tiling, sm_scale, num_iters, grad_only_new_kv = ctx.cfg
        dq, dkc, dvc = _refinement_grads(q, k_cache, v_cache, dout, tiling, sm_scale, num_iters, True)
        dk_new = _from_block_order(dkc[:, start_idx:end_idx], *tiling).to(k_cache.dtype)
        dv_new = _from_block_order(dvc[:, start_idx:end_idx], *tiling).to(v_cache.dtype)
        if grad_only_new_kv:
            dkc = dvc = None
        else:
            dkc, dvc = dkc.to(k_cache.dtype), dvc.to(v_cache.dtype)
        return dq.to(q.dtype), dkc, dvc, dk_new, dv_new, None, None, None, None, None, None, None


def _needs_grad(*ts):
    return torch.is_grad_enabled() and any(t.requires_grad for t in ts)


def monarch_attn_with_kv_cache(q, k_cache, v_cache, new_k, new_v, start_idx, end_idx, f_tied, h_reduce, w_reduce, h, w,
                               sm_scale=None, num_iters=1, grad_only_new_kv=False, heads_per_pass=0, one_kernel=False):
    """Writes new_k/new_v into k_cache/v_cache[:, start_idx:end_idx] (block order, in place) and
    returns one-iteration Monarch attention of q against the whole cache view.  `heads_per_pass` and `one_kernel`
    (no counterparts in the reference) bound the scratch and select the forward that keeps its intermediates in LDS.  Under
    autograd, `heads_per_pass` also keeps the forward from holding its intermediates, up to 2 GiB, for its backward."""
    if _needs_grad(q, k_cache, v_cache, new_k, new_v):
        if sm_scale is None:
            sm_scale = q.shape[-1] ** -0.5
        if num_iters != 1:
            return _MonarchCacheIterFn.apply(q, k_cache, v_cache, new_k, new_v, start_idx, end_idx,
                                             (f_tied, h_reduce, w_reduce, h, w), sm_scale, num_iters, grad_only_new_kv,
                                             heads_per_pass)
        return _MonarchCacheFn.apply(q, k_cache, v_cache, new_k, new_v, start_idx, end_idx,
                                     (f_tied, h_reduce, w_reduce, h, w), sm_scale, grad_only_new_kv, heads_per_pass)
    _check4("q", q)
    for name, t in (("k_cache", k_cache), ("v_cache", v_cache), ("new_k", new_k), ("new_v", new_v)):
        _check4(name, t, q.dtype, q.device)
    if k_cache.shape != v_cache.shape or new_k.shape != new_v.shape:
        raise ValueError("k/v shapes differ")
    if new_k.stride() != new_v.stride():
        new_v = new_v.contiguous()
        new_k = new_k.contiguous()
    n, size = new_k.shape, q.shape           # once: the smallest calls are host work
    if n[1] != end_idx - start_idx:
        raise ValueError(f"new_k holds {n[1]} tokens but end_idx - start_idx = {end_idx - start_idx}")
    if sm_scale is None:
        sm_scale = size[3] ** -0.5
    if n[0] != size[0] or n[2] != size[2] or n[3] != size[3]:      # not _like_q
        kv_cache_write(new_k, new_v, k_cache, v_cache, start_idx, end_idx, f_tied, h_reduce, w_reduce, h, w)
        return monarch_attn(q, k_cache, v_cache, f_tied, h_reduce, w_reduce, h, w, sm_scale=sm_scale, num_iters=num_iters,
                            heads_per_pass=heads_per_pass, kv_block_order=True, one_kernel=one_kernel)
    out = torch.empty(size, dtype=q.dtype, device=q.device)
    d = _desc(q, k_cache, v_cache, out, f_tied, h_reduce, w_reduce, h, w, sm_scale, 1, 0, num_iters, one_kernel)
    nbytes = monarch_workspace_bytes(d, heads_per_pass)
    ws = scratch(nbytes, q.device)
    if _KEPT:
        _drop_kept(q.device.index)
    with _on_device(q.device):
        _l.check(_l.load().sfm_monarch_attn_with_kv_cache(
            C.byref(d), q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), new_k.data_ptr(), new_v.data_ptr(),
            _l.strides3(new_k), start_idx, end_idx, out.data_ptr(), ws.data_ptr(), nbytes, _stream(q)))
    return out


def monarch_attn_with_kv_cache_static(q, k_cache, v_cache, new_k, new_v, start_idx, end_idx, f_tied, h_reduce, w_reduce, h, w,
                                      sm_scale=None, num_iters=1, out=None):
    """monarch_attn_with_kv_cache for callers that cannot allocate (HIP graph capture, serving loops): the scratch
    is the library's own per-GPU array (lib.STATIC_SCRATCH_BYTES) instead of a fresh tensor, and with `out` given
    nothing is allocated at all.  No autograd.  Calls on one GPU share the scratch and must not overlap."""
    _check4("q", q)
    for name, t in (("k_cache", k_cache), ("v_cache", v_cache), ("new_k", new_k), ("new_v", new_v)):
        _check4(name, t, q.dtype, q.device)
    if k_cache.shape != v_cache.shape or new_k.shape != new_v.shape or new_k.stride() != new_v.stride():
        raise ValueError("k/v shapes or strides differ")
    if not _like_q(q, new_k):
        raise ValueError(f"new_k {tuple(new_k.shape)} must have q's batches, heads and head_dim {tuple(q.shape)}")
    if new_k.shape[1] != end_idx - start_idx:
        raise ValueError(f"new_k holds {new_k.shape[1]} tokens but end_idx - start_idx = {end_idx - start_idx}")
    if sm_scale is None:
        sm_scale = q.shape[-1] ** -0.5
    if out is None:
        out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
    else:
        _check4("out", out, q.dtype, q.device)
        if out.shape != q.shape:
            raise ValueError("out must have q's shape")
    d = _desc(q, k_cache, v_cache, out, f_tied, h_reduce, w_reduce, h, w, sm_scale, 1, 0, num_iters)
    if _KEPT:
        _drop_kept(q.device.index)
    with _on_device(q.device):
        _l.check(_l.load().sfm_monarch_attn_with_kv_cache_static(
            C.byref(d), q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), new_k.data_ptr(), new_v.data_ptr(),
            _l.strides3(new_k), start_idx, end_idx, out.data_ptr(), _stream(q)))
    return out


def monarch_attn(q, k, v, f_tied, h_reduce, w_reduce, h, w, sm_scale=None, block_causal_size=None, num_iters=1,
                 heads_per_pass=0, kv_block_order=False, one_kernel=False):
    """One-iteration Monarch attention without a cache write; `block_causal_size` (tokens) masks
    block-frames of later causal blocks.  `kv_block_order=True` (no counterpart in the reference) says
    that k, v are a KV-cache view whose rows are already in Monarch block order, e.g. after
    prologue.qk_prologue wrote them.  `heads_per_pass` and `one_kernel` as in monarch_attn_with_kv_cache."""
    if _needs_grad(q, k, v):
        if sm_scale is None:
            sm_scale = q.shape[-1] ** -0.5
        if num_iters != 1:
            if block_causal_size is not None:
                raise ValueError("causal currently only supported for num_iters=1")
            return _MonarchIterFn.apply(q, k, v, (f_tied, h_reduce, w_reduce, h, w), sm_scale, num_iters, heads_per_pass,
                                        kv_block_order)
        return _MonarchFn.apply(q, k, v, (f_tied, h_reduce, w_reduce, h, w), sm_scale, block_causal_size,
                                heads_per_pass, kv_block_order)
    _check4("q", q)
    _check4("k", k, q.dtype, q.device)
    _check4("v", v, q.dtype, q.device)
    if k.stride() != v.stride():
        k, v = k.contiguous(), v.contiguous()
    if sm_scale is None:
        sm_scale = q.shape[-1] ** -0.5
    cbf = _causal_block_frames(q, k, (f_tied, h_reduce, w_reduce, h, w), block_causal_size, num_iters)
    out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
    d = _desc(q, k, v, out, f_tied, h_reduce, w_reduce, h, w, sm_scale, 1 if kv_block_order else 0, cbf, num_iters, one_kernel)
    nbytes = monarch_workspace_bytes(d, heads_per_pass)
    ws = scratch(nbytes, q.device)
    with _on_device(q.device):
        _l.check(_l.load().sfm_monarch_fwd(C.byref(d), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                                           ws.data_ptr(), nbytes, _stream(q)))
    return out
