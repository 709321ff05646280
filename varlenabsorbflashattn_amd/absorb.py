"""Ragged absorbed target attention -- drop-in for
``triton_target_attn_absorb`` (ta/interface.py:125-454).

``packed_target_attn`` keeps the reference signature.  For 16-bit inputs on
the matrix-core shapes it forms ``q_proj = q_raw W_Q`` and runs the attention
with ``u = q_proj W_K^T`` formed inside the attention kernel (u never reaches
memory in the forward); otherwise it projects ``u`` per head (this library's
projection kernels, or torch GEMMs for odd 16-bit widths, as in
ta/interface.py:429-435) and calls ``target_attn_inner``, whose forward and
backward run in ``libvafa.so``:
scores are taken directly against the raw ``X`` rows, ``aX = softmax(u X^T) X``
is accumulated on the fly and projected by ``W_V`` at the end.  The backward
is deterministic (dW_V and dX are reduced in a fixed order).
"""
from __future__ import annotations

import functools
import math
import os
import weakref
from typing import Optional

import numpy as np
import torch

from . import _lib

# Reference block sizes, kept for the (seg, block) tables that
# prepare_target_attn_indices returns (ta/interface.py:59-63).
_BT_Q_FWD = 16
_BT_K_BWD = 64

# prepare_target_attn_indices() remembers the host cu_seqlens behind the
# tables it returns, so a later validate=False call on the SAME, unmodified
# cu_seqlens tensors needs no device->host copy.  Keyed by id() of the query
# table with a weak reference to it; the cu_seqlens tensors are held by weak
# reference together with their version counters and data pointers, so any
# other pair of tensors (or an in-place change of these) takes the copy again.
_HOST_CU: dict = {}


def _cu_stamp(t):
    if not isinstance(t, torch.Tensor):
        return None
    return (weakref.ref(t), t._version, t.data_ptr())


def _stamp_matches(stamp, t) -> bool:
    if stamp is None or not isinstance(t, torch.Tensor):
        return False
    ref, version, data_ptr = stamp
    return ref() is t and t._version == version and t.data_ptr() == data_ptr


def _remember_host_cu(table: torch.Tensor, cu_q, cu_k, cu_q_h: np.ndarray,
                      cu_k_h: np.ndarray) -> None:
    key = id(table)
    _HOST_CU[key] = (weakref.ref(table, lambda _r, k=key: _HOST_CU.pop(k, None)),
                     _cu_stamp(cu_q), _cu_stamp(cu_k), cu_q_h, cu_k_h)


def _recall_host_cu(table: Optional[torch.Tensor], cu_q, cu_k):
    """Host copies taken when ``table`` was prepared, if ``cu_q`` / ``cu_k`` are
    the very tensors it was prepared from, unmodified since; else None."""
    if table is None:
        return None
    hit = _HOST_CU.get(id(table))
    if hit is None or hit[0]() is not table:
        return None
    if not (_stamp_matches(hit[1], cu_q) and _stamp_matches(hit[2], cu_k)):
        return None
    return hit[3], hit[4]


def _select_fwd_mode() -> str:
    """TRITON_TARGET_ATTN_FWD_MODE as in ta/interface.py:66-70.

    Both accepted modes run the same fused kernel here; the variable keeps
    its validation so existing configurations behave the same.
    """
    mode = os.environ.get("TRITON_TARGET_ATTN_FWD_MODE", "alpha").lower()
    if mode in ("direct", "alpha"):
        return mode
    raise ValueError("TRITON_TARGET_ATTN_FWD_MODE must be one of: direct, alpha")


def _select_dx_mode(n_k_chunks: int) -> str:
    """TRITON_TARGET_ATTN_DX_MODE as in ta/interface.py:73-85 (validation only:
    every mode maps to the deterministic dX kernel)."""
    mode = os.environ.get("TRITON_TARGET_ATTN_DX_MODE", "auto").lower()
    if mode in ("partial", "fused", "atomic"):
        return mode
    if mode != "auto":
        raise ValueError(
            "TRITON_TARGET_ATTN_DX_MODE must be one of: auto, partial, fused, atomic")
    return "fused" if n_k_chunks >= 1024 else "partial"


def _validate_cu_seqlens(cu_host: np.ndarray, shape, T: int, name: str) -> None:
    """ta/interface.py:92-106."""
    if len(shape) != 1 or cu_host.size < 2:
        raise ValueError(f"{name}: must be 1-D with len>=2, got {tuple(shape)}")
    _lib.validate_cu_absorb(cu_host, T, name)


def _next_power_of_2(x: int) -> int:
    if x < 1:
        raise ValueError(f"expected positive dimension, got {x}")
    return 1 << (x - 1).bit_length()


def prepare_target_attn_indices(cu_seqlens_q: torch.Tensor, cu_seqlens_k: torch.Tensor):
    """Chunk tables ``(q_idx [NT_q,2], k_idx [NT_k,2])`` (ta/interface.py:125-138).

    Same content as the reference (BT_Q=16, BT_K=64 rows ``(seg, block)``).
    Passing them back with ``validate=False`` together with the same
    cu_seqlens tensors skips every host round trip: the host cu_seqlens
    captured here are reused to look up the cached plan.  With other (or
    modified) cu_seqlens tensors the call copies them to the host again, so
    the plan always follows the cu_seqlens of the call, as the reference's
    kernels do (they read cu_seqlens on every call).
    """
    cu_q_h, cu_k_h = _lib.as_host_i64_pair(cu_seqlens_q, cu_seqlens_k)
    q_idx = torch.from_numpy(_lib.chunk_indices(cu_q_h, _BT_Q_FWD)).to(cu_seqlens_q.device)
    k_idx = torch.from_numpy(_lib.chunk_indices(cu_k_h, _BT_K_BWD)).to(cu_seqlens_k.device)
    _remember_host_cu(q_idx, cu_seqlens_q, cu_seqlens_k, cu_q_h, cu_k_h)
    return q_idx, k_idx


def _aligned(x: torch.Tensor) -> torch.Tensor:
    return x.clone() if x.data_ptr() % 16 != 0 else x


def _absorb_plan(T_q, T_k, H, D_KV, D_H, device, cu_seqlens_q, cu_seqlens_k,
                 q_chunk_indices, validate):
    """Validation (ta/interface.py:92-122, 176-201) and the cached device plan
    of one absorb call; host cu_seqlens come from the prepared index tables
    when they belong to these very tensors and validation is off."""
    known = _recall_host_cu(q_chunk_indices, cu_seqlens_q, cu_seqlens_k)
    if known is not None and not validate:
        cu_q, cu_k = known
    else:
        cu_q, cu_k = _lib.host_cu_pair(cu_seqlens_q, cu_seqlens_k)
    # the checks depend on the content and the token counts alone: a cached
    # plan of the same content that covers exactly these tokens passed them
    # (keys_ok: including the last one)
    key = _lib.plan_key("absorb", cu_q, cu_k, (H, D_KV, D_H), device)
    plan = _lib.cached_plan(key) if cu_q.ndim == 1 and cu_k.ndim == 1 else None
    known_ok = (plan is not None and plan.T_q == T_q and plan.T_k == T_k
                and (plan.keys_ok or not validate))
    if not known_ok:
        cu_q_h, cu_k_h = _lib.as_host_i64(cu_q), _lib.as_host_i64(cu_k)
        if validate:
            n_seg = cu_seqlens_q.numel() - 1
            assert cu_seqlens_k.numel() - 1 == n_seg, "segment count mismatch q vs k"
            _validate_cu_seqlens(cu_q_h, cu_seqlens_q.shape, T_q, "cu_seqlens_q")
            _validate_cu_seqlens(cu_k_h, cu_seqlens_k.shape, T_k, "cu_seqlens_k")
            _lib.check_active_have_keys(cu_q_h, cu_k_h)
        B_DKV = _next_power_of_2(D_KV)
        assert B_DKV <= 512, f"D_KV={D_KV} pads to {B_DKV}, which is too large for v1 tiles"
        if plan is None:
            plan = _lib.new_plan(key, cu_q_h, cu_k_h)
        plan.keys_ok = plan.keys_ok or bool(validate)
    if plan.T_q > T_q or plan.T_k > T_k:
        raise ValueError(
            f"cu_seqlens address {plan.info.T_q} query / {plan.info.T_k} key tokens but "
            f"the inputs hold {T_q} / {T_k}")
    if plan.info.n_fwd > 0:
        _select_fwd_mode()
    return plan.use()


class _TargetAttnFunction(torch.autograd.Function):
    """Inner op on projected u (ta/interface.py:141-321)."""

    @staticmethod
    def forward(ctx, u, X, W_V, cu_seqlens_q, cu_seqlens_k, scale, q_chunk_indices,
                k_chunk_indices, validate):
        T_q, H, D_KV = u.shape
        T_k, D_KV_x = X.shape
        D_KV_wv, H_wv, D_H = W_V.shape
        assert D_KV == D_KV_x == D_KV_wv, \
            f"D_KV mismatch: u={D_KV}, X={D_KV_x}, W_V={D_KV_wv}"
        assert H == H_wv, f"H mismatch: u={H}, W_V={H_wv}"
        assert u.dtype == X.dtype == W_V.dtype, \
            f"u/X/W_V must share dtype, got {u.dtype}/{X.dtype}/{W_V.dtype}"
        assert u.is_cuda and X.is_cuda and W_V.is_cuda, "all inputs must be CUDA"
        assert u.device == X.device == W_V.device, "u/X/W_V must be on same device"
        assert D_H in (16, 32, 64, 128, 256), f"D_H {D_H} not supported"
        _lib.dtype_code(u.dtype)
        u, X, W_V = (_aligned(t.contiguous()) for t in (u, X, W_V))
        plan = _absorb_plan(T_q, T_k, H, D_KV, D_H, u.device, cu_seqlens_q, cu_seqlens_k,
                            q_chunk_indices, validate)
        O, LSE = _lib.ops().absorb_fwd(u, X, W_V, plan.native, scale)
        ctx.save_for_backward(u, X, W_V, O, LSE)
        ctx.plan = plan
        ctx.scale = scale
        return O

    @staticmethod
    def backward(ctx, dO):
        u, X, W_V, O, LSE = ctx.saved_tensors
        if ctx.plan.info.n_kv > 0:
            _select_dx_mode(int(ctx.plan.info.n_kv))
        return *_lib.ops().absorb_bwd(u, X, W_V, O, LSE, dO, ctx.plan.native, ctx.scale), \
            None, None, None, None, None, None


def target_attn_inner(
    u: torch.Tensor,
    X: torch.Tensor,
    W_V: torch.Tensor,
    cu_seqlens_q: torch.Tensor,
    cu_seqlens_k: torch.Tensor,
    scale: Optional[float] = None,
    q_chunk_indices: Optional[torch.Tensor] = None,
    k_chunk_indices: Optional[torch.Tensor] = None,
    validate: bool = True,
) -> torch.Tensor:
    """Inner entry on projected ``u [T_q,H,D_KV]`` (ta/interface.py:324-354)."""
    if scale is None:
        scale = 1.0 / math.sqrt(W_V.shape[2])
    return _TargetAttnFunction.apply(
        u, X, W_V, cu_seqlens_q, cu_seqlens_k, float(scale),
        q_chunk_indices, k_chunk_indices, validate)


def _project_native(q_raw: torch.Tensor, W_Q: torch.Tensor, W_K: torch.Tensor) -> bool:
    """Whether this library's projection kernels take these operands: CUDA,
    one dtype, D_H a multiple of 8 and, in 16 bits, D_Q and D_KV too."""
    d_q = q_raw.shape[1]
    d_kv, _, D_H = W_K.shape
    if not (q_raw.is_cuda and W_Q.device == W_K.device == q_raw.device
            and W_Q.dtype == W_K.dtype == q_raw.dtype and D_H % 8 == 0):
        return False
    if q_raw.dtype == torch.float32:
        # (autocast applies to the torch formulation only)
        H = W_Q.shape[1]
        return (0 < d_q <= 65536 and 0 < d_kv <= 65536 and H * D_H <= 65536
                and H <= 1024 and not torch.is_autocast_enabled()
                and _project_f32_pays(q_raw.shape[0], H, d_q, d_kv, D_H,
                                      torch.is_grad_enabled() and
                                      any(t.requires_grad for t in (q_raw, W_Q, W_K))))
    return (q_raw.dtype in (torch.bfloat16, torch.float16)
            and d_q % 8 == 0 and d_kv % 8 == 0)


def _project_f32_pays(T_q: int, H: int, d_q: int, d_kv: int, D_H: int, grad: bool) -> bool:
    """Whether the fp32 projections run on this library's kernels rather than on
    torch's GEMMs: what either takes on large launches, from the rates measured
    there, and what torch's calls cost at least.

    The row GEMM streams its operands from L2 at 47 TFLOP/s over D_Q and 50 over
    D_KV; 25 where u's sums are shorter than 64 (D_H = 32), about half over widths
    that are not whole 16-byte chunks and where H D_H leaves half of its 64 columns
    empty.  Its backward runs at 44 (28 over such a D_KV).  Torch's reach 110, and 95
    backward, but multiply H blocks per D_KV, of which one is not zero, and take
    25 us, with a backward 100, longer to call.  us, torch / own, forward and forward
    + backward, H x D_H, D_Q, D_KV, tokens: 8 x 32, 256, 256, 2400 101 / 35 and 415 /
    101, 200k 1941 / 1658 and 6466 / 4210; 8 x 32, 968, 216, 10k 190 / 147, 20k 274 /
    280, 50k 2361 / 2086, 200k 7586 / 8303; 1 x 256, 256, 256, 5k 52 / 40, 10k 52 / 56 and
    208 / 184, 20k 307 / 367, 200k 552 / 996 and 2199 / 3299."""
    x = 2e-6 * T_q * H * D_H  # us x TFLOP/s per feature
    aligned = d_kv % 4 == 0
    own = d_q / (47 if d_q % 4 == 0 and H * D_H >= 64 else 23) + \
        d_kv / ((50 if D_H >= 64 else 25) * (1 if aligned else 0.63))
    blocks = d_q + H * d_kv
    if not grad:
        return x * (own - blocks / 110) < 25
    own += 2 * d_q / 44 + 2 * d_kv / (44 if aligned else 28)
    return x * (own - blocks * (1 / 110 + 2 / 95)) < 100


class _Project(torch.autograd.Function):
    """q_proj = q_raw W_Q, u[t,h,:] = q_proj[t,h,:] W_K[:,h,:]^T
    (ta/interface.py:434-435), forward and backward on the row-GEMM and
    weight-gradient kernels of ``vafa_absorb_project_fwd`` / ``_bwd`` (16-bit)
    and ``vafa_absorb_project_f32_fwd`` / ``_bwd``.  Each product is rounded
    once to the input dtype, as the reference's GEMMs and their autograd backward
    (dq_proj = du W_K per head, dq_raw = dq_proj W_Q^T, dW_Q = q_raw^T dq_proj,
    dW_K = du^T q_proj per head); the weight gradients are summed over fixed
    token chunks in order (deterministic)."""

    @staticmethod
    def forward(ctx, q_raw: torch.Tensor, W_Q: torch.Tensor, W_K: torch.Tensor) -> torch.Tensor:
        q_raw, W_Q, W_K = (_aligned(t.contiguous()) for t in (q_raw, W_Q, W_K))
        q_proj, u = _lib.ops().project_fwd(q_raw, W_Q, W_K)
        ctx.save_for_backward(q_raw, W_Q, W_K, q_proj)
        return u

    @staticmethod
    def backward(ctx, du: torch.Tensor):
        return _lib.ops().project_bwd(*ctx.saved_tensors, du, *ctx.needs_input_grad[:3])


@functools.lru_cache(maxsize=256)
def _fold_shape(H: int, d_kv: int, D_H: int, dtype: torch.dtype) -> bool:
    return bool(_lib.lib().vafa_absorb_fold_supported(H, d_kv, D_H, _lib.dtype_code(dtype)))


def _fold_native(q_raw, X, W_Q, W_K, W_V) -> bool:
    """Whether packed_target_attn can run with u folded into the attention
    kernel (vafa_absorb_fwd_full): the native projection's operands, X and
    W_V of the same dtype on the same device, and a shape of the folded
    matrix-core kernel."""
    if q_raw.dtype == torch.float32 or not _project_native(q_raw, W_Q, W_K):
        return False
    if X.dtype != q_raw.dtype or W_V.dtype != q_raw.dtype or not (X.is_cuda and W_V.is_cuda):
        return False
    if not (q_raw.device == X.device == W_Q.device == W_K.device == W_V.device):
        return False
    d_kv, H, D_H = W_K.shape
    return _fold_shape(H, d_kv, D_H, q_raw.dtype)


class _FoldedTargetAttn(torch.autograd.Function):
    """packed_target_attn with the u projection folded into the attention
    forward (ta/interface.py:429-435 followed by ta/interface.py:141-321).

    Forward (vafa_absorb_fwd_full): q_proj = q_raw W_Q (row-GEMM kernel,
    rounded to the input dtype), then the attention, whose workgroups form
    u = q_proj_h W_K,h^T for their own rows on the matrix cores -- u is never
    written to memory.
    Backward (vafa_absorb_bwd_full): u is formed once from the saved q_proj,
    in one launch with dAX and delta, then the inner backward gives du / dX /
    dW_V and the projection backward dq_raw / dW_Q / dW_K, as the unfused path."""

    @staticmethod
    def forward(ctx, q_raw, X, W_Q, W_K, W_V, cu_seqlens_q, cu_seqlens_k, scale,
                q_chunk_indices, k_chunk_indices, validate):
        T_k, d_kv = X.shape
        _, H, D_H = W_Q.shape
        q_raw, X, W_Q, W_K, W_V = (_aligned(t.contiguous()) for t in (q_raw, X, W_Q, W_K, W_V))
        plan = _absorb_plan(q_raw.shape[0], T_k, H, d_kv, D_H, X.device, cu_seqlens_q,
                            cu_seqlens_k, q_chunk_indices, validate)
        q_proj, O, LSE = _lib.ops().absorb_full_fwd(q_raw, X, W_Q, W_K, W_V, plan.native, scale)
        ctx.save_for_backward(q_raw, W_Q, W_K, q_proj, X, W_V, O, LSE)
        ctx.plan = plan
        ctx.scale = scale
        return O

    @staticmethod
    def backward(ctx, dO):
        if ctx.plan.info.n_kv > 0:
            _select_dx_mode(int(ctx.plan.info.n_kv))
        need_q, _, need_wq, need_wk = ctx.needs_input_grad[:4]
        return *_lib.ops().absorb_full_bwd(*ctx.saved_tensors, dO, ctx.plan.native, ctx.scale,
                                           need_q, need_wq, need_wk), \
            None, None, None, None, None, None


def _project_u(q_raw: torch.Tensor, W_Q: torch.Tensor, W_K: torch.Tensor) -> torch.Tensor:
    """u[t,h,:] = (q_raw[t] W_Q[:,h,:]) W_K[:,h,:]^T (ta/interface.py:434-435),
    contiguous ``[T_q, H, d_kv]``.

    CUDA operands run on ``_Project`` (both directions in this library's
    kernels) in fp32 up to the token counts of ``_project_f32_pays`` and, with
    D_Q, D_KV, D_H multiples of 8, in 16 bits.
    Other operands (odd 16-bit widths, the CPU) take the reference's own
    formulation on torch's GEMMs: q_proj =
    q_raw @ W_Q, then u = q_proj @ blockdiag(W_K[:,h,:]^T), ONE GEMM that
    writes u token-major (for finite q_proj the zero blocks add exact zeros
    to each fp32 sum, so every u element is the same sum of products as per
    head).
    """
    if _project_native(q_raw, W_Q, W_K):
        return _Project.apply(q_raw, W_Q, W_K)
    T_q, d_q = q_raw.shape
    _, H, D_H = W_Q.shape
    q_proj = q_raw @ W_Q.reshape(d_q, H * D_H)
    blocks = torch.block_diag(*[W_K[:, h, :].t() for h in range(H)])
    return (q_proj @ blocks).view(T_q, H, W_K.shape[0])


def packed_target_attn(
    q_raw: torch.Tensor,
    X: torch.Tensor,
    W_Q: torch.Tensor,
    W_K: torch.Tensor,
    W_V: torch.Tensor,
    *,
    cu_seqlens_q: Optional[torch.Tensor] = None,
    cu_seqlens_k: Optional[torch.Tensor] = None,
    q_seqinfo: Optional[torch.Tensor] = None,
    k_seqinfo: Optional[torch.Tensor] = None,
    q_chunk_indices: Optional[torch.Tensor] = None,
    k_chunk_indices: Optional[torch.Tensor] = None,
    scale: Optional[float] = None,
    bf16: bool = False,
    validate: bool = True,
) -> torch.Tensor:
    """Full ragged target attention with matrix absorption (ta/interface.py:357-445).

    q_raw ``[T_q,d_q]`` or ``[1,T_q,d_q]``; X ``[T_k,d_kv]`` or ``[1,T_k,d_kv]``;
    W_Q ``[d_q,H,D_H]``, W_K/W_V ``[d_kv,H,D_H]``.  Returns O ``[T_q,H,D_H]``
    in the compute dtype (bf16 when ``bf16=True``, else the input dtype).
    """
    if q_raw.dim() == 3:
        assert q_raw.shape[0] == 1, "batch must be 1 for packed varlen"
        q_raw = q_raw.squeeze(0)
    if X.dim() == 3:
        assert X.shape[0] == 1
        X = X.squeeze(0)

    T_q, d_q = q_raw.shape
    T_k, d_kv = X.shape
    d_q_wq, H, D_H = W_Q.shape
    d_kv_wk, H_wk, D_H_wk = W_K.shape
    d_kv_wv, H_wv, D_H_wv = W_V.shape
    assert d_q_wq == d_q, f"W_Q[0]={d_q_wq} != d_q={d_q}"
    assert d_kv_wk == d_kv and d_kv_wv == d_kv, "W_K/W_V d_kv mismatch"
    assert H == H_wk == H_wv, "H mismatch across W_Q/W_K/W_V"
    assert D_H == D_H_wk == D_H_wv, "D_H mismatch across W_Q/W_K/W_V"

    if cu_seqlens_q is None:
        assert q_seqinfo is not None
        cu_seqlens_q = _seqinfo_to_cu(q_seqinfo)
    if cu_seqlens_k is None:
        assert k_seqinfo is not None
        cu_seqlens_k = _seqinfo_to_cu(k_seqinfo)

    if bf16:
        q_raw, X, W_Q, W_K, W_V = (t if t.dtype == torch.bfloat16 else t.to(torch.bfloat16)
                                   for t in (q_raw, X, W_Q, W_K, W_V))

    if scale is None:
        scale = 1.0 / math.sqrt(D_H)
    if _fold_native(q_raw, X, W_Q, W_K, W_V):
        return _FoldedTargetAttn.apply(
            q_raw, X, W_Q, W_K, W_V, cu_seqlens_q, cu_seqlens_k, float(scale),
            q_chunk_indices, k_chunk_indices, validate)
    u = _project_u(q_raw, W_Q, W_K)
    return target_attn_inner(
        u, X, W_V, cu_seqlens_q, cu_seqlens_k, scale,
        q_chunk_indices=q_chunk_indices, k_chunk_indices=k_chunk_indices, validate=validate)


def _seqinfo_to_cu(seqinfo: torch.Tensor) -> torch.Tensor:
    """[n_seg] lengths -> [n_seg+1] int32 (ta/interface.py:448-454: asserts only)."""
    assert seqinfo.dim() == 1 and seqinfo.numel() >= 1
    s = _lib.as_host_i64(seqinfo)
    cu = np.zeros(s.size + 1, dtype=np.int64)
    cu[1:] = np.cumsum(s)
    return torch.from_numpy(cu.astype(np.int32)).to(seqinfo.device)
