"""Fused causal RACE attention layer: q, k, v in; out (and dq, dk, dv) out.

One autograd Function over the bf16 fused kernels (race_qkv_fwd / race_qkv_bwd):
the soft-hash of scaling/race_common.py:36-73 and the causal scan of
race_causal_cuda.py:47-69 run inside the same HIP kernels, so the [N,T,S] bucket
probabilities are never written to HBM. The forward saves only q, k, v and the
per-block bucket states; the backward recomputes the probabilities.

Grouped-query attention: q [B,Hq,T,D] with k, v [B,Hkv,T,D]; query head h reads
the bucket state of kv head h // (Hq // Hkv). With Hq == Hkv this is the
reference's multi-head layer.
"""
import math

import torch
from torch.autograd import Function

from . import _lib


def fused_supported(q, k, v, Kbits):
    """True when the bf16 fused kernels cover these inputs."""
    return (q.dtype == torch.bfloat16 and k.dtype == torch.bfloat16 and v.dtype == torch.bfloat16
            and q.dim() == 4 and q.shape[-1] in (64, 128) and 1 <= Kbits <= 4
            and q.device.type == "cuda")


def _bf16_rows(t):
    """A [B,H,T,D] bf16 view whose rows the kernels can read as 16-byte vectors."""
    sb, sh, st, sd = t.stride()
    if sd != 1 or t.data_ptr() % 16 or (sb | sh | st) % 8:
        t = t.clone(memory_format=torch.contiguous_format)  # (contiguous() keeps an odd address)
    return t


def _out_rows(B, H, T, D, dtype, device, bthd):
    """A new [B,H,T,D] tensor, contiguous or (bthd) in the memory order of [B,T,H,D]. No view: autograd
    refuses in-place changes to a view that a Function returns."""
    if bthd:
        return torch.empty_strided((B, H, T, D), (T * H * D, D, H * D, 1), dtype=dtype, device=device)
    return torch.empty(B, H, T, D, dtype=dtype, device=device)


def qkv_shape(q, k, L, Kbits, scale, eps, block=0):
    B, Hq, T, D = q.shape
    return _lib.qkv_shape(B, Hq, k.shape[1], T, D, L, Kbits, float(scale), float(eps), int(block))


class RaceAttentionFn(Function):
    """out = causal RACE(q, k, v); q [B,Hq,T,D], k/v [B,Hkv,T,D] bf16, planes_T [D, L*K].

    The gradients take the memory order of q, k and v, so that autograd hands them on without a
    layout copy; the output is contiguous, or with `bthd` in the memory order of [B,T,Hq,D]."""

    @staticmethod
    def forward(ctx, q, k, v, planes_T, L, Kbits, scale, eps, out_dtype, block, bthd=False):
        _lib.require_device(q, k, v, planes_T)
        if not fused_supported(q, k, v, Kbits):
            raise _lib.RaceError("fused RACE needs bf16 q/k/v with head dim 64 or 128 and K <= 4")
        B, Hq, T, D = q.shape
        if k.shape != (B, k.shape[1], T, D) or v.shape != k.shape or Hq % k.shape[1]:
            raise ValueError(f"q {tuple(q.shape)} / k {tuple(k.shape)} / v {tuple(v.shape)} mismatch")
        q, k, v = _bf16_rows(q), _bf16_rows(k), _bf16_rows(v)
        planes = _lib.f32_planes(planes_T)
        if planes.shape != (D, L * Kbits):
            raise ValueError(f"planes_T must be [{D}, {L * Kbits}], got {tuple(planes.shape)}")
        out_dtype = out_dtype or q.dtype
        sh = qkv_shape(q, k, L, Kbits, scale, eps, block)
        lib = _lib.lib()
        state = _lib.workspace(lib.race_qkv_state_bytes(sh), q.device)
        scratch = _lib.workspace(lib.race_qkv_scratch_bytes(sh, 0), q.device)
        out = _out_rows(B, Hq, T, D, out_dtype, q.device, bthd)
        qv, _ = _lib.view4(q)
        kv_, _ = _lib.view4(k)
        vv, _ = _lib.view4(v)
        ov = _lib.out_view4(out)
        _lib.check(lib.race_qkv_fwd(sh, qv, kv_, vv, _lib.ptr(planes), ov, _lib.dtype_code(out_dtype),
                                    _lib.ptr(state), state.numel(), _lib.ptr(scratch), scratch.numel(),
                                    _lib.stream_of(q)), "race_qkv_fwd")
        ctx.save_for_backward(q, k, v, planes, state)
        ctx.cfg = (L, Kbits, float(scale), float(eps), int(block))
        return out

    @staticmethod
    def backward(ctx, grad_out):
        q, k, v, planes, state = ctx.saved_tensors
        L, Kbits, scale, eps, block = ctx.cfg
        go = _bf16_rows(grad_out.to(torch.bfloat16))
        sh = qkv_shape(q, k, L, Kbits, scale, eps, block)
        lib = _lib.lib()
        scratch = _lib.workspace(lib.race_qkv_scratch_bytes(sh, 1), q.device)
        dq, dk, dv = (_lib.rows_like(t) for t in (q, k, v))
        views = [_lib.view4(t)[0] for t in (q, k, v, go)] + [_lib.out_view4(t) for t in (dq, dk, dv)]
        _lib.check(lib.race_qkv_bwd(sh, views[0], views[1], views[2], views[3], _lib.ptr(planes),
                                    _lib.ptr(state), state.numel(), views[4], views[5], views[6],
                                    _lib.ptr(scratch), scratch.numel(), _lib.stream_of(q)), "race_qkv_bwd")
        return dq, dk, dv, None, None, None, None, None, None, None, None


def race_causal_attention(q, k, v, planes_T, L, Kbits, scale=None, eps=1e-6, out_dtype=None, block=0):
    """Causal RACE attention of bf16 q [B,Hq,T,D], k/v [B,Hkv,T,D] -> [B,Hq,T,D].

    `scale` divides tanh(x . plane) (default sqrt(D) as scaling/race_common.py:46);
    `out_dtype` defaults to q's dtype; `block` sets tokens per workgroup (0: auto).
    """
    if scale is None:
        scale = math.sqrt(q.shape[-1])
    return RaceAttentionFn.apply(q, k, v, planes_T, L, Kbits, scale, eps, out_dtype, block)


def race_causal_attention_with_state(q, k, v, planes_T, L, Kbits, scale=None, eps=1e-6, out_dtype=None,
                                     state_out=None, bthd=False):
    """Forward only (no autograd): (out, A [B*Hkv,S], Bs [B*Hkv,S,D]) -- the output and
    the final bucket state (race_prefix_ref's A_final / B_final, race_common.py:88-90),
    which seeds race_attention_amd.decode.RaceDecodeState. `state_out` gives the (A, Bs)
    to write (contiguous fp32); new tensors otherwise. `bthd`: out is in the memory order of [B,T,Hq,D]."""
    _lib.require_device(q, k, v, planes_T)
    if scale is None:
        scale = math.sqrt(q.shape[-1])
    if not fused_supported(q, k, v, Kbits):
        raise _lib.RaceError("fused RACE needs bf16 q/k/v with head dim 64 or 128 and K <= 4")
    q, k, v = _bf16_rows(q), _bf16_rows(k), _bf16_rows(v)
    B, Hq, T, D = q.shape
    Hkv, S = k.shape[1], L << Kbits
    # (k and v may be larger than q's batch, tokens and head dim, v than k's heads: the rest is not read)
    if any(x.shape[0] < B or x.shape[1] < Hkv or x.shape[2] < T or x.shape[3] < D for x in (k, v)):
        raise ValueError(f"q {tuple(q.shape)} / k {tuple(k.shape)} / v {tuple(v.shape)} mismatch")
    planes = _lib.f32_planes(planes_T)
    out_dtype = out_dtype or q.dtype
    sh = qkv_shape(q, k, L, Kbits, scale, eps, 0)
    lib = _lib.lib()
    work = _lib.workspace(lib.race_qkv_state_bytes(sh), q.device)
    scratch = _lib.workspace(lib.race_qkv_scratch_bytes(sh, 0), q.device)
    out = _out_rows(B, Hq, T, D, out_dtype, q.device, bthd)
    if state_out is None:
        A = torch.empty(B * Hkv, S, dtype=torch.float32, device=q.device)
        Bs = torch.empty(B * Hkv, S, D, dtype=torch.float32, device=q.device)
    else:
        A, Bs = state_out
        if (A.shape != (B * Hkv, S) or Bs.shape != (B * Hkv, S, D) or not (A.is_contiguous() and Bs.is_contiguous())
                or A.dtype != torch.float32 or Bs.dtype != torch.float32 or A.device != q.device
                or Bs.device != q.device):
            raise ValueError(f"state_out must be contiguous fp32 [{B * Hkv},{S}] and [{B * Hkv},{S},{D}] on {q.device}")
    qv, kv_, vv = (_lib.view4(t)[0] for t in (q, k, v))
    ov = _lib.out_view4(out)
    _lib.check(lib.race_qkv_prefill(sh, qv, kv_, vv, _lib.ptr(planes), ov, _lib.dtype_code(out_dtype), _lib.ptr(A),
                                    _lib.ptr(Bs), _lib.ptr(work), work.numel(), _lib.ptr(scratch), scratch.numel(),
                                    _lib.stream_of(q)), "race_qkv_prefill")
    return out, A, Bs
