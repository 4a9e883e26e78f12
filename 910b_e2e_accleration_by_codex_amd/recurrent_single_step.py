"""Single-token gated delta rule on the HIP library (drop-in for src/recurrent_single_step.py:8-32).

Same signature, dtypes and semantics as the reference: q, k are l2-normalised in their own dtype
when ``use_qk_l2norm_in_kernel``, the update runs in fp32, the output has query's dtype and the
returned state is a NEW fp32 tensor (the input state is not mutated).  ``inplace=True`` is an
opt-in for callers that own the state (the engine): the kernel then updates ``initial_state`` in
place and returns it, so a following ``copy_`` of it onto itself can be skipped.
For T > 1 the reference falls back to the token loop (src/recurrent_single_step.py:10-13); here
the same loop runs one HIP step per token.
"""
import torch

from . import _lib


def _head_rows(x):
    """[N, T, H, D] as rows of H D values: (tensor whose H and D are dense, slot stride, token stride)."""
    if x.stride(3) != 1 or x.stride(2) != x.shape[3]:
        x = x.contiguous()
    return x, x.stride(0), x.stride(1)


def recurrent_single_step(query, key, value, g, beta, initial_state, output_final_state,
                          use_qk_l2norm_in_kernel=False, inplace=False, **kwargs):
    """query/key [N,T,Hqk,D] (Hqk == Hv after repeat_interleave, or Hv/r key heads), value
    [N,T,Hv,D] (bf16 or fp32, same dtype), g [N,T,Hv] (log decay), beta [N,T,Hv],
    initial_state [N,Hv,D,D] or None.  Returns (out [N,T,Hv,D] in query.dtype, state | None)."""
    if kwargs.get("cu_seqlens") is not None:
        raise NotImplementedError("recurrent_single_step: cu_seqlens is not supported (dense slots)")
    _lib.require_cuda(query, key, value, g, beta, initial_state)
    if key.dtype != query.dtype or value.dtype != query.dtype:
        raise TypeError("recurrent_single_step: query, key and value must share a dtype")
    N, T, Hqk, D = query.shape
    Hv = value.shape[2]
    if key.shape != query.shape or value.shape[:2] != (N, T) or value.shape[3] != D:
        raise ValueError(f"recurrent_single_step: shape mismatch q{tuple(query.shape)} "
                         f"k{tuple(key.shape)} v{tuple(value.shape)}")
    if g.shape != (N, T, Hv) or beta.shape != (N, T, Hv):
        raise ValueError("recurrent_single_step: g and beta must be [N, T, Hv]")
    if g.dtype != torch.float32:
        g = g.to(torch.float32)
    if beta.dtype not in (torch.float32, torch.bfloat16):
        beta = beta.to(torch.float32)
    state_in = None
    if initial_state is not None:
        if initial_state.shape != (N, Hv, D, D):
            raise ValueError(f"recurrent_single_step: state must be [{N},{Hv},{D},{D}]")
        if inplace and (initial_state.dtype != torch.float32 or not initial_state.is_contiguous()):
            raise ValueError("recurrent_single_step: inplace needs a contiguous fp32 state")
        state_in = _lib.f32_dense(initial_state)
    dev = query.device
    if inplace and initial_state is not None:
        state_out = state_in
    else:
        state_out = torch.empty((N, Hv, D, D), dtype=torch.float32, device=dev)
    out = torch.empty((N, T, Hv, D), dtype=query.dtype, device=dev)
    q, qn, qt = _head_rows(query)
    k, kn, kt = _head_rows(key)
    v, vn, vt = _head_rows(value)
    flags = (Hqk, Hv, D, _lib.dtype_code(query), int(bool(use_qk_l2norm_in_kernel)), _lib.stream_of(query))
    bcode = _lib.dtype_code(beta)
    if T == 1:
        g, beta = g.contiguous(), beta.contiguous()
        _lib.call("gdn_recurrent_step", q.data_ptr(), qn, k.data_ptr(), kn, v.data_ptr(), vn, g.data_ptr(),
                  beta.data_ptr(), bcode, _lib.ptr(state_in), state_out.data_ptr(), out.data_ptr(), N, *flags)
    else:
        es = q.element_size()
        cur = state_in
        step_out = torch.empty((N, Hv, D), dtype=query.dtype, device=dev)
        for t in range(T):
            gt, bt = g[:, t].contiguous(), beta[:, t].contiguous()
            _lib.call("gdn_recurrent_step", q.data_ptr() + t * qt * es, qn, k.data_ptr() + t * kt * es, kn,
                      v.data_ptr() + t * vt * es, vn, gt.data_ptr(), bt.data_ptr(), bcode, _lib.ptr(cur),
                      state_out.data_ptr(), step_out.data_ptr(), N, *flags)
            out[:, t].copy_(step_out)
            cur = state_out
    return out, (state_out if output_final_state else None)
