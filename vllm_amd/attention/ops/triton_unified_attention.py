"""The V1 engine's attention over the flash-layout KV cache: mirror of
vllm/attention/ops/triton_unified_attention.py:588-700 (`unified_attention`, same arguments)
over `vllm_amd_unified_attention` (HIP, prefill_attention.hip) instead of the Triton kernels."""
from __future__ import annotations

import torch

from ... import _torch_ops

_DT = (torch.float16, torch.bfloat16)
_FP8 = (torch.uint8, torch.float8_e4m3fn)


def _i32(t: torch.Tensor) -> torch.Tensor:
    return t if t.dtype == torch.int32 else t.to(torch.int32)


def unified_attention(q, k, v, out, cu_seqlens_q, max_seqlen_q, seqused_k, max_seqlen_k,
                      softmax_scale, causal, window_size, block_table, softcap, q_descale,
                      k_descale, v_descale, alibi_slopes=None, output_scale=None) -> None:
    assert causal, "Only causal attention is supported"
    assert q_descale is None, "Q scales not supported"
    if q.dtype not in _DT:
        raise RuntimeError(f"unified_attention: unsupported query dtype {q.dtype}")
    fp8 = k.dtype in _FP8
    if fp8:
        assert v.dtype in _FP8 and k_descale is not None and v_descale is not None
    else:
        assert k.dtype == q.dtype and v.dtype == q.dtype
    assert cu_seqlens_q.shape[0] == seqused_k.shape[0] + 1
    for t in (q, out, k, v):
        assert t.stride(-1) == 1
    cu_seqlens_q, seqused_k, block_table = _i32(cu_seqlens_q), _i32(seqused_k), _i32(block_table)
    assert block_table.stride(1) == 1 and cu_seqlens_q.is_contiguous() and seqused_k.is_contiguous()
    if output_scale is not None:
        assert out.dtype in _FP8
    else:
        assert out.dtype == q.dtype
    # (scratch for launches that split the keys -- the reference's segm_* tensors, :659-683 -- is allocated in there)
    _torch_ops.unified_attention(q, k, v, out, cu_seqlens_q, int(max_seqlen_q), seqused_k, int(max_seqlen_k),
                                 float(softmax_scale), 1 + int(window_size[0]), block_table, float(softcap or 0.0), k_descale, v_descale, alibi_slopes,
                                 output_scale)
