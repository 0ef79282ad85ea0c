"""Drop-ins for the reference's sparse-attention kernel wrappers.

``longcat_active`` keeps the argument meaning, casting and error behaviour of
``MatrixJiTSpatialAcceleration._longcat_active``
(P/matrix_jit_spatial_acceleration.py:663-729) and ``longcat_asymmetric``
those of ``MatrixCausalFrameLayerRelay._longcat_asymmetric``
(P/matrix_curvature_phase_frame_weave.py:8847-8917); both launch the gfx950
HIP kernel ``rcsa_sparse_attn_bf16`` instead of the external Triton
``_attn_fwd_bsa_align``.
"""
from __future__ import annotations

import torch

from . import ops


def longcat_active(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, indices: torch.Tensor,
                   counts: torch.Tensor, valid: torch.Tensor, block_size: int) -> torch.Tensor:
    """Block-sparse attention over packed ``[B, H, L, D]`` tensors.

    q/k/v are cast to bf16 and made contiguous; indices/counts to int32;
    ``valid`` (one flag per packed key token) to uint8.  The query grid is
    ceil(q_len / block_size) blocks of ``block_size`` rows, keys are read in
    ``block_size`` blocks.  Returns bf16 ``[B, H, Lq, D]``.
    """
    q = q.to(torch.bfloat16).contiguous()
    k = k.to(torch.bfloat16).contiguous()
    v = v.to(torch.bfloat16).contiguous()
    indices = indices.to(torch.int32).contiguous()
    counts = counts.to(torch.int32).contiguous()
    key_valid = valid.reshape(-1)
    if block_size % 32 == 0 and key_valid.numel() == k.shape[2] \
            and k.shape[2] % block_size == 0:
        # the validity as bits (32 keys a word): the attention then reads 8 bytes
        # per wavefront and block instead of staging the bytes (about 6% faster)
        ready = _lists_and_bits(q, k, indices, counts, key_valid, block_size, block_size)
        indices, counts, bits = ready or (indices, counts, ops.valid_bits(key_valid, block_size))
        return ops.sparse_attn_bf16(q, k, v, indices, counts, None, block_m=block_size,
                                    block_n=block_size, block_mask=bits, ordered=True)
    return ops.sparse_attn_bf16(q, k, v, indices, counts, key_valid.to(torch.uint8).contiguous(),
                                block_m=block_size, block_n=block_size)


def _lists_and_bits(q, k, indices, counts, key_valid, block_m, block_n):
    """(lists in ascending order, validity bits) from one launch where the order pays,
    else None (also when the lists have not the attention's form, which then refuses
    them itself)."""
    B, H, L, D = k.shape
    if not (indices.ndim == 4 and k.is_cuda
            and ops.order_pays(B * H, q.shape[2], L, 4 * D, block_m, block_n, indices.shape[3])):
        return None
    if (indices.is_cuda and counts.is_cuda and key_valid.is_cuda and counts.ndim == 3
            and all(t.shape[:2] in ((B, H), (1, H), (B, 1), (1, 1)) for t in (indices, counts))
            and ops.lists_cover(indices, counts, q.shape[2], block_m)):
        return ops.order_for_attention(indices, counts, q.shape, L, block_m, block_n,
                                       valid=key_valid)
    return None


def _bits_pay(q, k, block_m, block_n, max_k) -> bool:
    """Whether the validity as bits, whose forms of the attention are faster, is worth the
    launch that makes them: keys beyond an XCD's L2, and two rounds of query blocks or
    28 MB of listed blocks an XCD, 48 MB where its keys are 16 MB (64 x 128 blocks, 24
    heads x 3520 rows x 12 of 42 blocks 102 us against 145 with bytes, 8 x 1760 x 38 of 128
    63 against 71, 24 x 880 x 11 of 43 41.6 against 43.0, 8 x 1760 x 12 of 128 31 against
    29, 12 x 880 x 30 of 303 57.0 against 55.8)."""
    B, H, L, D = k.shape
    n_bh = B * H
    if not (k.is_cuda and ops.order_helps(n_bh, L, 4 * D, block_n, max_k)):
        return False
    least = 28 if -(-n_bh // 8) * L * 4 * D <= 16 << 20 else 48
    return (ops.two_rounds(n_bh, q.shape[2], block_m)
            or ops.listed_bytes(n_bh, q.shape[2], 4 * D, block_m, block_n, max_k) > least << 20)


def longcat_asymmetric(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                       indices: torch.Tensor, counts: torch.Tensor, key_valid: torch.Tensor,
                       *, query_block_size: int, key_block_size: int) -> torch.Tensor:
    """Asymmetric query/key storage; both lengths must be block aligned."""
    q = q.to(torch.bfloat16).contiguous()
    k = k.to(torch.bfloat16).contiguous()
    v = v.to(torch.bfloat16).contiguous()
    indices = indices.to(torch.int32).contiguous()
    counts = counts.to(torch.int32).contiguous()
    valid = key_valid.reshape(-1)  # (a bool's bytes are its uint8 values)
    valid = (valid.contiguous().view(torch.uint8) if valid.dtype == torch.bool
             else valid.to(torch.uint8).contiguous())
    if q.shape[2] % query_block_size or k.shape[2] % key_block_size:
        raise RuntimeError("asymmetric sparse storage is not block aligned")
    if key_block_size % 32 == 0 and valid.numel() == k.shape[2]:
        ready = _lists_and_bits(q, k, indices, counts, valid, query_block_size, key_block_size)
        bits = None
        if ready is not None:
            indices, counts, bits = ready
        elif indices.ndim == 4 and valid.device == k.device \
                and _bits_pay(q, k, query_block_size, key_block_size, indices.shape[3]):
            bits = ops.valid_bits(valid, key_block_size)
        if bits is not None:  # (a few blocks: the bytes, without another launch)
            return ops.sparse_attn_bf16(q, k, v, indices, counts, None,
                                        block_m=query_block_size, block_n=key_block_size,
                                        block_mask=bits, ordered=True)
    return ops.sparse_attn_bf16(q, k, v, indices, counts, valid, block_m=query_block_size,
                                block_n=key_block_size, ordered=True)
