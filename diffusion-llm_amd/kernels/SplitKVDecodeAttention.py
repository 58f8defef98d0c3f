"""Split-KV (FlashDecoding) attention for BD3-LM cached sampling, on MI355X.

Drop-in for the reference's kernels/SplitKVDecodeAttention.py:
`split_kv_decode_attention(q, k, v, block_size)` gives the same result as
block_sparse_decode_attention with the keys split across workgroups; each
range of keys writes a normalised fp32 partial and its LSE, merged with LSE
weights. Adds an optional `n_splits` (default: the reference rule
ceil(kv_len / SPLIT_N), :147): the most ranges the keys are cut into. Up to 64
queries are cut into no more than fill the GPU (256 workgroups over all
sequences, heads and query tiles), the call's result being the same;
bd3_decode_ranges tells the number. Runs bd3_decode_splitkv in libbd3attn.so.
"""
import torch
from torch import Tensor

from kernels._native import host
from kernels.BlockSparseDecodeAttention import _check_decode_inputs, block_sparse_decode_attention

# keys per split of the reference's default split rule
SPLIT_N = 256


def split_kv_decode_attention(
    q: Tensor,  # (batch, heads, q_len, head_dim): the last q_len positions
    k: Tensor,  # (batch, heads, kv_len, head_dim)
    v: Tensor,
    block_size: int,
    n_splits: int | None = None,
) -> Tensor:
    """Same result as block_sparse_decode_attention, with the keys split
    across workgroups so a decode step fills the GPU, into at most n_splits
    ranges (reference: kernels/SplitKVDecodeAttention.py:130-171)."""
    kv_len = k.shape[2]
    if q.shape[2] > 64 and n_splits is None:
        # prefill: many query tiles already fill the GPU (reference :140-142)
        return block_sparse_decode_attention(q, k, v, block_size)
    _check_decode_inputs(q, k, v)
    return host().decode(q, k, v, block_size, split_count(kv_len, n_splits))


def split_count(kv_len: int, n_splits: int | None) -> int:
    """n_splits, or the reference's count where it is None."""
    if n_splits is None:
        n_splits = -(-kv_len // SPLIT_N)
    assert 1 <= n_splits <= kv_len, "n_splits must be in [1, kv_len]"
    return n_splits
