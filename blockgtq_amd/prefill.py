"""Layer-major prefill into a packed cache.

All prompt tokens go through one transformer layer at a time: QKV + RoPE for
the whole prompt, one quantise-and-pack launch per K and V, causal attention
over the records just written, MLP.  No fp16 KV cache of the full model is
ever materialised; while a layer attends, its visible records lie dequantised in
a transient workspace (512 bytes a record and KV head).  Reference behaviour:
blockgtq/prefill.py:24-111.

As in the reference, attention inside the prompt sees the *quantised* keys and
values (what later decode steps will see), not the layer's fp16 K/V:
``bgtq_prompt_attn`` stages the records' values once per call, rotates the model's
queries itself and attends on the matrix cores.
"""
import torch

from . import ops
from .packed_kv_manager import run_decoder_stack


def _layer_matrices(cache, li):
    """Per-KV-head query transform (D, D) = permutation then rotation, stacked over the heads of layer
    ``li`` (built once)."""
    store = cache.__dict__.setdefault('_prefill_mats', {})
    if li not in store:
        qm = []
        for q8 in cache.quantizers[li]:
            m = torch.zeros(cache.hd, cache.hd, dtype=torch.float32, device=q8._block_rot_T.device)
            m[q8._head_perm] = q8._block_rot_T.float()           # q[:, head_perm] @ R^T == q @ m
            qm.append(m)
        store[li] = torch.stack(qm)
    return store[li]


def packed_prefill_attention(cache, li, q, T, q_pos_offset=0):
    """Causal attention of q (B, n_q, S, D) over records ``[0, T)`` of layer ``li``
    of a ``BlockGTQProductionCache``; returns (B, n_q, S, D) fp16."""
    B, n_q, S, D = q.shape
    rotate = not cache.quantizers[li][0]._q_perm_baked
    with torch.no_grad():
        if not rotate:
            q = q.to(torch.float16)
        elif q.dtype not in (torch.float16, torch.bfloat16):     # (the kernel rotates 16-bit queries)
            qg = q.reshape(B, cache.nkv, cache.gqa * S, D).float()
            q = (qg @ _layer_matrices(cache, li).unsqueeze(0)).to(torch.float16).reshape(B, n_q, S, D)
            rotate = False
        return ops.prefill_attention_records(
            cache.batched_args[li]['plans'], q, cache.k_packed[li], cache.k_norms[li], cache.v_packed[li], cache.v_norms[li], T,
            k_layout=cache._k_layout, v_layout=cache._v_layout, scale=cache.scale, is_causal=True,
            q_pos_offset=q_pos_offset, k_row_width=cache.k_bytes_per_tok, v_row_width=cache.vpb, rotate_q=rotate)


@torch.no_grad()
def layer_major_prefill(model, cache, prompt_ids, block_q=32, block_t=128):
    """Populate ``cache`` for positions ``[0, T)`` and set ``cache.seq_len = T``.

    ``prompt_ids`` is (B, T); B must match the cache's batch size.  ``block_q``
    and ``block_t`` tuned the reference's kernel and are ignored.
    """
    B, T = prompt_ids.shape
    pos = torch.arange(T, device=prompt_ids.device).unsqueeze(0).expand(B, -1)
    hidden = model.model.embed_tokens(prompt_ids)

    def attend(li, q, k, v):
        cache._encode_batched(li, k, v, 0)
        return packed_prefill_attention(cache, li, q, T)

    hidden = run_decoder_stack(model, hidden, pos, cache.nq, cache.nkv, cache.hd, attend)
    cache.seq_len = T
    return hidden


__all__ = ["layer_major_prefill", "packed_prefill_attention"]
