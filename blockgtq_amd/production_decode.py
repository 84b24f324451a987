"""Model glue around ``BlockGTQProductionCache`` for Llama-style HF models
(``model.model.embed_tokens / layers / norm``, ``model.lm_head``).

Reference behaviour: blockgtq/production_decode.py:11-99.
"""
import functools

import torch

from .packed_kv_manager import run_decoder_stack

_READ_IN_PLACE = (torch.float16, torch.bfloat16)      # what the encoders take as it lies


@torch.no_grad()
def production_decode_step(model, input_ids, position_ids, cache):
    """One decode step: embed -> per layer (norm, QKV, RoPE, packed encode +
    attention, MLP) -> final norm + lm_head.  Returns logits (B, 1, vocab)."""
    hidden = model.model.embed_tokens(input_ids)
    hidden = run_decoder_stack(model, hidden, position_ids, cache.nq, cache.nkv, cache.hd,
                               cache.encode_and_attend)
    cache.increment_seq_len()
    return model.lm_head(model.model.norm(hidden))


@torch.no_grad()
def production_prefill(model, input_ids, cache, chunk_encode=64):
    """Prefill with the model's own attention, then pack its fp16 K/V.

    Runs the HF forward with a ``DynamicCache`` (``_prompt_cache``), reads the post-RoPE K/V of
    every layer back and encodes the prompt's tokens into ``cache`` (positions a
    model adds behind them stay out).  ``chunk_encode`` bounded the reference
    encoder's temporaries by slicing the prompt; fp16 and bf16 rows are encoded
    where they lie, independently and without temporaries, so they go in one launch
    per layer whatever it is (a 2001-token prompt of 8 KV heads: 374 us in slices
    of 64, host bound, 28 us whole), and it bounds the fp16 copies that rows of
    other types or strides are converted to.  Returns the prompt logits.
    """
    prompt_len = input_ids.shape[1]
    position_ids = torch.arange(prompt_len, device=input_ids.device).unsqueeze(0)
    hf_cache = _prompt_cache()
    out = model(input_ids, position_ids=position_ids, past_key_values=hf_cache, use_cache=True)
    for li in range(cache.n_layers):
        k, v = _layer_kv(hf_cache, li)
        if k.dtype in _READ_IN_PLACE and v.dtype == k.dtype and k.stride(-1) == 1 and v.stride(-1) == 1:
            if k.size(2) > prompt_len:
                k, v = k[:, :, :prompt_len], v[:, :, :prompt_len]
            cache._encode_batched(li, k, v, 0)
            continue
        for lo in range(0, prompt_len, chunk_encode):
            hi = min(lo + chunk_encode, prompt_len)
            cache._encode_batched(li, k[:, :, lo:hi], v[:, :, lo:hi], lo)
    cache.seq_len = prompt_len
    del hf_cache
    return out.logits


def _whole(t):
    """Whether a tensor is all that its storage holds."""
    return t.untyped_storage().nbytes() <= t.numel() * t.element_size()


@functools.lru_cache(maxsize=None)
def _kept_layer():
    """The layer class of ``_prompt_cache`` and the one it stands for (None: a generation without layer objects)."""
    try:
        from transformers.cache_utils import DynamicLayer
    except ImportError:
        return None, None

    class KeptLayer(DynamicLayer):
        def update(self, key_states, value_states, *args, **kwargs):
            if (torch.compiler.is_compiling() or getattr(self, 'is_initialized', True) or
                    not (_whole(key_states) and _whole(value_states))):
                return super().update(key_states, value_states, *args, **kwargs)
            self.lazy_initialization(key_states, value_states)
            self.keys, self.values = key_states, value_states
            return key_states, value_states

    return KeptLayer, DynamicLayer


def _prompt_cache():
    """A ``DynamicCache`` that keeps the first K and V of a layer as the model hands them over.

    ``DynamicCache`` appends them to an empty tensor: two copies of the layer's K and V (20 of 47 us for a 2001-token
    prompt of 8 KV heads) of which nothing is left once the prompt is packed.  What is a part of a larger tensor (a
    projection of queries, keys and values in one) is still copied, so that the rest can be freed; what comes later is
    appended as ever."""
    from transformers import DynamicCache
    cache = DynamicCache()
    kept, plain = _kept_layer()
    if kept is not None and getattr(cache, 'layer_class_to_replicate', None) is plain:
        cache.layer_class_to_replicate = kept
    return cache


def _layer_kv(hf_cache, li):
    """K, V (B, n_kv, T, D) of layer ``li`` from either DynamicCache generation."""
    if hasattr(hf_cache, 'key_cache'):
        return hf_cache.key_cache[li], hf_cache.value_cache[li]
    layer = hf_cache.layers[li]
    return layer.keys, layer.values


__all__ = ["production_decode_step", "production_prefill"]
