"""Model glue around ``BlockGTQProductionCache`` for Llama-style HF models
(``model.model.embed_tokens / layers / norm``, ``model.lm_head``).

Reference behaviour: blockgtq/production_decode.py:11-99.
"""
import functools

import torch

from . import _host
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

    Runs the HF forward with a ``DynamicCache`` (``_prompt_cache``) and encodes the post-RoPE K/V of the
    prompt's tokens of every layer into ``cache`` (positions a model adds behind them stay out): a
    layer that the model hands over whole as it arrives, so that the model may write the same tensors again
    for its next layer, others behind the forward pass.  (A model that does so and then appends to or changes an
    earlier layer of the cache within one pass runs once more, with a cache that copies; what it reads there is what it
    has written since.)  ``chunk_encode`` bounded the reference
    encoder's temporaries by slicing the prompt; fp16 and bf16 rows are encoded
    where they lie, independently and without temporaries, so they go in one launch
    per layer whatever it is (a 2001-token prompt of 8 KV heads: 374 us in slices
    of 64, host bound, 26 us whole), and it bounds the fp16 copies that rows of
    other types or strides are converted to.  A forward pass that fails behind its first packed
    layer leaves ``cache`` empty.  Returns the prompt logits.
    """
    prompt_len = input_ids.shape[1]
    position_ids = torch.arange(prompt_len, device=input_ids.device).unsqueeze(0)
    home = _stream(input_ids)

    def pack(li, k, v):
        if k.dtype in _READ_IN_PLACE and v.dtype == k.dtype and k.stride(-1) == 1 and v.stride(-1) == 1:
            if k.size(2) > prompt_len:
                k, v = k[:, :, :prompt_len], v[:, :, :prompt_len]
            cache._encode_batched(li, k, v, 0)
            return
        for lo in range(0, prompt_len, chunk_encode):
            hi = min(lo + chunk_encode, prompt_len)
            cache._encode_batched(li, k[:, :, lo:hi], v[:, :, lo:hi], lo)

    def arrived(li, k, v):
        # (on another stream the cache's records may still be read by what was launched before: packed at the end)
        if li >= cache.n_layers or k.size(2) < prompt_len or _stream(k) != home:
            return False
        cache.seq_len = 0          # (until the forward pass is over: whatever was there, this layer's records are gone)
        pack(li, k, v)
        return True

    for copies in (False, True):
        hf_cache = _prompt_cache(arrived, copies)
        try:
            out = model(input_ids, position_ids=position_ids, past_key_values=hf_cache, use_cache=True)
        except _Refilled:
            continue
        packed = getattr(hf_cache, 'kept', {})
        rest = []
        for li in range(cache.n_layers):
            k, v = _layer_kv(hf_cache, li)
            was = packed.get(li)
            if was is None or was[0] is not k or was[1] is not v:   # (or appended to, cut, replaced since)
                rest.append((li, k, v))
        if not packed or hf_cache.refilled.isdisjoint(li for li, _, _ in rest):
            break
    for li, k, v in rest:
        pack(li, k, v)
    cache.seq_len = prompt_len
    del hf_cache
    return out.logits


class _Refilled(Exception):
    """Tokens were to be appended to kept ones that are gone."""


def _stream(t):
    return _host.module().stream(t) if t.is_cuda else None


def _whole(t):
    """Whether a tensor is all that its storage holds."""
    return type(t) is torch.Tensor and 0 < t.untyped_storage().nbytes() <= t.numel() * t.element_size()


def _kept_layer(Layer):
    """``Layer`` that takes its first K and V as they are."""

    class KeptLayer(Layer):
        def update(self, key_states, value_states, *args, **kwargs):
            if self.is_initialized or torch.compiler.is_compiling() or not (_whole(key_states) and _whole(value_states)):
                return super().update(key_states, value_states, *args, **kwargs)
            self.dtype, self.device, self.is_initialized = key_states.dtype, key_states.device, True
            self.keys, self.values = key_states, value_states
            return key_states, value_states

    return KeptLayer


def _stands_for(kept, plain):
    """Whether a layer with its first token kept has what one that copied it has, and grows by the next one alike."""
    one, kept, plain = torch.empty(1, 1, 1, 1, device="cpu"), kept(), plain()
    if kept.update(one, one)[0] is not one or kept.is_initialized is not True:
        return False
    plain.update(one, one)
    mine, theirs = vars(kept), vars(plain)
    return (mine.keys() == theirs.keys() and mine['keys'] is one and mine['values'] is one and
            all(torch.is_tensor(x) or x == mine[name] for name, x in theirs.items()) and
            kept.update(one, one)[0].shape == kept.keys.shape == kept.values.shape == (1, 1, 2, 1))


def _kept_cache(Cache):
    """``Cache`` with what ``_prompt_cache`` says of kept layers."""

    class KeptCache(Cache):
        def update(self, key_states, value_states, layer_idx, *args, **kwargs):
            if torch.compiler.is_compiling():
                return super().update(key_states, value_states, layer_idx, *args, **kwargs)
            if self.kept:
                self.look_for(key_states, value_states, layer_idx)
            keys, values = super().update(key_states, value_states, layer_idx, *args, **kwargs)
            if keys is key_states and values is value_states:
                if self.arrived is None or self.me == id(self) and self.arrived(layer_idx, keys, values):
                    self.kept[layer_idx] = keys, values
                else:
                    keys, values = keys.clone(), values.clone()
                    self.layers[layer_idx].keys, self.layers[layer_idx].values = keys, values
            return keys, values

        def look_for(self, key_states, value_states, layer_idx):
            for li in list(self.kept)[self.listed:]:
                for t in self.kept[li]:
                    self.where[t.untyped_storage().data_ptr()] = li
            self.listed = len(self.kept)
            for t in (key_states, value_states):
                if type(t) is torch.Tensor:
                    self.refilled.add(self.where.get(t.untyped_storage().data_ptr()))
            if layer_idx in self.refilled:
                raise _Refilled(f"the K and V kept of layer {layer_idx} were written again, and more tokens follow")

    return KeptCache


@functools.lru_cache(maxsize=None)
def _prompt_classes():
    """The cache class of ``_prompt_cache``, and its layer class with the one that stands for (None, None: a generation
    without layer objects, or with ones that start, hold or grow otherwise than a kept layer does)."""
    from transformers import DynamicCache
    try:
        from transformers.cache_utils import DynamicLayer
        kept = _kept_layer(DynamicLayer)
        if _stands_for(kept, DynamicLayer) and getattr(DynamicCache(), 'layer_class_to_replicate', None) is DynamicLayer:
            return DynamicCache, _kept_cache(DynamicCache), kept
    except (ImportError, AttributeError, KeyError, TypeError):
        pass
    return DynamicCache, None, None


def _prompt_cache(arrived=None, copies=False):
    """A ``DynamicCache`` that keeps the first K and V of a layer as the model hands them over.

    ``DynamicCache`` appends them to an empty tensor: two copies of the layer's K and V (20 of 47 us for a 2001-token
    prompt of 8 KV heads) of which nothing is left once the prompt is packed.  What is a part of a larger tensor (a
    projection of queries, keys and values in one) is still copied, so that the rest can be freed; what comes later is
    appended as ever.

    Nothing says that the model leaves a kept layer's tensors alone for the rest of its pass.  ``arrived(layer, k, v)``
    therefore reads them then and there; where it returns False they are copied after all.  Memory that comes back with
    another layer, or with more tokens of the same one, was filled again: the layer that was there is in ``refilled``,
    appending to it raises ``_Refilled``, and the pass has to be made again with ``copies``, a plain ``DynamicCache``."""
    plain, kept_cache, kept_layer = _prompt_classes()
    if copies or kept_cache is None:
        return plain()
    cache = kept_cache()
    cache.layer_class_to_replicate = kept_layer
    # me: not a copy of it that the model made; kept: layer -> K, V; where: address -> layer, of the first `listed` ones; refilled: layers whose memory came again
    cache.arrived, cache.me, cache.kept, cache.where, cache.listed, cache.refilled = arrived, id(cache), {}, {}, 0, set()
    return cache


def _layer_kv(hf_cache, li):
    """K, V (B, n_kv, T, D) of layer ``li`` from either DynamicCache generation."""
    if hasattr(hf_cache, 'key_cache'):
        return hf_cache.key_cache[li], hf_cache.value_cache[li]
    layer = hf_cache.layers[li]
    return layer.keys, layer.values


__all__ = ["production_decode_step", "production_prefill"]
