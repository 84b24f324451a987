"""``production_prefill`` on the CPU: which tokens it hands to the cache, in which pieces."""
import pytest
import torch

from blockgtq_amd.production_decode import production_prefill


class _Model:
    """Leaves ``extra`` more positions in its cache than the prompt has (a learned suffix, say)."""

    def __init__(self, k, v):
        self.k, self.v, self.logits = k, v, "logits"

    def __call__(self, input_ids, position_ids=None, past_key_values=None, use_cache=True):
        for li in range(2):
            past_key_values.update(self.k + li, self.v - li, li)
        return self


class _Cache:
    n_layers, seq_len = 2, 0

    def __init__(self):
        self.k, self.v, self.calls = [{}, {}], [{}, {}], []

    def _encode_batched(self, li, k, v, t_pos):
        self.calls.append((li, t_pos, k.shape[2]))
        for s in range(k.shape[2]):
            self.k[li][t_pos + s], self.v[li][t_pos + s] = k[:, :, s], v[:, :, s]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("extra", [0, 5])
@pytest.mark.parametrize("tokens,chunk", [(1, 64), (64, 64), (150, 64), (150, 1000)])
def test_prompt_tokens_once_and_nothing_past_them(dtype, extra, tokens, chunk):
    gen = torch.Generator().manual_seed(tokens)
    k, v = (torch.randn(1, 2, tokens + extra, 8, generator=gen).to(dtype) for _ in range(2))
    cache = _Cache()
    assert production_prefill(_Model(k, v), torch.zeros(1, tokens, dtype=torch.long), cache, chunk_encode=chunk) == "logits"
    assert cache.seq_len == tokens
    for li in range(2):
        assert sorted(cache.k[li]) == list(range(tokens))
        for s in range(tokens):
            assert torch.equal(cache.k[li][s], (k + li)[:, :, s]) and torch.equal(cache.v[li][s], (v - li)[:, :, s])
    # 16-bit tokens are read where they lie, in one launch a layer; others are converted first, a slice at a time
    most = chunk if dtype == torch.float32 else tokens
    assert max(n for _, _, n in cache.calls) <= most
    assert len(cache.calls) == 2 * -(-tokens // most)


def test_prompt_cache_keeps_whole_tensors_and_appends_to_them():
    from transformers import DynamicCache
    from blockgtq_amd.production_decode import _layer_kv, _prompt_cache
    gen = torch.Generator().manual_seed(3)
    k, v = (torch.randn(2, 7, 4, 8, generator=gen).transpose(1, 2) for _ in range(2))       # heads behind tokens in memory
    fused = torch.randn(2, 4, 7, 24, generator=gen)
    k1, v1 = torch.randn(2, 4, 3, 8, generator=gen), torch.randn(2, 4, 3, 8, generator=gen)
    ours, plain = _prompt_cache(), DynamicCache()
    assert isinstance(ours, DynamicCache) and ours.get_seq_length() == 0
    for c in (ours, plain):
        c.update(k, v, 0)
        c.update(fused[..., 8:16], fused[..., 16:], 1)
    assert ours.get_seq_length() == plain.get_seq_length() == 7
    assert _layer_kv(ours, 0)[0].data_ptr() == k.data_ptr() and _layer_kv(ours, 0)[1].data_ptr() == v.data_ptr()
    assert _layer_kv(ours, 1)[0].untyped_storage().nbytes() == 2 * 4 * 7 * 8 * 4            # (not the fused projection)
    before = k.clone()
    for c in (ours, plain):
        got = c.update(k1, v1, 0)
        assert torch.equal(got[0], torch.cat([k, k1], 2)) and torch.equal(got[1], torch.cat([v, v1], 2))
    assert ours.get_seq_length() == plain.get_seq_length() == 10 and torch.equal(k, before)
    for li in range(2):
        for a, b in zip(_layer_kv(ours, li), _layer_kv(plain, li)):
            assert torch.equal(a, b)
