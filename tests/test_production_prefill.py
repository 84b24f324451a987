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
