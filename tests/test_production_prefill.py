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


class _Reads(_Cache):
    """Reads what it is given when it is given it, as an encoder does."""

    def _encode_batched(self, li, k, v, t_pos):
        super()._encode_batched(li, k.clone(), v.clone(), t_pos)


class _Scratch:
    """Hands every layer's K and V over in the same two tensors, ``piece`` tokens at a time."""

    def __init__(self, k, v, piece, fails_at=None):
        self.k, self.v, self.piece, self.fails_at, self.logits, self.passes = k, v, piece, fails_at, "logits", 0

    def __call__(self, input_ids, position_ids=None, past_key_values=None, use_cache=True):
        self.passes += 1
        n = self.k.shape[-2]
        for lo in range(0, n, self.piece):
            buf_k, buf_v = torch.empty_like(self.k[0, :, :, lo:lo + self.piece]), torch.empty_like(self.v[0, :, :, lo:lo + self.piece])
            for li in range(self.k.shape[0]):
                if li == self.fails_at:
                    raise MemoryError("out of memory")
                buf_k.copy_(self.k[li, :, :, lo:lo + self.piece])
                buf_v.copy_(self.v[li, :, :, lo:lo + self.piece])
                got = past_key_values.update(buf_k, buf_v, li)
                assert torch.equal(got[0], self.k[li, :, :, :lo + self.piece])
                assert torch.equal(got[1], self.v[li, :, :, :lo + self.piece])
        return self


def _layers(tokens, dtype, n=3):
    gen = torch.Generator().manual_seed(tokens)
    return [torch.randn(n, 1, 2, tokens, 8, generator=gen).to(dtype) for _ in range(2)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("piece", [7, 50, 57])
def test_a_model_that_fills_the_same_tensors_for_every_layer(dtype, piece):
    k, v = _layers(57, dtype, 2)
    for tokens in (50, 57):                              # (the prompt ends inside what the model hands over, or with it)
        cache = _Reads()
        model = _Scratch(k, v, piece)
        production_prefill(model, torch.zeros(1, tokens, dtype=torch.long), cache)
        # the prompt at once, then more tokens: the first ones are gone by then, so the pass is made again
        assert model.passes == (2 if piece == tokens == 50 else 1)
        for li in range(2):
            assert sorted(cache.k[li]) == list(range(tokens))
            for s in range(tokens):
                assert torch.equal(cache.k[li][s], k[li][:, :, s]) and torch.equal(cache.v[li][s], v[li][:, :, s])


def test_tokens_behind_a_whole_prompt_and_a_changed_layer():
    k, v = _layers(30, torch.float16, 2)

    class Model:
        logits = "logits"

        def __call__(self, input_ids, past_key_values=None, **kwargs):
            for lo, hi in ((0, 20), (20, 30)):           # tensors of their own for every layer
                for li in range(2):
                    got = past_key_values.update(k[li, :, :, lo:hi].clone(), v[li, :, :, lo:hi].clone(), li)
                    assert torch.equal(got[0], k[li, :, :, :hi]) and torch.equal(got[1], v[li, :, :, :hi])
            past_key_values.layers[1].keys = past_key_values.layers[1].keys + 1
            return self

    cache = _Reads()
    production_prefill(Model(), torch.zeros(1, 20, dtype=torch.long), cache)
    for s in range(20):
        assert torch.equal(cache.k[0][s], k[0][:, :, s]) and torch.equal(cache.k[1][s], (k[1] + 1)[:, :, s])
        assert torch.equal(cache.v[0][s], v[0][:, :, s]) and torch.equal(cache.v[1][s], v[1][:, :, s])


def test_a_cache_that_is_copied_or_cut_in_the_pass():
    import copy
    k, v = _layers(20, torch.float16, 3)

    class Model(_Scratch):
        def __call__(self, input_ids, past_key_values=None, **kwargs):
            other = copy.deepcopy(past_key_values)
            super().__call__(input_ids, past_key_values=past_key_values)
            for li in range(3):                          # a second pass with a cache of its own
                other.update(self.k[li] + 1, self.v[li] + 1, li)
            past_key_values.layers[0].keys = past_key_values.layers[0].keys[:, :, 3:]
            past_key_values.layers[0].values = past_key_values.layers[0].values[:, :, 3:]
            return self

    model, cache = Model(k, v, 20), _Reads()
    production_prefill(model, torch.zeros(1, 17, dtype=torch.long), cache)
    assert model.passes == 2
    for s in range(17):
        assert torch.equal(cache.k[0][s], k[0][:, :, s + 3]) and torch.equal(cache.v[0][s], v[0][:, :, s + 3])
        assert torch.equal(cache.k[1][s], k[1][:, :, s]) and torch.equal(cache.v[1][s], v[1][:, :, s])


@pytest.mark.parametrize("fails_at,left", [(0, 9), (1, 0)])
def test_a_forward_pass_that_fails(fails_at, left):
    k, v = _layers(12, torch.float16, 2)
    cache = _Reads()
    cache.seq_len = 9                                    # of an earlier prompt: gone once a layer is packed over it
    with pytest.raises(MemoryError):
        production_prefill(_Scratch(k, v, 12, fails_at=fails_at), torch.zeros(1, 12, dtype=torch.long), cache)
    assert cache.seq_len == left


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_library_model_is_served_as_with_its_own_cache(dtype):
    from transformers import DynamicCache, Qwen2Config, Qwen2ForCausalLM
    from blockgtq_amd.production_decode import _layer_kv
    torch.manual_seed(5)
    model = Qwen2ForCausalLM(Qwen2Config(vocab_size=64, hidden_size=32, intermediate_size=48, num_hidden_layers=2,
                                         num_attention_heads=4, num_key_value_heads=2)).to(dtype).eval()
    ids, plain, cache = torch.randint(0, 64, (1, 19)), DynamicCache(), _Reads()
    logits = production_prefill(model, ids, cache, chunk_encode=8)
    with torch.no_grad():
        want = model(ids, past_key_values=plain, use_cache=True).logits
    assert torch.equal(logits, want) and cache.seq_len == 19
    for li in range(2):
        k, v = _layer_kv(plain, li)
        assert all(torch.equal(cache.k[li][s], k[:, :, s]) and torch.equal(cache.v[li][s], v[:, :, s]) for s in range(19))


@pytest.mark.parametrize("change", ["arguments", "no such method"])
def test_another_generation_of_the_cache_library(monkeypatch, change):
    """Layers that are set up otherwise than the installed library's: the prompt's K and V are copied, as the library has it."""
    from transformers import cache_utils
    from blockgtq_amd import production_decode
    Plain, Cache = cache_utils.DynamicLayer, cache_utils.DynamicCache

    class OtherLayer(Plain):
        if change == "arguments":
            def lazy_initialization(self, key_states):
                self.is_initialized = True
        else:
            @property
            def lazy_initialization(self):
                raise AttributeError("lazy_initialization")

        def __init__(self):
            self.held, self.is_initialized = Plain(), False

        def update(self, key_states, value_states, *args, **kwargs):
            self.keys, self.values = self.held.update(key_states, value_states, *args, **kwargs)
            self.is_initialized = True
            return self.keys, self.values

    class OtherCache(Cache):
        def __init__(self, *args, **kwargs):
            super().__init__(*args, **kwargs)
            self.layer_class_to_replicate = OtherLayer

    monkeypatch.setattr(cache_utils, "DynamicLayer", OtherLayer)
    monkeypatch.setattr(cache_utils, "DynamicCache", OtherCache)
    monkeypatch.setattr("transformers.DynamicCache", OtherCache)
    production_decode._prompt_classes.cache_clear()
    try:
        k, v = _layers(11, torch.float16, 2)
        cache = _Reads()
        production_prefill(_Scratch(k, v, 11), torch.zeros(1, 11, dtype=torch.long), cache)
    finally:
        production_decode._prompt_classes.cache_clear()
    for li in range(2):
        assert sorted(cache.k[li]) == list(range(11))
        for s in range(11):
            assert torch.equal(cache.k[li][s], k[li][:, :, s]) and torch.equal(cache.v[li][s], v[li][:, :, s])


@pytest.mark.gpu
@pytest.mark.parametrize("aside", [False, True])           # the model's layers on another stream: copied, packed at the end
def test_records_of_a_model_that_fills_the_same_tensors(aside):
    from blockgtq_amd import workloads as wl
    from blockgtq_amd.production_cache import BlockGTQProductionCache
    from blockgtq_amd.quantizer import build_batched_encode_args
    dev, n, T = "cuda:0", 3, 130
    w = wl.Workload("t", n, 4, 2, 1, T, 1e6, seed=51)
    drawn = [wl.calibrate_layer(w, li, dev) for li in range(n)]
    qs = [q for q, _ in drawn]
    ours, want = [BlockGTQProductionCache(qs, [build_batched_encode_args(q, device=dev) for q in qs],
                                          [[q8.build_kernel_args() for q8 in q] for q in qs], n, 2, 4, 128, T + 8, device=dev)
                  for _ in range(2)]
    k, v = (torch.stack(t) for t in zip(*[wl.draw_kv(w, drawn[li][1], T, li, dev) for li in range(n)]))
    for li in range(n):
        want._encode_batched(li, k[li], v[li], 0)
    side, scratch = torch.cuda.Stream(), _Scratch(k, v, T)

    def model(*args, **kwargs):
        if not aside:
            return scratch(*args, **kwargs)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            out = scratch(*args, **kwargs)
        torch.cuda.current_stream().wait_stream(side)
        return out

    production_prefill(model, torch.zeros(1, T, dtype=torch.long, device=dev), ours)
    for name in ("k_packed", "k_norms", "v_packed", "v_norms"):
        assert torch.equal(getattr(ours, name)[:, :, :, :T], getattr(want, name)[:, :, :, :T]), name
