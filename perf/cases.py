"""Workloads of the packed-KV path, one pass of each through the public entry points.

Five kinds of work:

``decode``   one decode step of some layers: append one token per sequence, attend over the packed
             cache (``BlockGTQKVManager.append_and_attend`` or
             ``BlockGTQProductionCache.encode_and_attend``), launched eagerly as a model's Python
             loop does or replayed as one HIP graph as a serving loop does;
``pack``     a whole fp16/bf16 prompt cache into the packed cache (``BlockGTQKVManager.init_from_cache``);
``chunks``   the same into the production cache in slices, as ``production_prefill`` does after the
             model's own forward pass;
``prompt``   causal attention of prompt tokens over packed records (``packed_prefill_attention``),
             whole prompts and later chunks of one;
``head``     ``fused_blockgtq_decode_attention``, the entry that takes one KV head's slice at a time.

Every case is a dict of plain values; ``listed()`` has the ones looked at every time, ``draw()`` gives
more of the same ranges.
"""
import dataclasses
import math

import torch

from blockgtq_amd import workloads as wl
from blockgtq_amd.kernels import fused_blockgtq_decode_attention
from blockgtq_amd.packed_kv_manager import BlockGTQKVManager
from blockgtq_amd.prefill import packed_prefill_attention
from blockgtq_amd.production_cache import BlockGTQProductionCache
from blockgtq_amd.production_decode import production_prefill
from blockgtq_amd.quantizer import build_batched_encode_args

DEV = "cuda:0"
D = 128
ROPE = 1e6
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
K_GROUPS = 5            # norm groups of a K record: one per bit width in use (1..5 bits at an average of 3)


def listed():
    geo8b = {"n_q": 32, "n_kv": 8}           # 4 query heads per KV head, 8 KV heads
    geo3b = {"n_q": 16, "n_kv": 2}           # 8 query heads per KV head, 2 KV heads
    k3v3 = {"k_bits": 3.0, "v_bits": 3, "min_bits": 1, "max_bits": 8}
    step = {"kind": "decode", "ragged": False, "sink": 0, "window": 0, "heavy_tail": False, **k3v3}
    return [
        # an existing call site that loops over KV heads, short context: the smallest call there is
        {"name": "head_call_b1_1k", "kind": "head", "batch": 1, "gqa": 4, "context": 1025, "nibble": False, **k3v3},
        # one user chatting: batch 1, 4k tokens, the model's Python loop in bf16
        {"name": "decode_8b_b1_4k_eager", "cache": "manager", "nibble": False, "graph": False, "dtype": "bf16",
         "batch": 1, "context": 4096, "layers": 4, **geo8b, **step, "max_bits": 5},
        # the headline: 8 sequences of 32k tokens, the whole step replayed as a graph
        {"name": "decode_3b_b8_32k_graph", "cache": "manager", "nibble": False, "graph": True, "dtype": "fp16",
         "batch": 8, "context": 32768, "layers": 6, **geo3b, **step},
        # the same sequences in the production cache's default layout (nibbles), eager, bf16 model
        {"name": "decode_3b_b8_32k_nibble_eager", "cache": "production", "nibble": True, "graph": False, "dtype": "bf16",
         "batch": 8, "context": 32768, "layers": 4, **geo3b, **step},
        # end-to-end generation after an 8k prompt: lengths kept on the device, one graph per token
        {"name": "decode_3b_b4_8k_graph", "cache": "production", "nibble": False, "graph": True, "dtype": "bf16",
         "batch": 4, "context": 8200, "layers": 8, **geo3b, **step, "max_bits": 5},
        # one very long document at 2 bits, heavy-tailed values, 0-bit blocks
        {"name": "decode_8b_b1_128k_k2v2_graph", "cache": "manager", "nibble": False, "graph": True, "dtype": "fp16",
         "batch": 1, "context": 131072, "layers": 2, **geo8b, **step, "k_bits": 2.0, "v_bits": 2, "min_bits": 0,
         "max_bits": 4, "heavy_tail": True},
        # a busy server: 32 ragged sequences, fp16 sink tokens and recent window beside the packed cache
        {"name": "decode_8b_b32_ragged_window_graph", "cache": "manager", "nibble": False, "graph": True, "dtype": "fp16",
         "batch": 32, "context": 16384, "layers": 2, **geo8b, **step, "ragged": True, "sink": 4, "window": 128},
        # a ragged batch at higher quality with an odd query group, eager
        {"name": "decode_gqa7_b12_ragged_k4v4_eager", "cache": "production", "nibble": False, "graph": False,
         "dtype": "fp16", "batch": 12, "context": 3001, "layers": 4, "n_q": 28, "n_kv": 4, **step, "ragged": True,
         "k_bits": 4.0, "v_bits": 4},
        # a batch of long prompts packed in one go
        {"name": "pack_3b_b4_8k", "kind": "pack", "batch": 4, "n_kv": 2, "context": 8192, "layers": 2, "dtype": "bf16",
         **k3v3},
        # one prompt packed in slices of 64 tokens behind the model's own prefill
        {"name": "pack_chunks_8b_b1_2k", "kind": "chunks", "batch": 1, "n_kv": 8, "context": 2001, "layers": 1,
         "chunk": 64, "nibble": True, "dtype": "bf16", **k3v3},
        # a batch of whole 8k prompts attending over the records just written
        {"name": "prompt_3b_b4_8k", "kind": "prompt", "batch": 4, **geo3b, "queries": 8192, "context": 8192,
         "nibble": False, "dtype": "bf16", **k3v3, "max_bits": 5},
        # a later chunk of one prompt
        {"name": "prompt_chunk_8b_b1_1k_of_4k", "kind": "prompt", "batch": 1, **geo8b, "queries": 1000,
         "context": 4100, "nibble": True, "dtype": "fp16", **k3v3},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _bits(rng):
    k, v, lo, hi = rng.choice([(3.0, 3, 1, 8), (3.0, 3, 1, 5), (2.0, 2, 0, 4), (4.0, 4, 1, 8), (2.5, 3, 1, 4),
                               (3.5, 4, 1, 6), (3.0, 2, 0, 5)])
    return {"k_bits": k, "v_bits": v, "min_bits": lo, "max_bits": hi}


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "decode", "pack", "chunks", "prompt", "prompt", "head"])
    bits = _bits(rng)
    dtype = rng.choice(["fp16", "bf16"])
    nibble = rng.random() < 0.35
    n_kv = rng.choice([1, 2, 4, 8])
    gqa = rng.choice([1, 2, 3, 4, 4, 5, 6, 7, 8, 8, 12, 16])
    if kind == "head":
        batch = _log(rng, 1, 8)
        return {"kind": kind, "batch": batch, "gqa": gqa, "context": _log(rng, 64, 65536 // batch), "nibble": nibble, **bits}
    if kind == "decode":
        batch = _log(rng, 1, 32)
        most = min(131072, 8 * 2 * 32768 // (batch * n_kv))
        cache = "production" if nibble else rng.choice(["manager", "production"])
        ragged = batch > 1 and rng.random() < 0.3
        buffered = cache == "manager" and rng.random() < 0.25
        context = _log(rng, 256 if buffered else 16, most)
        layers = max(1, min(rng.randint(1, 6), 6 * 8 * 2 * 32768 // (batch * n_kv * context)))
        return {"kind": kind, "cache": cache, "nibble": nibble, "graph": rng.random() < 0.5, "dtype": dtype,
                "batch": batch, "context": context, "layers": layers, "n_q": n_kv * gqa, "n_kv": n_kv,
                "ragged": ragged, "sink": 4 if buffered else 0, "window": rng.choice([64, 128]) if buffered else 0,
                "heavy_tail": rng.random() < 0.2, **bits}
    if kind == "pack":
        batch = _log(rng, 1, 16)
        return {"kind": kind, "batch": batch, "n_kv": n_kv, "context": _log(rng, 65, min(32768, 65536 // (batch * n_kv))),
                "layers": rng.randint(1, 2), "dtype": dtype, **bits}
    if kind == "chunks":
        batch = _log(rng, 1, 4)
        return {"kind": kind, "batch": batch, "n_kv": n_kv, "context": _log(rng, 100, 4096 // batch), "layers": 1,
                "chunk": rng.choice([64, 64, 100, 256]), "nibble": rng.random() < 0.6, "dtype": dtype, **bits}
    batch = _log(rng, 1, 4)
    queries = _log(rng, 16, 8192)
    before = 0 if rng.random() < 0.6 else _log(rng, 16, 16384 - queries)
    # no more query-record pairs than 4 x 16 heads over a whole 8k prompt
    while batch * n_kv * gqa * queries * (before + queries / 2) > 4 * 16 * 8192 * 4096:
        queries, before = max(16, queries * 3 // 4), before * 3 // 4
    return {"kind": kind, "batch": batch, "n_q": n_kv * gqa, "n_kv": n_kv, "queries": queries,
            "context": before + queries, "nibble": nibble, "dtype": dtype, **bits}


# ------------------------------------------------------------------------------------ preparation
def _workload(c, **kw):
    """The case's geometry.  Its seed is the one of the calibration, which a model has once; the data
    is drawn from ``_data(w, seed)``."""
    n_kv = c.get("n_kv", 1)
    n_q = c.get("n_q", n_kv * c.get("gqa", 1))
    return wl.Workload("case", c.get("layers", 1), n_q, n_kv, c["batch"], c["context"], ROPE,
                       k_bits=c["k_bits"], v_bits=c["v_bits"], min_bits=c["min_bits"], max_bits=c["max_bits"],
                       student_t_nu=4 if c.get("heavy_tail") else None, seed=1235, n_sink=c.get("sink", 0),
                       window=c.get("window", 0), **kw)


def _data(w, seed):
    return dataclasses.replace(w, seed=seed)


class _Prompt:
    """A model as ``production_prefill`` sees one: its forward pass leaves post-RoPE K and V in the
    cache it is given.  Here they are at hand already, so that a pass is the packing alone."""

    def __init__(self, kv):
        self.kv = kv

    def __call__(self, input_ids, position_ids=None, past_key_values=None, use_cache=True):
        for li, (k, v) in enumerate(self.kv):
            past_key_values.update(k, v, li)
        self.logits = None
        return self


class _PromptCache:
    """Per-layer K and V of a finished forward pass, as ``init_from_cache`` reads them."""

    def __init__(self, kv):
        self.key_cache = [k for k, _ in kv]
        self.value_cache = [v for _, v in kv]


def _production(c, w, max_T):
    quantizers, args, kernel_args, energies = [], [], [], []
    for li in range(w.n_layers):
        qs, e = wl.calibrate_layer(w, li, DEV)
        quantizers.append(qs)
        energies.append(e)
        args.append(build_batched_encode_args(qs, device=DEV))
        kernel_args.append([q.build_kernel_args() for q in qs])
    cache = BlockGTQProductionCache(quantizers, args, kernel_args, w.n_layers, w.n_kv, w.n_q, D, max_T, v_bits=w.v_bits,
                                    k_nibble=c["nibble"], v_nibble=c["nibble"], device=DEV, batch_size=w.batch)
    return cache, energies


def _prompt_kv(c, w, seed, energies, tokens):
    dt = DTYPES[c.get("dtype", "fp16")]
    return [tuple(t.to(dt) for t in wl.draw_kv(_data(w, seed), energies[li], tokens, li, DEV)) for li in range(w.n_layers)]


def _ids(w, tokens):
    return torch.zeros(w.batch, tokens, dtype=torch.long, device=DEV)


def _prepare_decode(c, seed):
    gen = torch.Generator().manual_seed(seed)
    T = c["context"]
    lens = None
    if c["ragged"]:
        lo = max(T // 16, c["sink"] + c["window"] + 1, 1)
        lens = torch.randint(lo, T + 1, (c["batch"],), generator=gen).tolist()
        lens[0] = T                                  # (the longest row is the declared context)
    w = _workload(c, seq_lens=lens)
    dt = DTYPES[c["dtype"]]
    if c["cache"] == "manager":
        owner, energies = wl.build_manager(w, DEV, max_T=T + 64)
        if owner.buffered:
            for li in range(w.n_layers):
                k, v = wl.draw_kv(_data(w, seed), energies[li], T, li, DEV)
                owner.fill_buffered(li, k, v, lens)
                del k, v
            owner.set_seq_lens(lens or [T] * w.batch)
        else:
            for li in range(w.n_layers):
                k, v = wl.draw_kv(_data(w, seed), energies[li], T, li, DEV)
                owner._encode_kv(li, k, v, 0)
                del k, v
            owner.seq_len = T
            if lens:
                owner.set_seq_lens(lens)
        step = owner.append_and_attend
        buffers = [owner._k_packed, owner._k_norms, owner._v_packed, owner._v_norms]
        if owner.buffered:
            buffers += [owner._buf_k, owner._buf_v]
    else:
        owner, energies = _production(c, w, T + 264)
        production_prefill(_Prompt(_prompt_kv(c, w, seed, energies, T)), _ids(w, T), owner, chunk_encode=max(T, 1))
        if lens:
            owner.set_seq_lens(lens)
        if c["graph"]:
            owner.use_device_lengths()
        step = owner.encode_and_attend
        buffers = [owner.k_packed, owner.k_norms, owner.v_packed, owner.v_norms]
    qs = [wl.draw_q(_data(w, seed), li, DEV, T).to(dt) for li in range(w.n_layers)]
    kvs = [tuple(t.to(dt) for t in wl.draw_kv(_data(w, seed), energies[li], 1, 1000 + li, DEV, pos0=T))
           for li in range(w.n_layers)]
    layers = range(w.n_layers)

    def one_step():
        return [step(li, qs[li], kvs[li][0], kvs[li][1]) for li in layers]

    if not c["graph"]:
        return {"run": lambda: [one_step(), buffers], "owner": owner}
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            one_step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = one_step()

    def replay():
        graph.replay()
        return [outs, buffers]

    return {"run": replay, "owner": owner, "graph": graph}


def _prepare_pack(c, seed):
    w = _workload(c)
    mgr, energies = wl.build_manager(w, DEV, max_T=c["context"] + 64)
    past = _PromptCache(_prompt_kv(c, w, seed, energies, c["context"]))

    def run():
        mgr.init_from_cache(past)
        return [mgr._k_packed, mgr._k_norms, mgr._v_packed, mgr._v_norms]

    return {"run": run}


def _prepare_chunks(c, seed):
    w = _workload(c)
    T = c["context"]
    cache, energies = _production(c, w, T + 64)
    model, ids = _Prompt(_prompt_kv(c, w, seed, energies, T)), _ids(w, T)

    def run():
        production_prefill(model, ids, cache, chunk_encode=c["chunk"])
        return [cache.k_packed, cache.k_norms, cache.v_packed, cache.v_norms]

    return {"run": run}


def _prepare_prompt(c, seed):
    w = _workload(c)
    T, S = c["context"], c["queries"]
    cache, energies = _production(c, w, T + 64)
    production_prefill(_Prompt(_prompt_kv(c, w, seed, energies, T)), _ids(w, T), cache, chunk_encode=T)
    gen = torch.Generator(device=DEV).manual_seed(seed + 77)
    # as a projection leaves them: (B, S, heads, D) in memory
    q = torch.randn(w.batch, S, w.n_q, D, generator=gen, device=DEV).to(DTYPES[c["dtype"]]).transpose(1, 2)
    return {"run": lambda: packed_prefill_attention(cache, 0, q, T, T - S)}


def _prepare_head(c, seed):
    w = _workload(c)
    T = c["context"]
    cache, energies = _production(c, w, T + 64)
    production_prefill(_Prompt(_prompt_kv(c, w, seed, energies, T)), _ids(w, T), cache, chunk_encode=T)
    q8, ka = cache.quantizers[0][0], cache.kernel_args[0][0]
    q = q8.rotate_q_for_packed_kernel(wl.draw_q(_data(w, seed), 0, DEV, T))
    slices = [t[0][:, :1, :T] for t in (cache.k_packed, cache.k_norms, cache.v_packed, cache.v_norms)]
    kp, kn, vp, vn = slices
    nibble = c["nibble"]

    def run():
        return fused_blockgtq_decode_attention(
            q, kp, kn, ka["codebook_flat"], ka["lut_offset"], ka["norm_group"], ka["segments_b"], vp, vn, q8.v_lut,
            v_bits=w.v_bits, v_rotation=q8._v_rot, k_nibble=nibble, v_nibble=nibble)

    return {"run": run, "owner": cache}


_PREPARE = {"decode": _prepare_decode, "pack": _prepare_pack, "chunks": _prepare_chunks, "prompt": _prepare_prompt,
            "head": _prepare_head}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return state["run"]()


# --------------------------------------------------------------------------------------- accounting
def _record_bytes(c):
    """Bytes of one token of one KV head: K codes, group norms, V codes, V norm."""
    if c.get("nibble"):
        return D // 2 + 2 * K_GROUPS + D // 2 + 2
    return D * c["k_bits"] / 8 + 2 * K_GROUPS + D * c["v_bits"] / 8 + 2


def work(case):
    c, rec = case, _record_bytes(case)
    B, T, L = c["batch"], c["context"], c.get("layers", 1)
    n_kv = c.get("n_kv", 1)
    n_q = c.get("n_q", n_kv * c.get("gqa", 1))
    if c["kind"] in ("decode", "head"):
        tokens = B * T * (0.53 if c.get("ragged") else 1.0)          # (ragged rows: even from T / 16 to T)
        fp16_rows = B * min(T, c.get("sink", 0) + c.get("window", 0))
        per_layer = n_kv * ((tokens - fp16_rows) * rec + fp16_rows * 4 * D)
        io = B * (n_q * 4 * D + (n_kv * (4 * D + rec) if c["kind"] == "decode" else 0))
        rotate = B * 2 * D * D * (n_q + 2 * n_kv) if c["kind"] == "decode" else 0
        return {"bytes": L * (per_layer + io), "flops": L * (4 * D * n_q * tokens + 2 * D * D * B * n_q + rotate)}
    if c["kind"] in ("pack", "chunks"):
        rows = B * n_kv * T * L
        return {"bytes": rows * (4 * D + rec), "flops": rows * (2 * D * D + 2 * D * 32 + 12 * D)}
    S = c["queries"]
    pairs = S * (T - S) + S * (S + 1) / 2
    return {"bytes": B * (n_q * S * 4 * D + n_kv * T * rec), "flops": B * n_q * (4 * D * pairs + 4 * D * D * S)}


def tolerance(case):
    """Packed bytes and stored norms follow from a fixed order of evaluation: the same, bit for bit.
    Attention outputs are fp16 results of fp16 operands (11-bit significands: probabilities,
    dequantised records and the output are each rounded once, 3e-4 apiece) summed in fp32."""
    if case["kind"] in ("pack", "chunks"):
        return "exact"
    return {"rel": 2e-3, "max": 2e-2}
