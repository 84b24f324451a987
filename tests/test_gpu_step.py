"""GPU: the one-call decode step and append (native layer handles) against the general path.

Both launch the same kernels on the same values (bf16 inputs are rounded to fp16 where they are
read, as ``.to(torch.float16)`` rounds them), so caches and outputs must agree bit for bit."""
import pytest
import torch

from blockgtq_amd import workloads as wl
from blockgtq_amd.production_cache import BlockGTQProductionCache
from blockgtq_amd.quantizer import build_batched_encode_args

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(w, energies, T, dtype):
    k, v = wl.draw_kv(w, energies[0], 1, 321, DEV, pos0=T)
    q = wl.draw_q(w, 0, DEV, T)
    # as a projection leaves them: heads behind tokens in memory
    return [t.to(dtype).transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("batch,context,ragged,window", [(1, 1, False, 0), (3, 130, True, 0), (2, 200, True, 64), (40, 70, False, 0)])
def test_manager_step_equals_general_path(dtype, batch, context, ragged, window):
    lens = [max(context - 3 * b, window + 5, 1) for b in range(batch)] if ragged else None
    w = wl.Workload("t", 1, 8, 2, batch, context, 1e6, seq_lens=lens, n_sink=4 if window else 0, window=window, seed=31)
    mgrs = []
    for _ in range(2):
        mgr, energies = wl.build_manager(w, DEV)
        wl.fill_cache(mgr, w, energies, DEV)
        mgrs.append(mgr)
    q, k, v = _inputs(w, energies, context, dtype)
    fast = mgrs[0].append_and_attend(0, q, k, v)
    general = mgrs[1]
    general._native = lambda li: general._ensure_storage()          # (no handle: every call goes the general way)
    slow = general.append_and_attend(0, q, k, v)
    assert fast.shape == (batch, 8, 1, 128) and fast.abs().max() > 0
    assert torch.equal(fast, slow)
    for name in ("_k_packed", "_k_norms", "_v_packed", "_v_norms") + (("_buf_k", "_buf_v") if window else ()):
        assert torch.equal(getattr(mgrs[0], name)[0], getattr(general, name)[0]), name


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("nibble,device_lengths,tokens", [(True, False, 1), (False, True, 1), (False, False, 65), (True, False, 200)])
def test_production_cache_step_and_append_equal_general_path(dtype, nibble, device_lengths, tokens):
    w = wl.Workload("t", 1, 12, 4, 2, 300, 1e6, seed=32)
    qs, e = wl.calibrate_layer(w, 0, DEV)
    k0, v0 = wl.draw_kv(w, e, tokens, 5, DEV)
    k0, v0 = k0.to(dtype), v0.to(dtype)
    caches = []
    for fast in (True, False):
        c = BlockGTQProductionCache([qs], [build_batched_encode_args(qs, device=DEV)], [[q.build_kernel_args() for q in qs]],
                                    1, 4, 12, 128, 320, k_nibble=nibble, v_nibble=nibble, device=DEV, batch_size=2)
        if not fast:
            c._native = lambda li: None
        c._encode_batched(0, k0, v0, 0)
        c.seq_len = tokens
        if device_lengths:
            c.use_device_lengths()
        caches.append(c)
    q, k, v = _inputs(w, [e], tokens, dtype)
    outs = [c.encode_and_attend(0, q, k, v) for c in caches]
    assert torch.equal(*outs) and outs[0].abs().max() > 0
    for name in ("k_packed", "k_norms", "v_packed", "v_norms"):
        assert torch.equal(getattr(caches[0], name), getattr(caches[1], name)), name


# (rows, query heads, KV heads, window): the buffered tokens' partial rides with the preparation up to 64 rows, from two
# query heads per KV head on and up to 3072 buffered tokens (4 of them sinks); beside each limit the launch of its own
@pytest.mark.parametrize("batch,n_q,n_kv,window", [(64, 8, 2, 60), (65, 8, 2, 60), (3, 2, 2, 60), (3, 10, 2, 61), (1, 4, 1, 3068), (1, 4, 1, 3069)])
def test_buffered_partial_with_and_without_the_preparation(batch, n_q, n_kv, window):
    context = window + 70
    lens = [max(context - 29 * b, window + 4) if b % 5 else context for b in range(batch)]      # (some rows fill just the buffer)
    w = wl.Workload("t", 1, n_q, n_kv, batch, context, 1e6, seq_lens=lens, n_sink=4, window=window, seed=34)
    mgrs = []
    for _ in range(2):
        mgr, energies = wl.build_manager(w, DEV)
        wl.fill_cache(mgr, w, energies, DEV)
        mgrs.append(mgr)
    q, k, v = _inputs(w, energies, context, torch.bfloat16)
    mgrs[1]._native = lambda li: mgrs[1]._ensure_storage()
    for _ in range(2):                                                                  # (the ring moves on)
        fast, slow = [m.append_and_attend(0, q, k, v) for m in mgrs]
        assert fast.abs().max() > 0 and torch.equal(fast, slow)
        for m in mgrs:
            m.increment_seq_len()
    for name in ("_k_packed", "_k_norms", "_v_packed", "_v_norms", "_buf_k", "_buf_v"):
        assert torch.equal(getattr(mgrs[0], name)[0], getattr(mgrs[1], name)[0]), name


def _pair(nibble=True, baked=False):
    """Two caches with the same 90 records, the second without native handles."""
    w = wl.Workload("t", 1, 12, 4, 2, 90, 1e6, seed=35)
    qs, e = wl.calibrate_layer(w, 0, DEV)
    for q8 in qs:
        q8._q_perm_baked = baked
    k0, v0 = wl.draw_kv(w, e, 90, 5, DEV)
    caches = []
    for fast in (True, False):
        c = BlockGTQProductionCache([qs], [build_batched_encode_args(qs, device=DEV)], [[q.build_kernel_args() for q in qs]],
                                    1, 4, 12, 128, 120, k_nibble=nibble, v_nibble=nibble, device=DEV, batch_size=2)
        if not fast:
            c._native = lambda li: None
        c._encode_batched(0, k0, v0, 0)
        c.seq_len = 90
        caches.append(c)
    return w, e, caches


def _step(caches, w, e, T, dtype=torch.float16):
    q, k, v = _inputs(w, [e], T, dtype)
    fast, slow = [c.encode_and_attend(0, q, k, v) for c in caches]
    for c in caches:
        c.increment_seq_len()
    assert fast.abs().max() > 0 and torch.equal(fast, slow)
    for name in ("k_packed", "k_norms", "v_packed", "v_norms"):
        assert torch.equal(getattr(caches[0], name), getattr(caches[1], name)), name
    return fast


def test_production_cache_handle_follows_its_attributes():
    """Scale, layout, row widths and storage may be set between steps; the next step goes by them."""
    w, e, caches = _pair()
    a = _step(caches, w, e, 90)
    for c in caches:
        c.scale *= 3
    assert not torch.equal(a, _step(caches, w, e, 91))
    for c in caches:                                                    # other storage behind the same tensor object
        c.v_norms.data = c.v_norms * 2
    _step(caches, w, e, 92)
    for c in caches:                                                    # other tensors
        c.k_packed, c.k_norms = c.k_packed.clone(), c.k_norms * 0.5
    _step(caches, w, e, 93)
    bit_packed = _pair(nibble=False)[2]
    for c, b in zip(caches, bit_packed):                                # another layout, with the storage that goes with it
        for name in ("_k_layout", "_v_layout", "k_bytes_per_tok", "vpb", "max_ng", "k_packed", "k_norms", "v_packed", "v_norms"):
            setattr(c, name, getattr(b, name))
        c.seq_len = 90
    _step(caches, w, e, 90)


@pytest.mark.parametrize("window", [0, 64])
def test_manager_handle_follows_its_attributes(window):
    w = wl.Workload("t", 1, 8, 2, 2, 150, 1e6, n_sink=4 if window else 0, window=window, seed=36)
    mgrs = []
    for _ in range(2):
        mgr, energies = wl.build_manager(w, DEV)
        wl.fill_cache(mgr, w, energies, DEV)
        mgrs.append(mgr)
    mgrs[1]._native = lambda li: None

    def step():
        q, k, v = _inputs(w, energies, 150, torch.float16)
        outs = [m.append_and_attend(0, q, k, v) for m in mgrs]
        assert outs[0].abs().max() > 0 and torch.equal(*outs)
        for name in ("_k_packed", "_k_norms", "_v_packed", "_v_norms") + (("_buf_k", "_buf_v") if window else ()):
            assert torch.equal(getattr(mgrs[0], name)[0], getattr(mgrs[1], name)[0]), name
        return outs[0]

    a = step()
    for m in mgrs:
        m.scale *= 3
    assert not torch.equal(a, step())
    for m in mgrs:
        m._v_norms.data = m._v_norms * 2
    step()
    for m in mgrs:
        m._k_norms, m._k_packed = m._k_norms * 0.5, [t.clone() for t in m._k_packed]
    step()
    if window:
        for m in mgrs:
            m._buf_k, m._buf_v = m._buf_k.clone(), m._buf_v * 2
        step()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_step_with_folded_rotation_and_strided_queries(dtype):
    """With the rotation in the projection the fp16 queries go to the attention as they lie: heads behind a gap, in rows of a
    wider projection.  (bf16 queries are converted on the general way.)"""
    w, e, caches = _pair(baked=True)
    q, k, v = _inputs(w, [e], 90, dtype)
    wide = torch.randn(2, 1, 12, 3, 128, device=DEV).to(dtype)
    wide[:, :, :, 1] = q.transpose(1, 2)
    strided = wide[:, :, :, 1].transpose(1, 2)
    assert strided.stride() != q.stride() and torch.equal(strided, q)
    fast, slow, plain = caches[0].encode_and_attend(0, strided, k, v), caches[1].encode_and_attend(0, strided, k, v), caches[1].encode_and_attend(0, q, k, v)
    assert fast.abs().max() > 0 and torch.equal(fast, slow) and torch.equal(fast, plain)


@pytest.mark.parametrize("owner", ["manager", "manager_window", "production_device_lengths"])
def test_replayed_step_equals_eager_steps(owner):
    """A captured step whose inputs are kept, replayed with eager work and synchronisations in between, against the same
    number of eager steps of a twin.  (Nothing increments the length: every step writes its token at one place.)"""
    T, dtype = 150, torch.bfloat16
    w = wl.Workload("t", 1, 8, 2, 3, T, 1e6, seq_lens=[T, T - 7, T - 70], n_sink=4 if owner == "manager_window" else 0,
                    window=64 if owner == "manager_window" else 0, seed=37)
    twins = []
    for _ in range(2):
        if owner == "production_device_lengths":
            qs, e = wl.calibrate_layer(w, 0, DEV)
            c = BlockGTQProductionCache([qs], [build_batched_encode_args(qs, device=DEV)], [[q.build_kernel_args() for q in qs]],
                                        1, 2, 8, 128, T + 8, device=DEV, batch_size=3)
            c._encode_batched(0, *wl.draw_kv(w, e, T, 5, DEV), 0)
            c.set_seq_lens(w.seq_lens)
            c.use_device_lengths()
            twins.append((c, c.encode_and_attend, ("k_packed", "k_norms", "v_packed", "v_norms")))
            energies = [e]
        else:
            m, energies = wl.build_manager(w, DEV)
            wl.fill_cache(m, w, energies, DEV)
            twins.append((m, m.append_and_attend, ("_k_packed", "_k_norms", "_v_packed", "_v_norms") + (("_buf_k", "_buf_v") if w.window else ())))
    q, k, v = _inputs(w, energies, T, dtype)
    (a, step, names), (b, eager, _) = twins
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(0, q, k, v)
    torch.cuda.current_stream().wait_stream(side)
    eager(0, q, k, v)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step(0, q, k, v)
    for i in range(3):
        for t in (q, k, v):                             # the same tensors with other values
            t.copy_(torch.randn(t.shape, device=DEV))
        graph.replay()
        want = eager(0, q, k, v)
        torch.cuda.synchronize()
        assert torch.isfinite(want).all() and want.abs().max() > 0 and torch.equal(out, want), i
        for name in names:
            assert torch.equal(getattr(a, name)[0], getattr(b, name)[0]), (i, name)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("offset", [0, 1])                      # new tokens on 16-byte boundaries, and off them (swapped by a launch of their own)
def test_buffered_step_slots(dtype, offset):
    """Slots at both ends of the buffer, behind the visible tokens and outside it (nothing enters, a row of zeros is packed)."""
    n_q, n_kv, W, B, context = 8, 2, 20, 7, 60
    w = wl.Workload("t", 1, n_q, n_kv, B, context, 1e6, seq_lens=[context] * B, n_sink=4, window=W - 4, seed=38)
    mgrs = []
    for _ in range(2):
        mgr, energies = wl.build_manager(w, DEV)
        wl.fill_cache(mgr, w, energies, DEV)
        mgrs.append(mgr)
    q, k, v = _inputs(w, energies, context, dtype)
    if offset:
        k, v = (torch.cat([torch.zeros_like(t[..., :1]), t], -1).contiguous()[..., 1:] for t in (k, v))
    i32 = dict(dtype=torch.int32, device=DEV)
    idx = (torch.arange(B, device=DEV), torch.tensor([0, W - 1, 5, -1, W, 11, 3], **i32), torch.arange(30, 30 + B, **i32),
           torch.tensor([41, 40, 1, 7, 41, 30, 0], **i32), torch.tensor([W, W, 6, W, W, 9, 1], **i32))
    mgrs[1]._native = lambda li: mgrs[1]._ensure_storage()
    for m in mgrs:
        m._buffered_step_indices = lambda: idx
    fast, slow = [m.append_and_attend(0, q, k, v) for m in mgrs]
    assert torch.isfinite(slow).all() and slow.abs().max() > 0 and torch.equal(fast, slow)
    for name in ("_k_packed", "_k_norms", "_v_packed", "_v_norms", "_buf_k", "_buf_v"):
        assert torch.equal(getattr(mgrs[0], name)[0], getattr(mgrs[1], name)[0]), name


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("n_q", [8, 14])                        # heads of a group all served at once, and a last one of three
def test_buffered_step_with_a_new_token_that_nobody_sees(bad, n_q):
    """A new token that is not finite, in a slot behind the visible ones: no output depends on it."""
    n_kv, W, B, context = 2, 20, 6, 60
    w = wl.Workload("t", 1, n_q, n_kv, B, context, 1e6, seq_lens=[context] * B, n_sink=4, window=W - 4, seed=39)
    mgrs = []
    for _ in range(2):
        mgr, energies = wl.build_manager(w, DEV)
        wl.fill_cache(mgr, w, energies, DEV)
        mgrs.append(mgr)
    q, k, v = _inputs(w, energies, context, torch.float16)
    k[:, :, :, 5], v[:, :, :, 7] = bad, bad
    i32 = dict(dtype=torch.int32, device=DEV)
    slots, seen = [11, 3, W - 1, 9, 13, W], [9, 1, 17, 9, 2, W]
    idx = (torch.arange(B, device=DEV), torch.tensor(slots, **i32), torch.arange(30, 30 + B, **i32),
           torch.tensor([41, 40, 1, 7, 0, 30], **i32), torch.tensor(seen, **i32))
    assert all(s >= n for s, n in zip(slots, seen))
    mgrs[1]._native = lambda li: mgrs[1]._ensure_storage()
    for m in mgrs:
        m._buffered_step_indices = lambda: idx
    fast, slow = [m.append_and_attend(0, q, k, v) for m in mgrs]
    assert torch.isfinite(slow).all() and slow.abs().max() > 0 and torch.equal(fast, slow)


# more than one round of work-groups and partitions of eight tiles: rows go out by falling length.  Ties, equal rows, rows of a
# few tokens, all 64 rows a step ranks and one more
@pytest.mark.parametrize("batch,n_kv,splits,window,kind", [(33, 8, 1, 0, "mixed"), (64, 1, 5, 0, "mixed"), (64, 8, 2, 0, "equal"), (9, 2, 16, 0, "mixed"),
                                                           (33, 4, 2, 64, "mixed"), (65, 4, 1, 0, "mixed")])
def test_rows_by_falling_length_change_nothing(batch, n_kv, splits, window, kind):
    context = max(700, 500 * splits)
    gen = torch.Generator().manual_seed(batch)
    lens = [context] * batch if kind == "equal" else torch.randint(window + 5 if window else 0, context + 1, (batch,), generator=gen).tolist()
    lens[0] = context
    lens[batch // 2] = lens[batch // 3]
    w = wl.Workload("t", 1, 2 * n_kv, n_kv, batch, context, 1e6, seq_lens=lens, n_sink=4 if window else 0, window=window, seed=37)
    mgrs = []
    for _ in range(2):
        mgr, energies = wl.build_manager(w, DEV)
        wl.fill_cache(mgr, w, energies, DEV)
        mgr.n_splits = splits
        mgrs.append(mgr)
    q, k, v = _inputs(w, energies, context, torch.float16)
    general = mgrs[1]
    general._native = lambda li: general._ensure_storage()          # (rows as they come)
    for _ in range(2):
        assert torch.equal(mgrs[0].append_and_attend(0, q, k, v), general.append_and_attend(0, q, k, v))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_token_rows_at_strides_beyond_32_bits(dtype):
    """New rows whose batch stride leaves 32 bits take the general preparation, others the one of single tokens (its last stride
    among them): the same step, also with heads that share a row of K and lie apart in V.  Cut to 32 bits, a stride of 2 ** 32
    would give the second row the tokens of the first."""
    w, e, caches = _pair()
    one = lambda t: t[:1].expand(2, -1, -1, -1)
    q, k, v = [t.contiguous() for t in _inputs(w, [e], 90, dtype)]
    outs = [caches[0].encode_and_attend(0, one(q), k[:1, :1].expand(2, 4, 1, 128), one(v)),
            caches[1].encode_and_attend(0, one(q).contiguous(), k[:1, :1].expand(2, 4, 1, 128).contiguous(), one(v).contiguous())]
    assert outs[0].abs().max() > 0 and torch.equal(*outs)
    w2 = wl.Workload("t", 1, 8, 2, 2, 90, 1e6, seed=38)
    memory = torch.empty(2 ** 32 + 1024, dtype=dtype, device=DEV)           # (8.6 GB, touched at both ends alone)
    got = []
    for stride in (None, 2 ** 32 - 128, 2 ** 32):
        mgr, energies = wl.build_manager(w2, DEV)
        wl.fill_cache(mgr, w2, energies, DEV)
        q, k, v = [t.contiguous() for t in _inputs(w2, energies, 90, dtype)]
        assert not torch.equal(k[0], k[1]) and not torch.equal(v[0], v[1])
        if stride:
            far = [memory.as_strided((2, 2, 1, 128), (stride, 128, 128, 1), at) for at in (0, 512)]
            k, v = [f.copy_(t) for f, t in zip(far, (k, v))]
        got.append((mgr.append_and_attend(0, q, k, v), mgr._k_packed[0], mgr._k_norms[0], mgr._v_packed[0], mgr._v_norms[0]))
    del memory, far, k, v
    torch.cuda.empty_cache()
    assert got[0][0].abs().max() > 0
    for other in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got[0], other))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("S", [1, 2, 5, 33])                 # (66 new rows leave the one launch)
def test_steps_of_several_new_tokens(S, dtype):
    """The preparation of any number of new tokens leaves the records that appends of one token each leave."""
    w, e, caches = _pair()
    for c in caches:                                         # room for 33
        for name in ("k_packed", "k_norms", "v_packed", "v_norms"):
            t = getattr(c, name)
            setattr(c, name, torch.cat([t, torch.zeros_like(t)], 3))
        c.max_T *= 2
    q, _, _ = _inputs(w, [e], 90, dtype)
    k, v = [t.to(dtype) for t in wl.draw_kv(w, e, S, 322, DEV, pos0=90)]
    fast, slow = [c.encode_and_attend(0, q, k, v) for c in caches]
    assert fast.abs().max() > 0 and torch.equal(fast, slow)
    for s in range(S):
        caches[1]._encode_batched(0, k[:, :, s:s + 1], v[:, :, s:s + 1], 90 + s)
    for name in ("k_packed", "k_norms", "v_packed", "v_norms"):
        assert torch.equal(getattr(caches[0], name), getattr(caches[1], name)), name


@pytest.mark.parametrize("bits", [3, 4])
@pytest.mark.parametrize("n_q", [8, 16, 24])                 # 4 and 8 query heads a KV head, and two launches
def test_nibble_records_with_and_without_a_known_code_width(bits, n_q):
    """Plans that say how wide V's codes are and copies that do not: the same records and outputs, native, general and the attention alone."""
    from blockgtq_amd import ops, plan as P
    w = wl.Workload("t", 1, n_q, 2, 2, 200, 1e6, k_bits=float(bits), v_bits=bits, seed=39)
    qs, e = wl.calibrate_layer(w, 0, DEV)
    k0, v0 = wl.draw_kv(w, e, 200, 5, DEV)
    q, k, v = _inputs(w, [e], 200, torch.float16)
    got = []
    for known in (True, False):
        c = BlockGTQProductionCache([qs], [build_batched_encode_args(qs, device=DEV)], [[q8.build_kernel_args() for q8 in qs]],
                                    1, 2, n_q, 128, 210, v_bits=bits, device=DEV, batch_size=2)
        plans = c.batched_args[0]['plans']
        assert plans.v_code_bits == bits
        if not known:
            plans = c.batched_args[0]['plans'] = plans.clone()
        assert P.attended_v_layout(plans, c._v_layout, c.vpb) == (P.V_NIBBLE4 if known and bits == 4 else P.V_NIBBLE)
        c._encode_batched(0, k0, v0, 0)
        c.seq_len = 200
        outs = [c.encode_and_attend(0, q, k, v), c._encode_and_attend_general(0, q, k, v)]
        outs.append(ops.decode_attention(plans, ops.rotate_q(plans, q[:, :, 0].contiguous(), 2), c.k_packed[0], c.k_norms[0],
                                         c.v_packed[0], c.v_norms[0], 201, k_layout=c._k_layout, v_layout=c._v_layout).unsqueeze(2))
        assert ops.last_decode_path() == ops.MFMA_PATH
        assert outs[0].abs().max() > 0 and all(torch.equal(outs[0], o) for o in outs)
        got.append([outs[0], c.k_packed, c.k_norms, c.v_packed, c.v_norms])
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("bits", [1, 2, 3, 4])
def test_nibble_records_behind_plans_written_over(bits):
    """Plans of 4-bit codes that other ones were copied over since: records and outputs of those, by every kernel."""
    from blockgtq_amd import _capi, ops, plan as P
    made = []
    for b in (4, bits):
        w = wl.Workload("t", 1, 8, 2, 2, 200, 1e6, k_bits=3.0, v_bits=b, seed=40)
        made.append((w,) + wl.calibrate_layer(w, 0, DEV))
    (_, q4, _), (w, qs, e) = made
    k0, v0 = wl.draw_kv(w, e, 200, 5, DEV)
    q, k, v = _inputs(w, [e], 200, torch.float16)
    want = build_batched_encode_args(qs, device=DEV)['plans']
    got = []
    for over in (False, True):
        c = BlockGTQProductionCache([qs], [build_batched_encode_args(q4 if over else qs, device=DEV)], [[q8.build_kernel_args() for q8 in qs]],
                                    1, 2, 8, 128, 210, v_bits=bits, device=DEV, batch_size=2)
        plans = c.batched_args[0]['plans']
        if over:
            assert P.attended_v_layout(plans, c._v_layout, c.vpb) == P.V_NIBBLE4
            plans.copy_(want)
        assert torch.equal(plans, want)
        c._encode_batched(0, k0, v0, 0)
        c.seq_len = 200
        outs = [c.encode_and_attend(0, q, k, v)]
        for path in (2, 1):                                  # matrix cores, any layout
            assert _capi.lib().bgtq_set_decode_path(path) == 0
            try:
                outs.append(ops.decode_attention(plans, ops.rotate_q(plans, q[:, :, 0].contiguous(), 2), c.k_packed[0], c.k_norms[0],
                                                 c.v_packed[0], c.v_norms[0], 201, k_layout=c._k_layout, v_layout=c._v_layout))
            finally:
                _capi.lib().bgtq_set_decode_path(0)
        got.append(outs + [c.k_packed, c.k_norms, c.v_packed, c.v_norms])
    assert got[0][0].abs().max() > 0 and all(torch.equal(a, b) for a, b in zip(*got))
