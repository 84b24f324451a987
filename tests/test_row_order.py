"""When a decode step ranks its rows and where the order lies: the library's rule, compiled for the CPU."""
import ctypes
import os
import re
import subprocess

import pytest
import torch

from blockgtq_amd import _capi, ops, workloads as wl
from blockgtq_amd.build import CSRC

DEV = "cuda:0"

_SHIM = """
#include <string.h>
#include "%s"
// A step of 40 rows x 2 heads x 3 queries whose buffers lie 16 MiB apart, with one of them moved to `out` + delta
static const uintptr_t OUT = 1ull << 30;
static bgtq_step step(const char* moved, int64_t delta) {
    bgtq_step s;
    memset(&s, 0, sizeof(s));
    uintptr_t at = OUT;
    s.B = 40; s.n_kv = 2; s.gqa = 3; s.S = 1; s.n_splits = 5; s.T = 50; s.max_T = 64;
    s.q_sb = 6 * 128; s.q_sh = 128;
    s.k_sb = s.v_sb = 2 * 128; s.k_sh = s.v_sh = 128; s.k_ss = s.v_ss = 128;
    s.k_row_width = 52; s.v_row_width = 48; s.norm_width = 4;
    s.kp_st = 52; s.kp_sh = 64 * 52; s.kp_sb = 2 * 64 * 52;
    s.vp_st = 48; s.vp_sh = 64 * 48; s.vp_sb = 2 * 64 * 48;
    s.kn_st = 4; s.kn_sh = 64 * 4; s.kn_sb = 2 * 64 * 4;
    s.vn_st = 1; s.vn_sh = 64; s.vn_sb = 2 * 64;
    s.win_W = 12; s.w_st = 128; s.w_sh = 12 * 128; s.w_sb = 2 * 12 * 128;
#define PLACE(f) s.f = (decltype(s.f))(at += 1 << 24); if (!strcmp(moved, #f)) s.f = (decltype(s.f))(OUT + delta);
    PLACE(plans) PLACE(q) PLACE(k) PLACE(v) PLACE(q_rot) PLACE(k_packed) PLACE(k_norms) PLACE(v_packed) PLACE(v_norms) PLACE(t_pos)
    PLACE(seq_lens) PLACE(partial_out) PLACE(partial_lse) PLACE(win_k) PLACE(win_v) PLACE(win_slot) PLACE(win_lens) PLACE(win_old)
    PLACE(win_out) PLACE(win_lse)
    s.out = (void*)OUT;
    return s;
}
extern "C" int fits(const char* moved, int64_t delta) { return bgtq_order_fits(step(moved, delta)); }
extern "C" int fits_out_off(int64_t by) { bgtq_step s = step("", 0); s.out = (void*)(OUT + by); return bgtq_order_fits(s); }
extern "C" int fits_backwards(const char* stride) {
    bgtq_step s = step("", 0);
#define TURN(f) if (!strcmp(stride, #f)) s.f = -s.f;
    TURN(q_sb) TURN(q_sh) TURN(k_sb) TURN(k_sh) TURN(k_ss) TURN(v_sb) TURN(v_sh) TURN(v_ss) TURN(kp_sb) TURN(kp_sh) TURN(kp_st)
    TURN(kn_sb) TURN(kn_sh) TURN(kn_st) TURN(vp_sb) TURN(vp_sh) TURN(vp_st) TURN(vn_sb) TURN(vn_sh) TURN(vn_st) TURN(w_sb) TURN(w_sh) TURN(w_st)
    return bgtq_order_fits(s);
}
extern "C" int fits_without(void) {
    bgtq_step s = step("", 0);
    s.q_rot = nullptr; s.t_pos = nullptr;
    s.win_k = s.win_v = s.win_old = nullptr; s.win_slot = s.win_lens = nullptr; s.win_out = s.win_lse = nullptr;
    return bgtq_order_fits(s);
}
extern "C" int orders(int B, int n_kv, int S, int T, int splits, int ragged) { return bgtq_orders_rows(B, n_kv, S, T, splits, ragged); }
extern "C" int rank(const int* lens, int n, int i) { return bgtq_row_rank(lens, n, i); }
extern "C" int64_t plan_bytes(void) { return sizeof(bgtq_head_plan); }
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    where = tmp_path_factory.mktemp("row_order")
    src, lib = where / "rule.cpp", where / "rule.so"
    src.write_text(_SHIM % os.path.join(CSRC, "bgtq_row_order.h"))
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__host__=", "-D__device__=", "-shared", "-fPIC", str(src), "-o", str(lib)], check=True)
    rule = ctypes.CDLL(str(lib))
    rule.fits.argtypes = [ctypes.c_char_p, ctypes.c_int64]
    rule.fits_out_off.argtypes = [ctypes.c_int64]
    rule.fits_backwards.argtypes = [ctypes.c_char_p]
    rule.plan_bytes.restype = ctypes.c_int64
    return rule


ORDER = 4 * 40
# bytes of each buffer of the step above
EXTENT = {"q": 40 * 6 * 128 * 2, "k": 40 * 2 * 128 * 2, "v": 40 * 2 * 128 * 2, "q_rot": 40 * 6 * 128 * 2, "plans": None,
          "k_packed": 40 * 2 * 64 * 52, "k_norms": 40 * 2 * 64 * 4 * 2, "v_packed": 40 * 2 * 64 * 48, "v_norms": 40 * 2 * 64 * 2,
          "t_pos": ORDER, "seq_lens": ORDER, "partial_out": 40 * 6 * 5 * 128 * 4, "partial_lse": 40 * 6 * 5 * 4,
          "win_k": 40 * 2 * 12 * 128 * 2, "win_v": 40 * 2 * 12 * 128 * 2, "win_slot": ORDER, "win_lens": ORDER,
          "win_old": 2 * 40 * 2 * 128 * 2, "win_out": 40 * 6 * 128 * 4, "win_lse": 40 * 6 * 4}


@pytest.mark.parametrize("field", list(EXTENT))
def test_the_order_shares_memory_with_no_buffer_of_the_step(rule, field):
    """The order is written while the step's inputs and scratch are in use: what shares memory with `out` keeps rows as they come."""
    size = EXTENT[field] or 2 * rule.plan_bytes()
    name = field.encode()
    assert rule.fits(b"", 0)
    for overlapping in (0, 4, ORDER - 4, -4, 4 - size):
        assert not rule.fits(name, overlapping)
    assert rule.fits(name, ORDER) and rule.fits(name, -size)


def test_strides_that_run_backwards_and_unaligned_outputs_keep_rows_as_they_come(rule):
    for stride in ("q_sb", "q_sh", "k_sb", "k_sh", "k_ss", "v_sb", "v_sh", "v_ss", "kp_sb", "kp_sh", "kp_st", "kn_sb", "kn_sh", "kn_st",
                   "vp_sb", "vp_sh", "vp_st", "vn_sb", "vn_sh", "vn_st", "w_sb", "w_sh", "w_st"):
        assert not rule.fits_backwards(stride.encode()), stride
    assert rule.fits_backwards(b"") and rule.fits_without()
    assert [rule.fits_out_off(by) for by in (0, 1, 2, 4)] == [1, 0, 0, 1]


def test_only_batches_that_one_work_group_ranks_are_ranked(rule):
    """One thread a row: as many rows as the launch has room for, whatever the number of new tokens (0 among them)."""
    T = 8192
    assert [rule.orders(B, 8, 1, T, 8, 1) for B in (1, 4, 5, 64, 65, 130, 10**6)] == [0, 0, 1, 1, 0, 0, 0]
    assert [rule.orders(B, 8, 0, T, 8, 1) for B in (1, 5, 64, 65, 130, 10**6)] == [0] * 6
    assert [rule.orders(16, 8, S, T, 8, 1) for S in (-1, 0, 1, 4, 5)] == [0, 0, 1, 1, 0]
    assert not rule.orders(16, 8, 1, T, 8, 0) and not rule.orders(16, 2, 1, T, 8, 1) and rule.orders(43, 2, 1, T, 3, 1)


def test_short_partitions_go_as_they_come(rule):
    """Eight tiles of 64 tokens in the longest partition at least."""
    assert [rule.orders(40, 8, 1, T, 1, 1) for T in (0, 1, 448, 449, 512, 2**31 - 1)] == [0, 0, 0, 1, 1, 1]
    assert [rule.orders(40, 8, 1, T, 3, 1) for T in (1344, 1345)] == [0, 1]
    assert [rule.orders(40, 8, 1, 8192, splits, 1) for splits in (0, 16, 19, 32)] == [0, 1, 0, 0]


@pytest.mark.parametrize("lens", [[5], [0, 0], [3, 1, 2], [7] * 64, [0, 9, 0, 9, 4, -1, 4, 2**31 - 1], [i * 37 % 11 for i in range(64)]])
def test_rank_is_the_stable_order_by_falling_length(rule, lens):
    ranks = [rule.rank((ctypes.c_int * len(lens))(*lens), len(lens), i) for i in range(len(lens))]
    assert sorted(range(len(lens)), key=lambda i: ranks[i]) == sorted(range(len(lens)), key=lambda i: -lens[i])
    assert sorted(ranks) == list(range(len(lens)))


# --------------------------------------------------------------------------------------- the entry itself, on the GPU
_C = {"int32_t": ctypes.c_int32, "int64_t": ctypes.c_int64, "float": ctypes.c_float}


def _step_type():
    """bgtq_step as the header declares it."""
    body, = re.findall(r"typedef struct bgtq_step \{(.*?)\} bgtq_step;", open(os.path.join(CSRC, "../../include/bgtq.h")).read(), re.S)
    fields = []
    for kind, names in re.findall(r"(?:const )?(\w+)\s*([^;]*);", body):
        for name in names.split(","):
            fields.append((name.strip(" *"), ctypes.c_void_p if "*" in name else _C[kind]))
    return type("Step", (ctypes.Structure,), {"_fields_": fields})


def _filled(batch, n_kv, gqa, context, window=0, seed=41, dtype=torch.float16):
    gen = torch.Generator().manual_seed(seed)
    lens = torch.randint(window + 5 if window else 0, context + 1, (batch,), generator=gen).tolist()
    lens[0] = context
    w = wl.Workload("t", 1, gqa * n_kv, n_kv, batch, context, 1e6, seq_lens=lens, n_sink=4 if window else 0, window=window, seed=seed)
    mgr, energies = wl.build_manager(w, DEV)
    wl.fill_cache(mgr, w, energies, DEV)
    k, v = wl.draw_kv(w, energies[0], 1, 321, DEV, pos0=context)
    return mgr, *[t.to(dtype).contiguous() for t in (wl.draw_q(w, 0, DEV, context), k, v)]


def _step(mgr, q, k, v, splits, place=lambda out, scratch: out, S=1, empty=()):
    """bgtq_decode_step on layer 0; `place` says where the output lies, given one of its own and the scratch buffers; the rows of
    `empty` see no record."""
    B, n_q, n_kv = q.shape[0], q.shape[1], k.shape[1]
    kp, kn, vp, vn = mgr._k_packed[0], mgr._k_norms[0], mgr._v_packed[0], mgr._v_norms[0]
    f32, f16 = dict(dtype=torch.float32, device=DEV), dict(dtype=torch.float16, device=DEV)
    scratch = {"q_rot": torch.zeros(B, n_q, 128, **f16), "partial_out": torch.zeros(B, n_q, splits, 128, **f32),
               "partial_lse": torch.zeros(B, n_q, splits, **f32), "q": q, "k": k, "v": v}
    s = _step_type()()
    s.plans = mgr._batched_args[0]["plans"].data_ptr()
    s.B, s.n_kv, s.gqa, s.S, s.n_splits, s.scale = B, n_kv, n_q // n_kv, S, splits, mgr.scale
    s.x_dtype = int(q.dtype == torch.bfloat16)
    s.q_sb, s.q_sh = q.stride(0), q.stride(1)
    s.k_sb, s.k_sh, s.k_ss = s.v_sb, s.v_sh, s.v_ss = k.stride()[:3]
    s.k_packed, s.kp_sb, s.kp_sh, s.kp_st = kp.data_ptr(), *kp.stride()[:3]
    s.k_norms, s.kn_sb, s.kn_sh, s.kn_st = kn.data_ptr(), *kn.stride()[:3]
    s.v_packed, s.vp_sb, s.vp_sh, s.vp_st = vp.data_ptr(), *vp.stride()[:3]
    s.v_norms, s.vn_sb, s.vn_sh, s.vn_st = vn.data_ptr(), *vn.stride()
    s.k_row_width, s.norm_width, s.v_row_width, s.max_T = mgr._k_rows[0], kn.shape[-1], mgr._vpb, kp.shape[2]
    if mgr.buffered:
        ar, slot, t_pos, lens, buf_len = mgr._buffered_step_indices()
        bk, bv = mgr._buf_k[0], mgr._buf_v[0]
        s.win_k, s.win_v, s.win_W = bk.data_ptr(), bv.data_ptr(), bk.shape[2]
        s.w_sb, s.w_sh, s.w_st = bk.stride()[:3]
        s.win_slot, s.win_lens = slot.data_ptr(), buf_len.data_ptr()
        scratch.update(win_old=torch.zeros(2, B, n_kv, 128, **f16), win_out=torch.zeros(B, n_q, 128, **f32), win_lse=torch.zeros(B, n_q, **f32))
        s.T = mgr.seq_len + 1 - mgr.n_sink - mgr.window
    else:
        t_pos, lens = mgr._seq_lens, mgr._seq_lens + S
        s.T = mgr.seq_len + S
    lens = lens.clone()
    lens[list(empty)] = 0
    s.t_pos, s.seq_lens = t_pos.data_ptr(), lens.data_ptr()
    out = place(torch.zeros(B, n_q, 128, **f16), scratch)
    for name, t in dict(scratch, out=out).items():
        setattr(s, name, t.data_ptr())
    fn = _capi.lib().bgtq_decode_step
    fn.restype, fn.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_void_p]
    _capi.check(fn(ctypes.byref(s), _capi.stream_ptr(DEV)), "bgtq_decode_step")
    torch.cuda.synchronize()
    return out.clone()


def _over_win_old(out, scratch):
    flat = torch.zeros(out.numel() + scratch["win_old"].numel(), dtype=torch.float16, device=DEV)
    scratch["win_old"] = flat[:scratch["win_old"].numel()].view_as(scratch["win_old"])
    return flat[:out.numel()].view_as(out)


@pytest.mark.gpu
@pytest.mark.parametrize("shared,window", [("q_rot", 0), ("q_rot", 64), ("q", 0), ("q", 64), ("win_old", 64)])
def test_output_over_a_buffer_that_is_dead_before_the_merge(shared, window):
    """264 work-groups, ragged: rows by falling length where the output is apart, as they come where it is not."""
    outs = []
    for place in (lambda out, scratch: out, lambda out, scratch: scratch[shared].view_as(out)):
        mgr, q, k, v = _filled(33, 4, 2, 1000, window)
        if shared == "win_old":
            place = _over_win_old if outs else place
        outs.append(_step(mgr, q, k, v, 2, place))
    assert torch.isfinite(outs[0]).all() and outs[0].abs().max() > 0 and torch.equal(*outs)


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [33, 130])
def test_step_without_new_tokens(batch):
    """Attention over what is there, more rows than a work-group ranks among them."""
    mgr, q, k, v = _filled(batch, 4, 2, 300)
    got = _step(mgr, q, k, v, 2, S=0)
    plans, cache = mgr._batched_args[0]["plans"], (mgr._k_packed[0], mgr._k_norms[0], mgr._v_packed[0], mgr._v_norms[0])
    want = ops.decode_attention(plans, ops.rotate_q(plans, q[:, :, 0], 4), *cache, mgr.seq_len, seq_lens=mgr._seq_lens, n_splits=2,
                                scale=mgr.scale, k_row_width=mgr._k_rows[0], v_row_width=mgr._vpb)
    assert torch.isfinite(got).all() and got.abs().max() > 0 and torch.equal(got, want.view_as(got))


# query heads a KV head (9 .. 16 are two launches over one order), types, buffer; new tokens off 16 bytes enter the buffer in a
# launch of its own, and so does the buffer's attention with one query head a KV head
@pytest.mark.gpu
@pytest.mark.parametrize("gqa,dtype,window,off", [(7, torch.float16, 0, 0), (12, torch.bfloat16, 0, 0), (1, torch.bfloat16, 0, 0), (2, torch.bfloat16, 64, 0),
                                                  (12, torch.float16, 64, 0), (4, torch.float16, 64, 1), (1, torch.float16, 64, 0)])
def test_rows_by_falling_length_and_as_they_come_are_the_same(gqa, dtype, window, off):
    """Rows that see nothing and rows of one length among them; the cache as well."""
    steps = []
    for place in (lambda out, scratch: out, lambda out, scratch: scratch["q_rot"]):
        mgr, q, k, v = _filled(33, 4, gqa, 1000, window, dtype=dtype)
        if off:
            k, v = [torch.cat([t.new_zeros(off), t.flatten()])[off:].view_as(t) for t in (k, v)]
        out = _step(mgr, q, k, v, 2, place, empty=(3, 4, 32))
        steps.append([out, mgr._k_packed[0], mgr._k_norms[0], mgr._v_packed[0], mgr._v_norms[0]] + ([mgr._buf_k, mgr._buf_v] if window else []))
    assert torch.isfinite(steps[0][0]).all() and all(torch.equal(a, b) for a, b in zip(*steps))
    assert (steps[0][0].flatten(1).abs().amax(1) > 0).tolist() == [window > 0 or b not in (3, 4, 32) for b in range(33)]


@pytest.mark.gpu
@pytest.mark.parametrize("window", [0, 64])
def test_captured_step_replays_by_falling_length(window):
    """Every replay against a step of the general path (rows as they come), inputs held."""
    (mgr, q, k, v), (general, *_) = _filled(33, 4, 2, 1000, window), _filled(33, 4, 2, 1000, window)
    mgr.n_splits = general.n_splits = 2
    general._native = lambda li: general._ensure_storage()
    assert torch.equal(mgr.append_and_attend(0, q, k, v), general.append_and_attend(0, q, k, v))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = mgr.append_and_attend(0, q, k, v)
    for turn in range(4):
        q.add_(0.125), k.mul_(1.25), v.mul_(-0.75)
        want = general.append_and_attend(0, q, k, v)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.isfinite(out).all() and torch.equal(out, want), turn
