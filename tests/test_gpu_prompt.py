"""GPU: prompt attention with a workspace (staged records, queries rotated inside, partitions merged)
against the kernel that takes rotated queries and no workspace.

Both dequantise to the same fp16 records and sum in fp32; they round probabilities, outputs and
rotated queries to fp16 from sums in another order, i.e. each value is off by at most one rounding
(2^-11 of it, 3e-4 on average) in three places: 2e-3 of the output's norm bounds them together."""
import numpy as np
import pytest
import torch

from blockgtq_amd import _capi, ops, plan as P, workloads as wl
from blockgtq_amd.quantizer import build_batched_encode_args, encode_k_into, encode_v_into

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _cache(B, n_kv, T, kl, vl, bits):
    k_bits, v_bits, lo, hi = bits
    w = wl.Workload("t", 1, n_kv, n_kv, B, T, 1e6, k_bits=k_bits, v_bits=v_bits, min_bits=lo, max_bits=hi, seed=51)
    qs, e = wl.calibrate_layer(w, 0, DEV)
    args = build_batched_encode_args(qs, device=DEV)
    return args, qs, _encode(args, *wl.draw_kv(w, e, T, 3, DEV), kl, vl)


def _no_workspace(args, q_rot, cache, T, off, causal, kl, vl, unrotate):
    kp, kn, vp, vn = cache
    B, n_q, S, _ = q_rot.shape
    n_kv = kp.shape[1]
    out = torch.empty_like(q_rot)
    p = _capi.ptr
    _capi.check(_capi.lib().bgtq_prefill_attn(
        p(args['plans']), p(q_rot), *q_rot.stride()[:3], p(kp), *kp.stride()[:3], kp.shape[-1], p(kn), *kn.stride()[:3],
        p(vp), *vp.stride()[:3], vp.shape[-1], p(vn), *vn.stride(), B, n_kv, n_q // n_kv, S, T, off, int(causal), kl, vl,
        128 ** -0.5, int(unrotate), p(out), *out.stride()[:3], _capi.stream_ptr()), "bgtq_prefill_attn")
    return out


# (B, n_kv, query heads per KV head, queries, records, first position): one row, a long context for few rows
# (partitions and merge), odd groups, groups wider than the small work-group, tile edges, rows that see nothing
# of the last tile, many rows
@pytest.mark.parametrize("B,n_kv,gqa,S,T,off", [
    (1, 1, 1, 1, 1, 0), (1, 2, 1, 16, 3000, 2984), (2, 1, 7, 37, 137, 100), (1, 2, 40, 9, 640, 631), (1, 1, 130, 5, 129, 124),
    (1, 1, 4, 64, 64, 0), (1, 1, 4, 65, 65, 0), (1, 2, 3, 300, 500, 50), (1, 8, 4, 1000, 1000, 0)])
@pytest.mark.parametrize("kl,vl,bits,dtype", [(P.K_BITPACKED, P.V_BITPACKED, (3.0, 3, 1, 5), torch.bfloat16),
                                              (P.K_MIXED, P.V_NIBBLE, (2.5, 2, 0, 8), torch.float16)])
def test_prompt_attention_equals_the_kernel_without_workspace(B, n_kv, gqa, S, T, off, kl, vl, bits, dtype):
    args, qs, cache = _cache(B, n_kv, T, kl, vl, bits)
    gen = torch.Generator(device=DEV).manual_seed(S + T)
    q = torch.randn(B, S, n_kv * gqa, 128, generator=gen, device=DEV).to(dtype).transpose(1, 2)
    rot = []
    for h, q8 in enumerate(qs):
        m = torch.zeros(128, 128, dtype=torch.float64, device=DEV)
        m[q8._head_perm] = q8._block_rot_T.double()
        rot.append((q[:, h * gqa:(h + 1) * gqa].double() @ m).half())
    q_rot = torch.cat(rot, 1).contiguous()
    for causal, unrotate in ((True, True), (False, False)):
        want = _no_workspace(args, q_rot, cache, T, off, causal, kl, vl, unrotate).float()
        kw = dict(k_layout=kl, v_layout=vl, is_causal=causal, q_pos_offset=off, unrotate=unrotate)
        got = {"rotated": ops.prefill_attention_packed(args['plans'], q_rot, *cache, T, **kw)}
        got["raw"] = ops.prefill_attention_packed(args['plans'], q, *cache, T, rotate_q=True, **kw)
        for name, g in got.items():
            assert g.shape == want.shape and torch.isfinite(g).all()
            assert (g.float() - want).norm() <= 2e-3 * want.norm(), name


def _plans_of(bits):
    k_bits, v_bits, lo, hi = bits
    w = wl.Workload("t", 1, 1, 1, 1, 64, 1e6, k_bits=k_bits, v_bits=v_bits, min_bits=lo, max_bits=hi, seed=52)
    return build_batched_encode_args(wl.calibrate_layer(w, 0, DEV)[0], device=DEV)


def _encode(args, k, v, kl, vl):
    B, n_kv, T, _ = k.shape
    kw = P.cache_row_bytes(args['max_mixed_bytes'] if kl == P.K_MIXED else args['max_tpb'])
    vw = 64 if vl == P.V_NIBBLE else args['v_packed_bytes']
    kp = torch.zeros(B, n_kv, T, kw, dtype=torch.uint8, device=DEV)
    kn = torch.zeros(B, n_kv, T, args['max_n_groups'], dtype=torch.float16, device=DEV)
    vp = torch.zeros(B, n_kv, T, P.cache_row_bytes(vw), dtype=torch.uint8, device=DEV)[..., :vw]
    vn = torch.zeros(B, n_kv, T, dtype=torch.float16, device=DEV)
    encode_k_into(args['plans'], k, kp, kn, 0, kw, kn.shape[-1], kl)
    encode_v_into(args['plans'], v, vp, vn, 0, vw, vl)
    return kp, kn, vp, vn


@pytest.mark.parametrize("bits", [(4.0, 4, 1, 8), (5.0, 3, 3, 8)])
@pytest.mark.parametrize("kl,vl", [(P.K_BITPACKED, P.V_BITPACKED), (P.K_MIXED, P.V_NIBBLE)])
def test_records_with_several_raw_byte_segments(bits, kl, vl):
    """5- and 6-bit codes and wider in one record, both kernels against fp64 attention over the records that another kernel
    dequantises: probabilities and outputs are rounded to fp16 once each, 2^-11 of their size at most."""
    T, S = 200, 64
    args = _plans_of(bits)
    assert (args['plans_np'][0]['seg_bw'] > 4).sum() > 1
    gen = torch.Generator(device=DEV).manual_seed(6)
    k, v = (torch.randn(1, 1, T, 128, generator=gen, device=DEV).half() for _ in range(2))
    cache = _encode(args, k, v, kl, vl)
    k_hat, v_hat = (t.double() for t in ops.dequant_kv(args['plans'], *cache, T, k_layout=kl, v_layout=vl))
    q = torch.randn(1, 2, S, 128, generator=gen, device=DEV).half()
    want = torch.softmax(q.double() @ k_hat.transpose(2, 3).contiguous() * 128 ** -0.5, 3) @ v_hat
    got = ops.prefill_attention_packed(args['plans'], q, *cache, T, k_layout=kl, v_layout=vl, is_causal=False, unrotate=False)
    for g in (got, _no_workspace(args, q, cache, T, 0, False, kl, vl, False)):
        assert (g.double() - want).norm() <= 2 ** -10 * want.norm()


# query heads wider than the small work-group over a split context: the merge with eight waves a group of rows, and with one
@pytest.mark.parametrize("gqa,S,T,off", [(130, 3, 2000, 1997), (130, 40, 1100, 1060), (256, 2, 900, 890)])
def test_wide_query_groups_over_a_split_context(gqa, S, T, off):
    test_prompt_attention_equals_the_kernel_without_workspace(1, 1, gqa, S, T, off, P.K_MIXED, P.V_NIBBLE, (2.5, 2, 0, 8), torch.float16)


# work-groups of two teams: an early block whose first team has no tile, a ragged end, teams that still leave partitions to merge
@pytest.mark.parametrize("n_kv,gqa,S,T,off", [(8, 4, 800, 800, 0), (8, 3, 1000, 1801, 777), (4, 4, 1000, 1027, 27)])
def test_two_teams_over_one_block_of_rows(n_kv, gqa, S, T, off):
    test_prompt_attention_equals_the_kernel_without_workspace(1, n_kv, gqa, S, T, off, P.K_MIXED, P.V_NIBBLE, (2.5, 2, 0, 8), torch.float16)
    test_prompt_attention_equals_the_kernel_without_workspace(1, n_kv, gqa, S, T, off, P.K_BITPACKED, P.V_BITPACKED, (3.0, 3, 1, 5), torch.bfloat16)


# staging in shares of two tiles, the last of one; fewer (row, head) pairs than XCDs, and more
@pytest.mark.parametrize("B,n_kv,T", [(2, 3, 5800), (3, 4, 2817)])
def test_several_tiles_to_a_staging_work_group(B, n_kv, T):
    assert 512 < -(-T // 64) * B * n_kv <= 1024 and -(-T // 64) % 2 == 1
    test_prompt_attention_equals_the_kernel_without_workspace(B, n_kv, 2, 20, T, T - 20, P.K_MIXED, P.V_NIBBLE, (2.5, 2, 0, 8), torch.float16)


def test_small_probabilities_count_in_the_denominator():
    """Each query has one strong record among the first and 65 535 weak ones, e^-18 of it apiece and below the smallest fp16
    number once the reference lies 4 octaves above the strong score; together they are 4e-3 of the denominator.
    As fp16 values they lose most of that.  The numerator may drop them: over thousands of unrelated values
    they come to some 1e-4 of the output; the rest of the bound is the output's own rounding (2^-11 at most)."""
    T, gqa, n = 65536, 16, 32
    args = _plans_of((4.0, 4, 1, 8))
    gen = torch.Generator(device=DEV).manual_seed(5)
    x = torch.randn(1, 1, T, 128, generator=gen, device=DEV)
    cache = _encode(args, x.half(), torch.randn(1, 1, T, 128, generator=gen, device=DEV).half(), P.K_BITPACKED, P.V_BITPACKED)
    k_hat, v_hat = (t[0, 0].double() for t in ops.dequant_kv(args['plans'], *cache, T))
    own = k_hat[:n]
    q = (own / own.square().sum(1, keepdim=True) * 18 * 128 ** 0.5).half()      # a score of 18 on the own record, 0 +- 1.6 elsewhere
    p = torch.softmax(q.double() @ k_hat.T * 128 ** -0.5, 1)
    assert (1 - p.max(1).values).min() > 2e-3
    want = p @ v_hat
    rows = q.repeat(4096 // n, 1).expand(1, gqa, 4096, 128)                     # (enough rows that the context is not split)
    got = ops.prefill_attention_packed(args['plans'], rows, *cache, T, is_causal=False, unrotate=False)
    got = got[0].reshape(-1, n, 128)
    assert torch.equal(got, got[:1].expand_as(got))
    assert (got[0].double() - want).norm() <= 6e-4 * want.norm()


@pytest.mark.parametrize("shift", [0, 14])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_rotation_keeps_the_bits_of_small_entries(shift, dtype):
    """The rotation counts with all its fp32 bits, whatever the size of its entries: entries scaled by 2^-14 against queries
    scaled by 2^14 give the same products.  An fp32 sum of 128 terms lands on the other side of an fp16 midpoint in about
    2^-24 sqrt(128) / 2^-12 of the cases, 3e-3, so 70 % of the rows meet none and agree bit for bit; 0.4 is asked for."""
    n_kv, S, T = 2, 256, 200
    args, qs, cache = _cache(1, n_kv, T, P.K_BITPACKED, P.V_BITPACKED, (3.0, 3, 1, 5))
    gen = torch.Generator(device=DEV).manual_seed(9)
    q = torch.randn(1, n_kv, S, 128, generator=gen, device=DEV).mul(0.7).clamp(-3.9, 3.9).to(dtype)
    rot = []
    for h, q8 in enumerate(qs):
        m = torch.zeros(128, 128, dtype=torch.float64, device=DEV)
        m[q8._head_perm] = q8._block_rot_T.double()
        rot.append((q[:, h:h + 1].double() @ m).half())
    want = ops.prefill_attention_packed(args['plans'], torch.cat(rot, 1), *cache, T, scale=0.5, is_causal=False, unrotate=False)
    small = args['plans_np'].copy()
    small['k_rot_T'] *= np.float32(2.0 ** -shift)
    got = ops.prefill_attention_packed(P.upload_plans(small, DEV), q * 2.0 ** shift, *cache, T, scale=0.5, is_causal=False,
                                       unrotate=False, rotate_q=True)
    same = (got == want).all(-1).float().mean().item()
    assert same >= 0.4, same


def test_many_query_rows_in_one_call():
    """65 600 tokens of 32 query heads on one KV head, more groups of 32 rows than one grid dimension holds: as two halves."""
    args, _, cache = _cache(1, 1, 70, P.K_BITPACKED, P.V_BITPACKED, (3.0, 3, 1, 5))
    S = 65600
    q = torch.randn(1, 32, S, 128, device=DEV, dtype=torch.float16)
    got = ops.prefill_attention_records(args['plans'], q, *cache, 70, is_causal=False)
    for part in (slice(0, S // 2), slice(S // 2, S)):
        assert torch.equal(got[:, :, part], ops.prefill_attention_records(args['plans'], q[:, :, part], *cache, 70, is_causal=False))


def test_workspace_covers_the_records_that_are_seen():
    """A causal call near the start of a long cache stages what its rows see: 100 records, not 40 000."""
    T = 40000
    args, _, cache = _cache(1, 1, T, P.K_BITPACKED, P.V_BITPACKED, (3.0, 3, 1, 5))
    q = torch.randn(1, 4, 60, 128, device=DEV, dtype=torch.float16)
    want = ops.prefill_attention_packed(args['plans'], q, *[t[:, :, :100] for t in cache], 100, q_pos_offset=40)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    got = ops.prefill_attention_packed(args['plans'], q, *cache, T, q_pos_offset=40)
    torch.cuda.synchronize()
    assert torch.cuda.max_memory_allocated() - before < 2 << 20
    assert torch.equal(got, want)


@pytest.mark.parametrize("rotate", [False, True])
def test_without_room_for_the_workspace(rotate):
    """8 heads of 32 768 records stage into 134 MB.  Where the device has no room for that the kernel that takes none attends
    (records of one tile at a time in LDS; the two agree as in the first test)."""
    B, n_kv, T, S = 1, 8, 32768, 24
    args, qs, cache = _cache(B, n_kv, T, P.K_BITPACKED, P.V_BITPACKED, (3.0, 3, 1, 5))
    q = torch.randn(B, S, 4 * n_kv, 128, device=DEV).half().transpose(1, 2)
    kw = dict(q_pos_offset=T - S, rotate_q=rotate)
    want = ops.prefill_attention_records(args['plans'], q, *cache, T, **kw).float()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / total)
    try:
        got = ops.prefill_attention_records(args['plans'], q, *cache, T, **kw).float()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert (got - want).norm() <= 2e-3 * want.norm()
