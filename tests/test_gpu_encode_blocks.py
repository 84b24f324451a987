"""GPU: the prompt-sized encoder (blocks of 16 rows on the matrix cores) against the single-row encoder.

Both promise the same order of evaluation, so codes, records and norms agree bit for bit.  Calls of
at most 32 rows take the single-row encoder, which the checker's tests pin; larger ones take blocks, dealt to
waves (many) or split over the waves of a work-group (few)."""
import pytest
import torch

from blockgtq_amd import plan as P, workloads as wl
from blockgtq_amd.quantizer import build_batched_encode_args, encode_k_into, encode_v_into

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _plans(n_kv, bits, seed=41):
    k_bits, v_bits, lo, hi = bits
    w = wl.Workload("t", 1, n_kv, n_kv, 1, 64, 1e6, k_bits=k_bits, v_bits=v_bits, min_bits=lo, max_bits=hi, seed=seed)
    qs, _ = wl.calibrate_layer(w, 0, DEV)
    return build_batched_encode_args(qs, device=DEV)


def _encode(args, x, kl, vl, quant, T, slice_rows=None, k_width=None, row_pad=0):
    B, H, S, _ = x.shape
    kw = k_width or P.cache_row_bytes(args['max_mixed_bytes'] if kl == P.K_MIXED else args['max_tpb'])
    vw = 64 if vl == P.V_NIBBLE else args['v_packed_bytes']
    G = args['max_n_groups']
    kp = torch.full((B, H, T, kw + row_pad), 0xA5, dtype=torch.uint8, device=DEV)[..., :kw]
    kn = torch.full((B, H, T, G), 7.0, dtype=torch.float16, device=DEV)
    vp = torch.full((B, H, T, vw + row_pad), 0xA5, dtype=torch.uint8, device=DEV)[..., :vw]
    vn = torch.full((B, H, T), 7.0, dtype=torch.float16, device=DEV)
    step = slice_rows or S
    for lo in range(0, S, step):
        xs = x[:, :, lo:lo + step]
        encode_k_into(args['plans'], xs, kp, kn, 3 + lo, kw, G, kl, quant)
        encode_v_into(args['plans'], xs, vp, vn, 3 + lo, vw, vl)
    return kp, kn, vp, vn


def _same(a, b):
    for x, y in zip(a, b):
        if x.dtype == torch.float16:
            x, y = x.contiguous().view(torch.int16), y.contiguous().view(torch.int16)
        assert torch.equal(x, y)


# rows of a batch row, heads: remainders of a 16-row block, one block, few blocks, more blocks than waves
@pytest.mark.parametrize("S,n_kv,B", [(33, 1, 1), (17, 2, 3), (48, 3, 1), (250, 4, 1), (2049, 5, 1), (4099, 2, 2)])
@pytest.mark.parametrize("bits,kl,vl", [((3.0, 3, 1, 8), P.K_BITPACKED, P.V_BITPACKED), ((3.0, 3, 1, 8), P.K_MIXED, P.V_NIBBLE),
                                        ((2.0, 2, 0, 4), P.K_BITPACKED, P.V_BITPACKED), ((4.0, 4, 0, 8), P.K_MIXED, P.V_BITPACKED),
                                        ((1.0, 1, 0, 3), P.K_BITPACKED, P.V_BITPACKED)])
def test_blocks_equal_single_rows(S, n_kv, B, bits, kl, vl):
    args = _plans(n_kv, bits)
    gen = torch.Generator(device=DEV).manual_seed(S)
    x = (torch.randn(B, n_kv, S, 128, generator=gen, device=DEV) * torch.rand(B, n_kv, S, 1, generator=gen, device=DEV) * 30).half()
    x[0, 0, 5] = 0                                              # a row of zeros
    quant = P.QUANT_EXACT if S == 250 else P.QUANT_LUT256
    small = 32 // B
    _same(_encode(args, x, kl, vl, quant, S + 9), _encode(args, x, kl, vl, quant, S + 9, small))


@pytest.mark.parametrize("S", [50, 3000])
@pytest.mark.parametrize("kl", [P.K_BITPACKED, P.K_MIXED])
def test_blocks_with_odd_strides_and_nonfinite_rows(S, kl):
    """Rows off 16-byte boundaries and records off dwords; an infinity or NaN reaches only its own group."""
    args = _plans(2, (3.0, 3, 0, 5), seed=43)
    gen = torch.Generator(device=DEV).manual_seed(S)
    x = torch.randn(1, 2, S, 131, generator=gen, device=DEV).half()[..., 1:129]
    width = args['max_mixed_bytes'] if kl == P.K_MIXED else args['max_tpb']
    want = _encode(args, x, kl, P.V_BITPACKED, P.QUANT_LUT256, S + 9, 32, width, 3)
    _same(_encode(args, x, kl, P.V_BITPACKED, P.QUANT_LUT256, S + 9, None, width, 3), want)
    odd = [(0, 7, 3, float("inf")), (1, S - 2, 100, float("nan")), (1, 20, 64, float("-inf"))]
    for h, s, d, v in odd:
        x[0, h, s, d] = v
    got = _encode(args, x, kl, P.V_BITPACKED, P.QUANT_LUT256, S + 9, None, width, 3)
    for h, s, d, _ in odd:
        p = args['plans_np'][h]
        hit = int(p['group_of'][list(p['head_perm']).index(d)])
        for g in range(int(p['n_seg'])):
            if g == hit:
                continue
            assert got[1][0, h, 3 + s, g] == want[1][0, h, 3 + s, g]
            if kl == P.K_BITPACKED:
                lo = int(p['seg_pack_off'][g])
                hi = lo + P.segment_bytes(int(p['seg_bw'][g]), int(p['seg_len'][g]))
                assert torch.equal(got[0][0, h, 3 + s, lo:hi], want[0][0, h, 3 + s, lo:hi])
        assert not torch.isfinite(got[3][0, h, 3 + s])          # (V: one norm a row)
        for t in (got, want):                                   # every other row is untouched
            for o in t:
                o[0, h, 3 + s] = 0
    _same(got, want)


def test_blocks_drop_positions_outside_the_cache():
    args = _plans(1, (3.0, 3, 1, 8))
    x = torch.randn(2, 1, 40, 128, device=DEV).half()
    kw, G = P.cache_row_bytes(args['max_tpb']), args['max_n_groups']
    kp = torch.full((2, 1, 60, kw), 0xA5, dtype=torch.uint8, device=DEV)
    kn = torch.full((2, 1, 60, G), 7.0, dtype=torch.float16, device=DEV)
    pos = torch.tensor([30, -10], dtype=torch.int32, device=DEV)
    encode_k_into(args['plans'], x, kp, kn, pos, kw, G, P.K_BITPACKED)
    want, wn = _encode(args, x, P.K_BITPACKED, P.V_BITPACKED, P.QUANT_LUT256, 43, 16)[:2]
    assert torch.equal(kp[0, 0, 30:], want[0, 0, 3:33]) and torch.equal(kp[1, 0, :30], want[1, 0, 13:])
    assert (kp[0, 0, :30] == 0xA5).all() and (kp[1, 0, 30:] == 0xA5).all() and (kn[1, 0, 30:] == 7.0).all()


# 8 heads of K or V: 64 blocks are still a work-group each, from 65 on two waves share a block (3 of them a work-group, the
# last work-group not full; exactly 8), from 257 on every wave has its own (9 a work-group, in one round; 17, in two)
@pytest.mark.parametrize("S", [1024, 1025, 2010, 4096, 4097, 8200])
@pytest.mark.parametrize("bits,kl,vl", [((3.0, 3, 1, 8), P.K_MIXED, P.V_NIBBLE), ((4.0, 4, 0, 8), P.K_BITPACKED, P.V_BITPACKED)])
def test_blocks_by_waves_per_block(S, bits, kl, vl):
    args = _plans(8, bits, seed=47)
    gen = torch.Generator(device=DEV).manual_seed(S)
    x = (torch.randn(1, 8, S, 128, generator=gen, device=DEV) * torch.rand(1, 8, S, 1, generator=gen, device=DEV) * 30).half()
    x[0, 0, 5] = 0
    x[0, 3, S - 1, 77] = float("inf")                          # (the other rows of its block take another way)
    got, want = _encode(args, x, kl, vl, P.QUANT_LUT256, S + 9), _encode(args, x, kl, vl, P.QUANT_LUT256, S + 9, 32)
    for o in got + want:
        o[0, 3, 3 + S - 1] = 0
    _same(got, want)


@pytest.mark.parametrize("S", [100, 1100, 4100])
def test_blocks_over_the_whole_fp16_range(S):
    """Rows of any finite fp16 values, of few of the largest, of subnormals only and of zeros, as blocks and one by one."""
    args = _plans(8, (3.0, 3, 0, 8), seed=48)
    gen = torch.Generator(device=DEV).manual_seed(S)
    x = torch.randint(0, 0x7C00, (1, 8, S, 128), generator=gen, device=DEV, dtype=torch.int16)
    x[:, :, 1::5] &= 0x3FF                                     # subnormals
    x[:, :, 2::5] *= (torch.rand(1, 8, len(range(2, S, 5)), 128, generator=gen, device=DEV) < 0.05)
    x[:, :, 3::5] = 0
    x[:, :, 4::5] = x[:, :, 4::5] // 8 + 0x3000                # of one size
    x = torch.where(torch.rand(x.shape, generator=gen, device=DEV) < 0.5, x, x | -0x8000).view(torch.float16)
    _same(_encode(args, x, P.K_MIXED, P.V_NIBBLE, P.QUANT_LUT256, S + 9), _encode(args, x, P.K_MIXED, P.V_NIBBLE, P.QUANT_LUT256, S + 9, 32))


def test_segment_tables_of_the_block_encoder():
    """`rot_span` covers the rows that 16 columns' segments reach, the segment nibbles repeat `group_of`."""
    for bits in ((3.0, 3, 1, 8), (2.0, 2, 0, 4), (1.0, 1, 0, 3)):
        for p in _plans(2, bits)['plans_np']:
            seg = p['lut_image'][P.K_BITPACKED][P.LUT_KSEG // 4:][:16].reshape(4, 4)
            rot = p['k_rot_T'].reshape(128, 128)
            for k in range(128):
                assert (int(seg[k % 4, k // 32]) >> (4 * ((k // 4) % 8))) & 15 == max(int(p['group_of'][k]), 0)
                lo, hi = int(p['rot_span'][k // 16]) & 15, int(p['rot_span'][k // 16]) >> 4
                rows = [r for r in range(128) if rot[r, k] and p['group_of'][k] >= 0]
                assert all(16 * lo <= r < 16 * hi for r in rows)
