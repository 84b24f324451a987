// Dequantisation of one 64-token tile of packed records in LDS, shared by the prompt-phase kernels (internal).
//
// Raw K and V records, their norms and the plan's pair tables lie in LDS (V table at address 0, K tables at
// BGTQ_VLUT_BYTES); 8 waves write an fp16 K tile [token][dim] (packed-dim order, rows KROW bytes apart) and a
// transposed fp16 V tile [dim][token] (rows VTROW bytes apart), both fp16(centroid * norm).
#pragma once
#include "bgtq_lds.h"

namespace {

constexpr int DQ_MT = 64;                       // tokens per tile
constexpr int DQ_WAVES = 8;
constexpr int DQ_THR = 64 * DQ_WAVES;
constexpr int DQ_VUPT = 16 * 32 / DQ_THR;       // V tile: 32 token pairs x 16 units over the threads
constexpr int DQ_UPW = (BGTQ_MAX_UNITS + DQ_WAVES - 1) / DQ_WAVES;   // K units per wave
constexpr int DQ_KROW = BGTQ_D * 2 + 16;        // bytes of a K tile row: rows 4 banks apart
constexpr int DQ_VTROW = DQ_MT * 2 + 16;        // bytes of a transposed V tile row (one dim, 64 tokens)
constexpr int DQ_TILE_BYTES = DQ_MT * DQ_KROW + BGTQ_D * DQ_VTROW;

__device__ __forceinline__ uint32_t pk_mul_f16(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_pk_mul_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// Copies the tables of head plan P for the layouts in use: every wave its share of 1 KB chunks.
__device__ __forceinline__ void dq_load_tables(const bgtq_head_plan& P, int kl, bool vnib, int vbw, int wave, uint32_t voff) {
    const uint8_t* vimg = (const uint8_t*)P.vlut_image[vnib ? 1 : 0];
    const uint8_t* kimg = (const uint8_t*)P.lut_image[kl];
    const int vbytes = (vnib || vbw == 4) ? 1024 : (1 << (2 * vbw)) * 128;
    const int kbytes = kl == BGTQ_K_MIXED ? BGTQ_LUTM_KEND : BGTQ_LUT_KEND;
    const int vch = (vbytes + 1023) >> 10, kch = (kbytes + 1023) >> 10;
    for (int cc = wave; cc < vch + kch; cc += DQ_WAVES) {
        const uint8_t* src;
        uint32_t dst;
        int left;
        if (cc < vch) { src = vimg + cc * 1024; dst = cc * 1024; left = vbytes - cc * 1024; }
        else { src = kimg + (cc - vch) * 1024; dst = BGTQ_VLUT_BYTES + (cc - vch) * 1024; left = kbytes - (cc - vch) * 1024; }
        dma16(voff, src, __builtin_amdgcn_readfirstlane(dst), __builtin_amdgcn_ballot_w64((int)voff < left));
    }
}

struct TileDequant {
    // The K units of this wave (w, w + DQ_WAVES, then the third round shifted by half: the first waves also issue
    // loads): their parameters stay in scalar registers.  A unit the wave does not have reads valid addresses and
    // stores nothing (len 0).
    struct KUnit { uint32_t rot[4], mask, tab, repm, off, d0x2, seg2; int len; bool raw; };
    KUnit ku[DQ_UPW];
    uint32_t rep, vrot[4], vfmask, vbase, vcol;
    int lane, tp, up, vbw;

    __device__ __forceinline__ void init(const bgtq_head_plan& P, int kl, bool vnib, int tid) {
        lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        vbw = vnib ? 4 : (int)P.v_bits;                          // bits of a V code as stored
        const bool vrep = !vnib && vbw <= 3;                     // V pair table replicated over the banks
        const int n_units = min(P.n_units[kl], BGTQ_MAX_UNITS), n_pair = min(P.n_pair_units[kl], n_units);
        const uint32_t kend = P.kend[kl], kfirst0 = P.kfirst[kl][0], kfirst1 = P.kfirst[kl][1];
        rep = ((uint32_t)lane & 31u) * 4u;
        // V: thread (token pair tp, unit up); code pair e of a unit's raw word is brought to the table-index position by
        // a rotation (the V table sits at LDS address 0).  Neighbouring lanes take neighbouring units of one token pair:
        // a half-wave then reads 16 token pairs (records 96 bytes apart fall on 8 banks) instead of 32
        tp = (tid >> 1) & 31;
        up = 2 * (tid >> 6) + (tid & 1);
        // Column order of the V^T tile: inside every group of 16 tokens, token x sits at position
        // 8 ((x >> 2) & 1) + 4 (x >> 3) + (x & 3), so that the 8 tokens {4 g + i, 8 + 4 g + i} a half-wave g contracts
        // in one MFMA step are 16 contiguous bytes.  Tokens 2 tp and 2 tp + 1 stay neighbours: byte offset of their dword
        vcol = (uint32_t)(8 * (tp >> 3) + 4 * ((tp >> 1) & 1) + 2 * ((tp >> 2) & 1) + (tp & 1)) * 4;
        const int vtsh = vrep ? 7 : 2;
#pragma unroll
        for (int e = 0; e < 4; e++) vrot[e] = (uint32_t)(2 * vbw * e - vtsh) & 31u;
        vfmask = ((1u << (2 * vbw)) - 1u) << vtsh;
        vbase = vrep ? rep : 0u;
#pragma unroll
        for (int i = 0; i < DQ_UPW; i++) {
            const int u = i < 2 ? wave + i * DQ_WAVES : i * DQ_WAVES + (wave + DQ_WAVES / 2) % DQ_WAVES;
            const bool have = u < n_units;
            const int uu = have ? u : 0;
            const uint32_t dsc = P.kunit[kl][uu];
            ku[i].len = have ? (int)(dsc >> 8) & 0xFF : 0;
            ku[i].d0x2 = (dsc & 0xFF) * 2;
            ku[i].raw = have && ku[i].len > 0 && u >= n_pair;
            const bool pair = have && ku[i].len > 0 && u < n_pair;
#pragma unroll
            for (int e = 0; e < 4; e++) ku[i].rot[e] = pair ? P.kprog[kl][uu][e] : 0u;
            ku[i].mask = pair ? P.kprog[kl][uu][4] : 0u;
            ku[i].tab = ku[i].len > 0 ? P.kprog[kl][uu][5] : (uint32_t)BGTQ_VLUT_BYTES;
            ku[i].repm = pair ? P.kprog[kl][uu][6] : 0u;
            ku[i].off = ku[i].len == 0 ? 0u : uu == 0 ? kfirst0 : uu == 1 ? kfirst1 : P.kprog[kl][uu - 2][7];
            ku[i].seg2 = ku[i].len == 0 ? 0u : 2u * (uint32_t)__builtin_popcount(kend & ((1u << uu) - 1u));
        }
    }

    // LDS addresses: this lane's K record and its norm row, the tile's first V norm and V record, the two tiles.
    // nt records are the tile's own; the rows behind them hold stale bytes and get norm 0 (their products must
    // stay finite).  K and V go through the same three stages together, without a branch between them, so
    // that all LDS round trips of a stage overlap: codes and norms, table lookups, products and stores.
    __device__ __forceinline__ void run(uint32_t krow_l, uint32_t knrow_l, uint32_t vnorm0, uint32_t vrec0, int vrow, int nt,
                                        uint32_t ktile, uint32_t vtile) const {
        uint32_t nn[DQ_UPW], kw[DQ_UPW][4];
        uint2v rr[DQ_UPW];
        uint32_t nrm[2], vr[DQ_VUPT][2], vw[DQ_VUPT][2][4];
        // ---- stage 1
#pragma unroll
        for (int i = 0; i < DQ_UPW; i++) {
            const uint32_t n16 = lds_at<uint16_t>(knrow_l + ku[i].seg2);
            nn[i] = lane < nt ? n16 | (n16 << 16) : 0u;
            rr[i] = lds_codes8(krow_l + ku[i].off);
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t n16 = lds_at<uint16_t>(vnorm0 + (uint32_t)(2 * tp + j) * 2);
            nrm[j] = 2 * tp + j < nt ? n16 | (n16 << 16) : 0u;
        }
#pragma unroll
        for (int uu = 0; uu < DQ_VUPT; uu++)
#pragma unroll
            for (int j = 0; j < 2; j++)
                vr[uu][j] = lds_codes4(vrec0 + (uint32_t)(2 * tp + j) * vrow + (uint32_t)((DQ_VUPT * up + uu) * vbw));
        // ---- stage 2
#pragma unroll
        for (int i = 0; i < DQ_UPW; i++) {
            const uint32_t r = rr[i].x;
            const uint32_t base = and_or(rep, ku[i].repm, ku[i].tab);
#pragma unroll
            for (int e = 0; e < 4; e++)
                kw[i][e] = lds_at<uint32_t>(and_or(__builtin_amdgcn_alignbit(r, r, ku[i].rot[e]), ku[i].mask, base));
        }
#pragma unroll
        for (int uu = 0; uu < DQ_VUPT; uu++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    vw[uu][j][e] = lds_at<uint32_t>(and_or_v(__builtin_amdgcn_alignbit(vr[uu][j], vr[uu][j], vrot[e]), vfmask, vbase));
#pragma unroll
        for (int i = 0; i < DQ_UPW; i++) {
            if (ku[i].raw) {                                     // (wave-uniform) one byte per code, one fp16 per table entry
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t x = e < 2 ? rr[i].x : rr[i].y;
                    const uint32_t c0 = ku[i].tab + ((x >> ((e & 1) * 16)) & 0xFF) * 2;
                    const uint32_t c1 = ku[i].tab + ((x >> ((e & 1) * 16 + 8)) & 0xFF) * 2;
                    kw[i][e] = (uint32_t)lds_at<uint16_t>(c0) | ((uint32_t)lds_at<uint16_t>(c1) << 16);
                }
            }
        }
        // ---- stage 3.  A dim pair past the unit's last dim goes to the 16 spare bytes at the end of the lane's
        // K tile row, which nothing reads.
        const uint32_t krow_t = ktile + (uint32_t)lane * DQ_KROW;
#pragma unroll
        for (int i = 0; i < DQ_UPW; i++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                lds_put<uint32_t>(krow_t + (2 * e < ku[i].len ? ku[i].d0x2 + e * 4 : (uint32_t)(BGTQ_D * 2)), pk_mul_f16(kw[i][e], nn[i]));
#pragma unroll
        for (int uu = 0; uu < DQ_VUPT; uu++) {
            const int u = DQ_VUPT * up + uu;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t w0 = pk_mul_f16(vw[uu][0][e], nrm[0]), w1 = pk_mul_f16(vw[uu][1][e], nrm[1]);
                // (dim 8u + 2e of both tokens), (dim 8u + 2e + 1 of both tokens)
                const uint32_t lo = __builtin_amdgcn_perm(w1, w0, 0x05040100u);
                const uint32_t hi = __builtin_amdgcn_perm(w1, w0, 0x07060302u);
                lds_put<uint32_t>(vtile + (uint32_t)(8 * u + 2 * e) * DQ_VTROW + vcol, lo);
                lds_put<uint32_t>(vtile + (uint32_t)(8 * u + 2 * e + 1) * DQ_VTROW + vcol, hi);
            }
        }
    }
};

}  // namespace
