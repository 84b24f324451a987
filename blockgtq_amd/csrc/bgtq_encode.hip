// K / V quantise-and-pack kernels and the query rotation for gfx950.
//
// Arithmetic contract (what "bit-exact" means for the packed bytes): every
// reduction over coordinates is a chain of fused multiply-adds in ascending
// packed-dim order starting from +0, square roots and divisions are IEEE
// correctly rounded, and the rotation of coordinate j of a group spanning dims
// [s, e) is fma(xhat[k], R_T[k][j], acc) for k = s .. e-1 (skipped altogether,
// y = xhat, when the group's rotation block is the identity).  This file is
// compiled with floating-point contraction off so nothing else fuses.
//
// Two encoders keep it: a work-group of 128 threads for every row of a decode append (encode_row: thread j
// owns packed dim j during normalise / rotate / quantise and output byte j while packing), and blocks of 16
// rows on the matrix cores for anything larger (encode_blocks).
#include <algorithm>
#include <type_traits>

#include "bgtq_decode.h"
#include "bgtq_lds.h"

namespace {

constexpr int D = BGTQ_D;
constexpr int NT = 128;  // threads per work-group


struct EncodeArgs {
    const bgtq_head_plan* plans;
    const uint16_t* x;          // fp16 [B][n_kv][S][128]
    int64_t x_sb, x_sh, x_ss;
    int B, n_kv, S;
    uint8_t* packed;            // cache records, or nullptr
    int64_t p_sb, p_sh, p_st;
    int row_width;
    uint16_t* norms;            // fp16 cache norms, or nullptr
    int64_t n_sb, n_sh, n_st;
    int norm_width;
    const int32_t* t_pos;
    int t_pos_scalar;
    int max_T;                  // token capacity of the cache: records at positions outside [0, max_T) are dropped
    int layout;
    int quant_mode;
    uint8_t* codes_out;         // [N][128] unpacked codes, or nullptr
    float* norms_f32_out;       // K: [N][norm_width] fp32; or nullptr
    int corrected;              // K codes path: emit corrected norms
    int bf16;                   // x holds bf16: rounded to fp16 as it is read
};

// One byte of the LSB-first stream of bw-bit codes (bw <= 4) covers the codes first .. first + n - 1,
// the first of them from its bit `skip` on.  None of this depends on the row: the plan holds it per
// record byte (enc_byte, enc_vbyte).
struct StreamSlot { int first, n, skip; };
// All (at most 8) code reads are issued at once: the append of a few rows is bound by latency, one LDS
// round trip per code is what a loop would cost.
__device__ inline unsigned stream_byte_batched(const uint8_t* codes, StreamSlot s, int bw) {
    unsigned c[8];
#pragma unroll
    for (int i = 0; i < 8; i++) c[i] = codes[s.first + min(i, s.n - 1)];
    unsigned w = 0;
#pragma unroll
    for (int i = 0; i < 8; i++)
        if (i < s.n) w |= c[i] << (i * bw);
    return (w >> s.skip) & 0xFFu;
}

// Row n of the [B][S] input is (batch b, step s).  The row count fits 32 bits (the launchers
// check), so this is one 32-bit division instead of the 64-bit software routine.
__device__ inline void split_row(int64_t n, int S, int& b, int& s) {
    const unsigned q = (unsigned)n / (unsigned)S;
    b = (int)q;
    s = (int)((unsigned)n - q * (unsigned)S);
}

// Plan tables a work-group needs, copied to LDS with one burst of independent loads:
// every later table access is an LDS read instead of one more dependent trip to memory.
struct StagedK {
    int hdr[56];                 // n_seg .. seg_identity, as at the start of bgtq_head_plan
    uint8_t code_lut[BGTQ_MAX_SEGMENTS * BGTQ_LUT_BINS];
    float centroids[BGTQ_MAX_SEGMENTS * 32];   // first 32 levels of every segment (bw <= 5)
};
struct StagedV {
    int v_bits;
    float centroids[16];
    float boundaries[16];
};
constexpr int H_NSEG = 0, H_NZERO = 1, H_NOPACK_START = 4, H_NOPACK_LEN = 5, H_VBITS = 6;
constexpr int H_BW = 8, H_START = 16, H_LEN = 24, H_PACK_OFF = 32, H_IDENT = 48;

// The 128 x 128 fp32 rotation as 4096 pieces of 16 bytes: thread j fetches pieces j, j + 128, ...
// (a wave reads 1 KB of consecutive addresses per instruction) and later parks them at the same
// offsets in LDS, where thread j reads column j (consecutive lanes, consecutive banks).
static_assert(offsetof(bgtq_head_plan, k_rot_T) % 16 == 0 && offsetof(bgtq_head_plan, v_rot_T) % 16 == 0 &&
              sizeof(bgtq_head_plan) % 16 == 0, "rotations are read 16 bytes at a time");
typedef float rot_piece __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void fetch_rotation(const float* M, const int j, rot_piece (&st)[D / 4]) {
#pragma unroll
    for (int i = 0; i < D / 4; i++) st[i] = ((const rot_piece*)M)[i * NT + j];
}
__device__ __forceinline__ void park_rotation(float* rot_s, const int j, const rot_piece (&st)[D / 4]) {
#pragma unroll
    for (int i = 0; i < D / 4; i++) ((rot_piece*)rot_s)[i * NT + j] = st[i];
}

// Sum of x[k]^2 over a whole row of D values in LDS (V) as ONE fmaf chain in increasing k.  The reads
// of a batch are all issued before its first fmaf (left to itself the compiler waits for every few reads in
// turn), AHEAD: under the chain of the batch before (3 trips to LDS less; 50 registers more, which the launch with the
// window does not have); the chain itself runs at the 8 clocks of a dependent instruction.
template <bool AHEAD>
__device__ __forceinline__ float chain_sumsq_row(const float* x) {
    constexpr int CB = 32;
    float ss = 0.f;
    float4 v[AHEAD ? 2 : 1][CB / 4];
    auto load = [&](const int blk) {
#pragma unroll
        for (int i = 0; i < CB / 4; i++) v[AHEAD ? blk & 1 : 0][i] = *(const float4*)&x[CB * blk + 4 * i];
    };
    if (AHEAD) load(0);
#pragma unroll
    for (int blk = 0; blk < D / CB; blk++) {
        if (!AHEAD) load(blk);
        else if (blk + 1 < D / CB) load(blk + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < CB / 4; i++) {
            const float4 x4 = v[AHEAD ? blk & 1 : 0][i];
            ss = __builtin_fmaf(x4.x, x4.x, ss);
            ss = __builtin_fmaf(x4.y, x4.y, ss);
            ss = __builtin_fmaf(x4.z, x4.z, ss);
            ss = __builtin_fmaf(x4.w, x4.w, ss);
        }
        if (AHEAD) __builtin_amdgcn_sched_barrier(0);
    }
    return ss;
}

// The same over x[k0 .. k1 - 1], lanes with ranges of their own: eight values at a time, the next eight
// under them (a term 0 * 0 leaves the sum as it is; 15 values past the range are readable).  K's corrected norm, whose
// loop waited for every value by itself: 8 rows x 2 heads of 32k nibble records 154.4 -> 150.7 us a pass of four layers.
// (K's first norm gains nothing by it: 0 to +0.7 % on whole passes.)
__device__ __forceinline__ float chain_sumsq_span(const float* x, const int k0, const int k1) {
    float ss = 0.f, v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = x[k0 + i];
    for (int k = k0; k < k1; k += 8) {
        float w[8];
#pragma unroll
        for (int i = 0; i < 8; i++) w[i] = x[k + 8 + i];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float m = k + i < k1 ? v[i] : 0.f;
            ss = __builtin_fmaf(m, m, ss);
        }
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = w[i];
    }
    return ss;
}

// Thread j = 0 .. 127 of its row.  PAIRED: the V row and the K row of one token by the two halves of a work-group, which
// meet the same barriers (V's chains have fewer stages, K's barriers are met all the same).  ring: the row is the token that leaves slot
// ring->slot[b] of the fp16 buffer, and the new one takes its place.
struct RingArgs {
    const int32_t* slot;
    uint16_t* buf; int64_t b_sb, b_sh, b_st; int W;
    const uint16_t* in; int64_t in_sb, in_sh; int bf16;
};
template <bool IS_V, bool PAIRED = false>
__device__ __forceinline__ void encode_row(const EncodeArgs& a, const int row, const int h, const int j, float* rot_s, const RingArgs* ring = nullptr) {
    __shared__ __align__(16) float xh_s[IS_V ? D : 4];       // V: the normalised row, beside the raw one (a barrier less)
    __shared__ __align__(16) float xs[2 * D];     // (the row, then zeros: the compact rotation reads up to BGTQ_ROT_COL values past a segment's start)
    __shared__ float nrm[BGTQ_MAX_SEGMENTS];
    __shared__ float nrm_out[BGTQ_MAX_SEGMENTS];
    __shared__ uint8_t cds[D];
    __shared__ uint16_t xraw[D];
    __shared__ typename std::conditional<IS_V, StagedV, StagedK>::type sp;

    const bgtq_head_plan& P = a.plans[h];

    // ---- 0. one burst: plan tables, the raw row and its position, the rotation column ----
    if constexpr (IS_V) {
        if (j == 0) sp.v_bits = P.v_bits;
        if (j < 16) { sp.centroids[j] = P.v_centroids[j]; sp.boundaries[j] = P.v_boundaries[j]; }
    } else {
        if (j < 56) sp.hdr[j] = ((const int*)&P)[j];
#pragma unroll
        for (int i = 0; i < 4; i++)
            ((uint32_t*)sp.code_lut)[j + i * NT] = ((const uint32_t*)&P.code_lut[0][0])[j + i * NT];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int e = j + i * NT;                        // segment e / 32, level e % 32
            sp.centroids[e] = P.k_centroids[e >> 5][e & 31];
        }
    }
    xs[D + j] = 0.f;
    int b, s;
    split_row(row, a.S, b, s);
    uint16_t xr = 0;
    if (!ring) {
        xr = a.x[b * a.x_sb + h * a.x_sh + s * a.x_ss + j];
    } else {
        const int slot = ring->slot[b];
        if (slot >= 0 && slot < ring->W) {
            uint16_t* at = ring->buf + b * ring->b_sb + h * ring->b_sh + (int64_t)slot * ring->b_st + j;
            const uint16_t fresh = ring->in[b * ring->in_sb + h * ring->in_sh + j];
            xr = *at;
            *at = bgtq_in16(fresh, ring->bf16);
        }
    }
    const int t = (a.t_pos ? a.t_pos[b] : a.t_pos_scalar) + s;
    int4 k_dim = {0, 0, 0, 0};
    uint2 k_byte = {0u, 0u};
    float lut_off = 0.f, lut_scale = 0.f;                    // K: this dim's cell-search parameters
    if constexpr (!IS_V) {
        k_dim = *(const int4*)P.enc_dim[j];
        k_byte = *(const uint2*)P.enc_byte[a.layout == BGTQ_K_MIXED ? 1 : 0][j];
        lut_off = P.lut_offset[j];
        lut_scale = P.lut_inv_scale[j];
    } else if (j < D / 2) {
        k_byte = *(const uint2*)P.enc_vbyte[a.layout == BGTQ_V_NIBBLE ? 1 : 0][j];
    }
    // Latency bound.  K: the whole rotation matrix is requested now, before anything else is known (which
    // rows a thread needs is only known once the plan is in LDS), 16 bytes a lane and contiguous across
    // the wave (32 loads a thread), and parked in LDS (rot_s) ahead of the rotation, which then reads its
    // column from there.  Where no rotated segment is longer than BGTQ_ROT_COL dims, the plan also holds
    // every dim's rotation column cut down to its segment, which goes straight into registers (12 wide
    // loads instead of 32 and no trip through LDS).
    // V's rotation is dense and is needed later than its row: its column comes straight into registers
    // (the plan holds v_rot_T four rows interleaved: 16-byte loads, contiguous across the threads).
    constexpr int RC = BGTQ_ROT_COL;
    rot_piece rst[IS_V ? 1 : D / 4];
    float rc[IS_V ? D : RC];
    bool compact = false;
    if constexpr (IS_V) {
#pragma unroll
        for (int i = 0; i < D / 4; i++) {
            const float4 v = *(const float4*)P.v_rot_T4[i][j];
            rc[4 * i] = v.x; rc[4 * i + 1] = v.y; rc[4 * i + 2] = v.z; rc[4 * i + 3] = v.w;
        }
    } else {
        compact = P.rot_compact[0] != 0;                     // (uniform)
        if (compact) {
#pragma unroll
            for (int i = 0; i < RC / 4; i++) {
                const float4 v = *(const float4*)&P.k_rot_cols[j][4 * i];
                rc[4 * i] = v.x; rc[4 * i + 1] = v.y; rc[4 * i + 2] = v.z; rc[4 * i + 3] = v.w;
            }
        } else {
            fetch_rotation(P.k_rot_T, j, rst);
        }
    }
    if constexpr (!IS_V || PAIRED) __syncthreads();     // (K reads the staged header next; V's staged tables are first read two barriers on)

    // ---- per-thread static data, read ready-made from the plan (requested in the first burst) ----
    int n_seg = 1, g = 0, gs = 0, ge = D, ident = 0, src_dim = j;
    if constexpr (!IS_V) {
        n_seg = sp.hdr[H_NSEG];
        g = k_dim.x;
        gs = k_dim.y;
        ge = k_dim.z;
        ident = k_dim.w & 0xFF;
        src_dim = k_dim.w >> 8;
    }
    // output byte j: 0: zero fill, 1: bit stream, 2: raw byte copy
    const int mode = (int)(k_byte.x & 3u);
    const int bw = (int)((k_byte.x >> 2) & 15u);
    const StreamSlot slot{0, (int)(k_byte.x >> 8), (int)((k_byte.x >> 6) & 3u)};
    const int c0 = (int)k_byte.y;                       // (the slot's first code is folded into the base)

    // ---- 1. the row to LDS, gathered by head_perm (K) -------------
    if constexpr (IS_V) {              // (no gather: a thread converts its own value)
        xs[j] = bgtq_h2f(bgtq_in16(xr, a.bf16));
        if constexpr (PAIRED) __syncthreads();
    } else {
        xraw[j] = bgtq_in16(xr, a.bf16);
        __syncthreads();
        xs[j] = bgtq_h2f(xraw[src_dim]);
    }
    __syncthreads();

    // ---- 2. group norms: thread gg runs one sequential chain; V alone: every thread the same one, so that none waits for it.
    // (With the reads ahead, two barriers and a trip through LDS less, 4 rows x 2 heads of 8k tokens take 155.3 -> 153.3 us a
    // pass of eight layers, one row x 8 heads of 4k 67.3 -> 66.6 of four.)
    float v_norm = 0.f;
    if constexpr (IS_V && !PAIRED) {
        v_norm = __builtin_sqrtf(chain_sumsq_row<true>(xs) + 1e-30f);
    } else if (j < BGTQ_MAX_SEGMENTS) {
        float n = 0.f;
        if (j < n_seg) {
            float ss = 0.f;
            if constexpr (IS_V) {
                ss = chain_sumsq_row<false>(xs);
            } else {                           // short ranges: the batches would mostly run masked
                const int k0 = sp.hdr[H_START + j], k1 = k0 + sp.hdr[H_LEN + j];
#pragma unroll 8
                for (int k = k0; k < k1; k++) ss = __builtin_fmaf(xs[k], xs[k], ss);
            }
            n = __builtin_sqrtf(ss + 1e-30f);
        }
        nrm[j] = n;
    }
    if constexpr (!IS_V || PAIRED) __syncthreads();       // (V alone goes on with its own sum)

    // ---- 3. normalise -------------------------------------------------------
    float xh = 0.f;
    if (g >= 0) {
        const float n = IS_V && !PAIRED ? v_norm : nrm[g];
        const float safe = (n > (IS_V ? 1e-8f : 1e-10f)) ? n : 1.0f;
        xh = xs[j] / safe;
    }
    if constexpr (IS_V) xh_s[j] = xh;
    else xs[j] = xh;          // only this thread ever touched xs[j] since the barrier
    if constexpr (!IS_V) { if (!compact) park_rotation(rot_s, j, rst); }
    __syncthreads();

    // ---- 4. rotate ------------------------------------------------------------
    // The chain of the contract above; the values of a batch are read from LDS ahead of the products
    // that consume them.
    float y = 0.f;
    if (ident || g < 0) {
        y = xh;
    } else if constexpr (IS_V) {
        constexpr int CB = 32;
        float4 xv[2][CB / 4];
        auto load = [&](const int blk) {
#pragma unroll
            for (int i = 0; i < CB / 4; i++) xv[blk & 1][i] = *(const float4*)&xh_s[blk * CB + 4 * i];
        };
        load(0);
#pragma unroll
        for (int blk = 0; blk < D / CB; blk++) {
            if (blk + 1 < D / CB) load(blk + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < CB / 4; i++) {
                const float4 x4 = xv[blk & 1][i];
                const int k = blk * CB + 4 * i;
                y = __builtin_fmaf(x4.x, rc[k], y);
                y = __builtin_fmaf(x4.y, rc[k + 1], y);
                y = __builtin_fmaf(x4.z, rc[k + 2], y);
                y = __builtin_fmaf(x4.w, rc[k + 3], y);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    } else if (compact) {
        // The column is in registers and is zero past the segment's end, so the chain runs over
        // BGTQ_ROT_COL terms for every dim without a length test: a term x * 0 leaves the sum as it
        // is (the row is followed by zeros, so every x read is finite).
        constexpr int CB = 16;
        float xv[2][CB];
        auto load = [&](const int blk) {
#pragma unroll
            for (int i = 0; i < CB; i++) xv[blk & 1][i] = xs[gs + blk * CB + i];
        };
        load(0);
#pragma unroll
        for (int blk = 0; blk < RC / CB; blk++) {
            if (blk + 1 < RC / CB) load(blk + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < CB; i++) y = __builtin_fmaf(xv[blk & 1][i], rc[blk * CB + i], y);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {                                    // column j of the parked rotation
        constexpr int CB = 16;
        for (int k0 = gs; k0 < ge; k0 += CB) {
            float rk[CB], xv[CB];
#pragma unroll
            for (int i = 0; i < CB; i++) {
                const int k = min(k0 + i, ge - 1);
                rk[i] = rot_s[k * D + j];
                xv[i] = xs[k];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < CB; i++)
                if (k0 + i < ge) y = __builtin_fmaf(xv[i], rk[i], y);
        }
    }

    // ---- 5. scalar quantise ---------------------------------------------------
    const bool need_cent = IS_V || a.layout == BGTQ_K_MIXED || a.corrected;
    int code = 0;
    if constexpr (IS_V) {
        // (all 15 slots are read at once; those past the codebook's last boundary are skipped)
        const int nb = (1 << sp.v_bits) - 1;
        float bd[15];
#pragma unroll
        for (int i = 0; i < 15; i++) bd[i] = sp.boundaries[i];
#pragma unroll
        for (int i = 0; i < 15; i++) code += (i < nb && y > bd[i]) ? 1 : 0;
    } else if (g >= 0) {
        if (a.quant_mode == BGTQ_QUANT_EXACT) {
            const int nb = (1 << sp.hdr[H_BW + g]) - 1;
            for (int i = 0; i < nb; i++) code += (P.k_boundaries[g][i] < y) ? 1 : 0;
        } else {
            float c = (y - lut_off) * lut_scale;
            c = fminf(fmaxf(c, 0.0f), (float)(BGTQ_LUT_BINS - 1));
            code = sp.code_lut[g * BGTQ_LUT_BINS + (int)c];
        }
    }
    cds[j] = (uint8_t)code;
    // centroid of the chosen code for the norm correction below; it is parked in xs
    // after the barrier (K: other threads may still be reading xs in their rotation)
    if (need_cent) {
        if constexpr (IS_V) y = sp.centroids[code];
        else y = g < 0 ? 0.f : code < 32 ? sp.centroids[g * 32 + code] : P.k_centroids[g][code];
    }
    // (V's last reads of xs were the norm's, ahead of the barrier before the rotation)
    if constexpr (!IS_V || PAIRED) __syncthreads();
    if (need_cent) xs[j] = y;
    __syncthreads();

    // ---- 6. norms to store (raw or divided by ||centroids[codes]||) ---------
    // The second wave's chain: the first one packs the record meanwhile (neither needs anything of the
    // other).
    const int gg = j - 64;
    const bool has_norm = gg >= 0 && gg < BGTQ_MAX_SEGMENTS;
    if (has_norm) {
        float out = 0.f;
        if (gg < n_seg) {
            const float n = IS_V && !PAIRED ? v_norm : nrm[gg];
            if constexpr (IS_V) {
                const float cn = __builtin_sqrtf(chain_sumsq_row<!PAIRED>(xs) + 1e-20f);
                out = n / (cn > 1e-10f ? cn : 1.0f);
            } else if (a.layout == BGTQ_K_MIXED || a.corrected) {
                const int k0 = sp.hdr[H_START + gg];
                out = n / fmaxf(__builtin_sqrtf(chain_sumsq_span(xs, k0, k0 + sp.hdr[H_LEN + gg])), 1e-10f);
            } else {
                out = n;
            }
        }
        nrm_out[gg] = out;
    }

    // ---- 7a. unpacked outputs (codes path) ------------------------------------
    if (a.codes_out) {                                  // (uniform)
        __syncthreads();
        a.codes_out[(int64_t)row * D + j] = cds[j];
        if (IS_V) {
            if (j == 0 && a.norms) a.norms[row] = bgtq_f2h(nrm_out[0]);
        } else if (a.norms_f32_out && j < BGTQ_MAX_SEGMENTS && j < a.norm_width) {
            a.norms_f32_out[(int64_t)row * a.norm_width + j] = nrm_out[j];
        }
        return;
    }
    if (t < 0 || t >= a.max_T) return;                  // a position outside the cache: the record is dropped

    // ---- 7b. cache norms, by the threads that made them ------------------------
    if (has_norm && gg < (IS_V ? 1 : a.norm_width))
        a.norms[b * a.n_sb + h * a.n_sh + (int64_t)t * a.n_st + gg] = bgtq_f2h(nrm_out[gg]);

    // ---- 8. pack: thread j produces output byte j ---------------
    if (j < a.row_width) {
        unsigned v = 0;
        if (mode == 1)      v = stream_byte_batched(&cds[c0], slot, bw);
        else if (mode == 2) v = cds[c0];
        a.packed[b * a.p_sb + h * a.p_sh + (int64_t)t * a.p_st + j] = (uint8_t)v;
    }
}

template <bool IS_V>
__global__ __launch_bounds__(NT) void encode_kernel(EncodeArgs a) {
    __shared__ __align__(16) float rot_s[IS_V ? 4 : D * D];
    encode_row<IS_V>(a, blockIdx.x, blockIdx.y, threadIdx.x, rot_s);
}
// ================================================================================================
// Prompt-sized encoder: blocks of 16 rows, rotations and V's corrected norms on the fp32 matrix cores, norms as chains of a lane.
//
// v_mfma_f32_16x16x4_f32 adds its four products to the accumulator one after the other, each as one fused
// multiply-add rounded to nearest with subnormals kept: such instructions over ascending k are the contract's
// fmaf chain bit for bit.  Terms outside a dim's own segment are x * 0 and leave its sum as it is (x finite; a
// block whose norms are not all finite takes scalar chains instead).
//
// A block stays in one wave from the raw rows to the codes: lane (li, lg) of 16 x 4 holds dims k = 4 kk + lg
// of row li in 32 registers, which is the A operand of step kk as it is.
//   norms    lane = row for V, (row, one of four groups) for K: chains of mixed multiply-adds on the raw fp16 values,
//            one instruction a dim (V in the diagonal of X X^T: 32 matrix instructions, 1024 clocks, here 128 of 2.5)
//   xhat     x / norm from the norm's rounded reciprocal, in registers (div_by below)
//   rotate   16 columns at a time against the rotation in LDS, stored in operand order (one 16-byte read a lane
//            feeds four steps, no bank conflicts); K takes only the steps its columns' segments reach
//   codes    four rows of one column per lane, straight from the accumulator
//   corrected norms  the centroids of the codes: V the diagonal of X X^T, K lane = (row, group): its chains of 16 dims with
//            a dependent code, centroid and product read each took 17 k of a block's 64 k clocks, these take 7 k
//   packing  a lane makes four bytes of a record: a byte is a dot product of four code bytes with powers of two
//
// CS waves share a block and split its columns, groups, rows to load and rows to pack.  CS 1 (many blocks): 16 waves
// share a rotation, each walks blocks of its own and no barrier is met on the way.  CS 2 (at most 8 blocks a
// work-group): as many waves a compute unit again where CS 1 would leave half of it empty.  CS 4 (few rows): a
// work-group of 4 waves a block, two of them a compute unit.
// CS 1 is bound by the matrix cores and vector issue in turn: an fp32 matrix instruction keeps its SIMD's vector unit busy
// for its whole 32 clocks (two waves, one of either kind: the sum of both times), and a V block has 288 of them.  65 536
// records each of K and V (4 x 8192 tokens, 2 heads, K3V3): 135 us as two launches of 16-row tiles on the vector units (there
// the dense V rotation alone is 55 us of FMA), 61 us in one with norms as diagonals, a compare and an add for every
// boundary of a V cell and quotients of two residual steps, 56 with what is here, 53 with the priorities below.  CS 2 and CS 4 are bound by one block's chain; 8 heads,
// nibble records, against groups one after the other in K's norms and CS 1 from 513 blocks on: 128 tokens 18.3 -> 13.1 us,
// 600 26.7 -> 18.2, 2001 30.4 -> 24.2, 9000 (CS 1) 89.6 -> 68.9; bit-packed records (no corrected K norms) 12.4 -> 11.4,
// 20.6 -> 15.8, 23.9 -> 21.8, 70.1 -> 61.3.
// ================================================================================================
constexpr int RROW = D * 2 + 16;        // bytes from one raw row to the next: rows 4 banks apart
constexpr int CROW = D + 8;             // bytes from one row of codes to the next (a byte's window of codes may reach 8 past the last)

struct TileArgs { EncodeArgs k, v; int k_groups, v_groups; };      // work-groups per head of each kind (0: none)

template <int CS>
struct EncodeLds {
    static constexpr int NW = CS == 4 ? 4 : 16;               // waves at most
    static constexpr int NB = NW / CS;                        // blocks at a time
    float rot[D / 4][D][4];             // the rotation, [step][column][k % 4]
    alignas(16) uint8_t raw[NB][16 * RROW];                   // raw rows [row][k % 4][k / 4] fp16, later the codes
    float2 nrm[NB][BGTQ_MAX_SEGMENTS][16];                    // (norm, its reciprocal) per group and row
    int64_t dst[NB][16], ndst[NB][16];  // a row's record and norm offsets, -1: dropped
    uint4 pack[D];                      // per record byte: first code, its bits (offset | width << 8), dot weights of the next ones
    float cent[BGTQ_MAX_SEGMENTS * 32];
    uint8_t lut[BGTQ_MAX_SEGMENTS * BGTQ_LUT_BINS];
    int hdr[56];
    float2 bin[D];                      // K cell search of a packed dim
    int8_t group[D];                    // its group, -1: a 0-bit dim
    alignas(16) uint16_t place[D];      // source dim -> byte offset in a raw row
};

// x / d correctly rounded from y = RN(1 / d), for x a finite fp16 value, and d and y normal (Markstein: a quotient within one
// unit in the last place and a correctly rounded reciprocal give the rounded quotient after one residual step.  x * y can be
// 1.5 units off, but no quotient of an 11-bit x lies near enough to a midpoint: tests/test_quotient.py compares all 2^10 x 2^23
// mantissas.)
__device__ __forceinline__ float div_by(float x, float2 dy) {
    const float q = x * dy.y;
    return __builtin_fmaf(__builtin_fmaf(-dy.x, q, x), dy.y, q);
}

template <int CS, bool IS_V>
__device__ __forceinline__ void encode_blocks(const EncodeArgs& a, const int h, const int first, const int stride, EncodeLds<CS>& L) {
    const int NW = CS == 4 ? 4 : (int)blockDim.x >> 6, NTHR = NW * 64, NB = NW / CS;       // (at least 4 waves)
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const bgtq_head_plan& P = a.plans[h];
    const int64_t N = (int64_t)a.B * a.S;
    const int n_blocks = (int)((N + 15) / 16);
    const bool need_cent = IS_V || a.layout == BGTQ_K_MIXED || a.corrected;

    // ---- once per work-group: tables and the rotation (64 KB, straight from the plan into LDS).  Everything is
    // requested in one burst: every thread loads, the ones past a table's end its last words, and stores behind all loads (a
    // load inside `if (tid < ..)` is waited for there, and K's tables were six round trips one after the other: 19.3 -> 18.6 us for
    // 8 heads of 2001 tokens)
    constexpr int RT = CS == 4 ? 4 : 1;                       // K: 4 x 4 pieces of the rotation in flight a thread
    float4 rot4[RT][4];
    auto fetch_rot = [&](int at) {                            // (k_rot_T is zero outside a column's own segment)
#pragma unroll
        for (int n = 0; n < RT; n++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int piece = min(at + n * NTHR, D * D / 16 - 1);        // rows 4 (piece / 32) .., columns 4 (piece % 32) ..
                rot4[n][r] = *(const float4*)&P.k_rot_T[((piece >> 5) * 4 + r) * D + (piece & 31) * 4];
            }
    };
    if constexpr (IS_V) {                                     // (the plan holds it in this order)
        const uint32_t dst = (uint32_t)(uintptr_t)(lds_ptr_t)(uint8_t*)&L.rot[0][0][0];
        const uint8_t* src = (const uint8_t*)&P.v_rot_T4[0][0][0];
        for (int c = wave * 4; c < 64; c += NW * 4) dma_full<4>((uint32_t)lane * 16, uniform_ptr(src + c * 1024), dst + c * 1024);
    } else {
        fetch_rot(tid);
    }
    // ---- CS waves a block: the block's place in the work-group, this wave's part of it
    const int slot = CS == 1 ? wave : wave / CS, part = CS == 1 ? 0 : wave % CS;
    const bool wide = ((a.x_sb | a.x_sh | a.x_ss) & 7) == 0 && ((uintptr_t)a.x & 15) == 0;
    // (batch row, step) of row r of the block whose first row is step s0 of batch row b0
    auto row_of = [&](int b0, int s0, int r, int& b, int& s) {
        b = b0;
        s = s0 + r;
        if (s >= a.S) { const unsigned q = (unsigned)s / (unsigned)a.S; b += (int)q; s -= (int)q * a.S; }
    };
    // Raw rows, 16 lanes a row, 8 values each.  AHEAD: with the tables (8 heads of 128 tokens 14.0 -> 11.5 us, of 2001
    // 17.5 -> 16.4; with a wave a block V's waves came to the matrix core together and the registers spilled: 31.4 -> 35.3)
    constexpr int PASS = 4 / CS;
    constexpr bool AHEAD = CS > 1;
    uint4 x4[PASS];
    auto fetch_rows = [&](int blk) {
        const unsigned n0 = (unsigned)blk * 16u;
        const int b0 = (int)(n0 / (unsigned)a.S), s0 = (int)(n0 - (unsigned)b0 * (unsigned)a.S);
#pragma unroll
        for (int p = 0; p < PASS; p++) {
            const int r = 4 * (part * PASS + p) + (lane >> 4);
            x4[p] = uint4{0, 0, 0, 0};
            if ((int64_t)n0 + r < N) {
                int b, s;
                row_of(b0, s0, r, b, s);
                const uint16_t* src = a.x + b * a.x_sb + h * a.x_sh + s * a.x_ss + (lane & 15) * 8;
                if (wide) x4[p] = *(const uint4*)src;
                else {
                    uint32_t w[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) w[i] = (uint32_t)src[2 * i] | ((uint32_t)src[2 * i + 1] << 16);
                    x4[p] = uint4{w[0], w[1], w[2], w[3]};
                }
            }
        }
    };
    if (AHEAD) fetch_rows(first * NB + slot);
    int n_seg = 1, v_bits = 0, n_zero = 0;
    float bd[15];                                             // V boundaries (+inf past the last)
    uint2 byte_of = {0u, 0u};
    uint32_t seg_of[4] = {0, 0, 0, 0};                        // group of dim 4 kk + lg, 4 bits each
    const int td = tid & (D - 1);
    if constexpr (IS_V) {
        v_bits = P.v_bits;
#pragma unroll
        for (int b = 0; b < 15; b++) bd[b] = P.v_boundaries[b];
        const float cent = P.v_centroids[tid & 15];
        byte_of = *(const uint2*)P.enc_vbyte[a.layout == BGTQ_V_NIBBLE ? 1 : 0][tid & (D / 2 - 1)];
        if (tid < 16) L.cent[tid] = cent;
        if (tid >= D / 2) byte_of = uint2{0u, 0u};
        if (tid < D) L.place[tid] = (uint16_t)(((tid & 3) * (D / 4) + (tid >> 2)) * 2);
    } else {
        n_seg = P.n_seg;
        n_zero = P.n_zero_dims;
        constexpr int LUT_WORDS = BGTQ_MAX_SEGMENTS * BGTQ_LUT_BINS / 4, N_CENT = BGTQ_MAX_SEGMENTS * 32;
        static_assert(N_CENT <= 256 && LUT_WORDS <= 512, "at least 256 threads, two words of the cell tables each");
        const uint4 segs = ((const uint4*)((const uint8_t*)P.lut_image[BGTQ_K_BITPACKED] + BGTQ_LUT_KSEG))[lg];
        const int hdr = ((const int*)&P)[min(tid, 55)];
        const uint32_t* cells = (const uint32_t*)&P.code_lut[0][0];
        const uint32_t cell0 = cells[min(tid, LUT_WORDS - 1)], cell1 = cells[min(tid + NTHR, LUT_WORDS - 1)];
        const float cent = (&P.k_centroids[0][0])[(min(tid, N_CENT - 1) >> 5) * (int)(sizeof(P.k_centroids[0]) / sizeof(float)) + (tid & 31)];
        const int4 dim = *(const int4*)P.enc_dim[td];
        const float2 bin = {P.lut_offset[td], P.lut_inv_scale[td]};
        byte_of = *(const uint2*)P.enc_byte[a.layout == BGTQ_K_MIXED ? 1 : 0][td];
        seg_of[0] = segs.x; seg_of[1] = segs.y; seg_of[2] = segs.z; seg_of[3] = segs.w;
        if (tid < 56) L.hdr[tid] = hdr;
        if (tid < LUT_WORDS) ((uint32_t*)L.lut)[tid] = cell0;
        if (tid + NTHR < LUT_WORDS) ((uint32_t*)L.lut)[tid + NTHR] = cell1;
        if (tid < N_CENT) L.cent[tid] = cent;
        if (tid < D) {                                        // packed dim k lies at [k % 4][k / 4] of a raw row
            L.group[tid] = (int8_t)dim.x;
            L.place[dim.w >> 8] = (uint16_t)(((tid & 3) * (D / 4) + (tid >> 2)) * 2);
            L.bin[tid] = bin;
        }
        // The rotation, four rows interleaved on the way (as 256 loads of 16 columns of a row into LDS 0.4 us more).  A thread's
        // columns leave in an order of its own, from column (tid / 4) % 4 of the four on: 16 lanes then write 256 bytes of 64
        // banks.
        for (int at = tid;;) {
#pragma unroll
            for (int n = 0; n < RT; n++) {
                const int piece = at + n * NTHR, turn = (piece >> 2) & 3;
                if (piece >= D * D / 16) continue;
                float x[4][4];                                // [row][columns from `turn` on]
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float c[4] = {rot4[n][r].x, rot4[n][r].y, rot4[n][r].z, rot4[n][r].w};
                    float half[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) half[i] = turn & 2 ? c[(i + 2) & 3] : c[i];
#pragma unroll
                    for (int i = 0; i < 4; i++) x[r][i] = turn & 1 ? half[(i + 1) & 3] : half[i];
                }
#pragma unroll
                for (int i = 0; i < 4; i++)
                    *(float4v*)L.rot[piece >> 5][(piece & 31) * 4 + ((i + turn) & 3)] = (float4v){x[0][i], x[1][i], x[2][i], x[3][i]};
            }
            at += RT * NTHR;
            if (at - tid >= D * D / 16) break;                // (uniform)
            fetch_rot(at);
        }
    }
    const int lpr = a.row_width > 64 ? 32 : 16;               // packing: lanes per row, lane = record dword dw
    const int dw = lane & (lpr - 1);
    const bool dwords = ((a.row_width | a.p_st | a.p_sb | a.p_sh) & 3) == 0 && ((uintptr_t)a.packed & 3) == 0;
    if (tid < D) {
        // byte = (code 0 >> skip) + sum over the next codes of code << (its position in the byte)
        const uint2 e = a.packed && tid < a.row_width ? byte_of : uint2{0u, 0u};
        const int mode = (int)(e.x & 3u), bw = (int)((e.x >> 2) & 15u), skip = (int)((e.x >> 6) & 3u), n = (int)(e.x >> 8);
        uint4 p = {e.y, 0u, 0u, 0u};
        if (mode == 2 || (mode == 1 && n > 0)) p.y = (uint32_t)skip | ((8u - skip) << 8);
#pragma unroll
        for (int c = 1; c < 8; c++) {
            const uint32_t w = mode == 1 && c < n ? 1u << ((c * bw - skip) & 31) : 0u;
            if (c < 4) p.z |= w << (8 * c);
            else p.w |= (w >> 4) << (8 * (c - 4));            // (1-bit codes only: the second four make a nibble of their own)
        }
        L.pack[tid] = p;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // this wave's share of the rotation
    __syncthreads();
    // (a stream of 1-bit codes; groups are in ascending width)
    const bool two_dots = IS_V ? v_bits == 1 && a.layout == BGTQ_V_BITPACKED : L.hdr[H_BW] == 1 && a.layout == BGTQ_K_BITPACKED;

    uint8_t* raw = L.raw[slot];
    auto meet = [&]() {
        asm volatile("" ::: "memory");
        if (CS > 1) __syncthreads();
        else __builtin_amdgcn_wave_barrier();                 // (a wave's LDS accesses keep their order)
        asm volatile("" ::: "memory");
    };
    // (neighbouring blocks to the waves of one work-group; CS > 1: launch_blocks() has a place for every block, so there is
    // one round, with the rows fetched above, and every wave of it goes for the barriers' sake: rows past the last are zeros and
    // stored nowhere.  Told so by a `break` at the end the compiler has K of 2001 tokens x 8 heads take 58 us for 16)
    for (int round = first * NB; CS == 1 ? round + slot < n_blocks : round < n_blocks; round += stride * NB) {
        const int blk = round + slot;
        // The oldest wave of a SIMD would run ahead, and the youngest end alone with a matrix core that it fills by half
        // (56 -> 53 us at 65 536 records): waves that are behind go first, by blocks left and by halves of a block.
        const bool more = round + stride * NB + slot < n_blocks;
        if (CS == 1) { if (more) __builtin_amdgcn_s_setprio(3); else __builtin_amdgcn_s_setprio(1); }
        const unsigned n0 = (unsigned)blk * 16u;
        const int b0 = (int)(n0 / (unsigned)a.S), s0 = (int)(n0 - (unsigned)b0 * (unsigned)a.S);
        // ---- raw rows to LDS
        if (!AHEAD) fetch_rows(blk);
        {
            const int rc = lane & 15;
            const uint4 at = *(const uint4*)&L.place[rc * 8];
            const uint32_t at2[4] = {at.x, at.y, at.z, at.w};
            if (lane < 16 && part == 0) {                     // where the rows go
                int64_t dst = -1, nd = -1;
                if ((int64_t)n0 + lane < N) {
                    int b, s;
                    row_of(b0, s0, lane, b, s);
                    const int64_t t = (int64_t)(a.t_pos ? a.t_pos[b] : a.t_pos_scalar) + s;
                    if (a.codes_out) dst = nd = (int64_t)n0 + lane;
                    else if (t >= 0 && t < a.max_T) {
                        dst = b * a.p_sb + h * a.p_sh + t * a.p_st;
                        nd = b * a.n_sb + h * a.n_sh + t * a.n_st;
                    }
                }
                L.dst[slot][lane] = dst;
                L.ndst[slot][lane] = nd;
            }
#pragma unroll
            for (int p = 0; p < PASS; p++) {
                uint8_t* row = raw + (4 * (part * PASS + p) + (lane >> 4)) * RROW;
                uint32_t w[4] = {x4[p].x, x4[p].y, x4[p].z, x4[p].w};
                if (a.bf16) {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        w[i] = (uint32_t)bgtq_in16((uint16_t)w[i], 1) | ((uint32_t)bgtq_in16((uint16_t)(w[i] >> 16), 1) << 16);
                }
                if constexpr (IS_V) {                         // dims 8 rc + g and 8 rc + 4 + g are neighbours
#pragma unroll
                    for (int g = 0; g < 4; g++)
                        *(uint32_t*)(row + g * (D / 2) + rc * 4) =
                            __builtin_amdgcn_perm(w[2 + (g >> 1)], w[g >> 1], g & 1 ? 0x07060302u : 0x05040100u);
                } else {
#pragma unroll
                    for (int i = 0; i < 8; i++)
                        *(uint16_t*)(row + ((at2[i >> 1] >> (16 * (i & 1))) & 0xFFFFu)) = (uint16_t)(w[i >> 1] >> (16 * (i & 1)));
                }
            }
        }
        meet();
        // ---- A operands (K reads them once its norms are known)
        const uint8_t* arow = raw + li * RROW + lg * (D / 2);
        float A[D / 4];
        auto load_a = [&](int q) {                            // dims 32 q + 4 i + lg
            const half8 v = *(const half8*)(arow + 16 * q);
#pragma unroll
            for (int i = 0; i < 8; i++) A[8 * q + i] = (float)v[i];
        };
        // ---- norms
        bool finite = true;
        const bool diag = (li >> 2) == lg;                    // lane (li, lg) holds (row 4 lg + r, row li) of X X^T in register r
        auto diagonal = [&](const float4v& sum) { return li & 2 ? (li & 1 ? sum[3] : sum[2]) : (li & 1 ? sum[1] : sum[0]); };
        float2 v_nrm = {0.f, 0.f};                            // V: of row li
        if constexpr (IS_V) {
            float sum = 0.f;
#pragma unroll
            for (int q = 0; q < D / 32; q++) {
                half8 v[4];
#pragma unroll
                for (int c = 0; c < 4; c++) v[c] = *(const half8*)(raw + li * RROW + c * (D / 2) + 16 * q);
#pragma unroll
                for (int i = 0; i < 8; i++)
#pragma unroll
                    for (int c = 0; c < 4; c++) sum = __builtin_fmaf((float)v[c][i], (float)v[c][i], sum);
                __builtin_amdgcn_sched_barrier(0);
            }
            const float n = __builtin_sqrtf(sum + 1e-30f);
            v_nrm = float2{n, 1.0f / n};
        } else {
            // lane = (row li, group 4 p + lg): 64 chains side by side, over the blocks of 16 dims that the group touches
            for (int p = part; 4 * p < n_seg; p += CS) {
                const int g = 4 * p + lg, s = g < n_seg ? L.hdr[H_START + g] : 0, e = g < n_seg ? s + L.hdr[H_LEN + g] : 0;
                const uint8_t* at = raw + li * RROW + (s >> 4) * 8;
                int lo = s & 15, hi = e - (s & ~15);          // the group's dims, from this block's first one on
                float sum = 0.f;
                uint2 w[4];                                   // dims c, c + 4, c + 8, c + 12 of the block
                auto fetch = [&]() {                          // (reads past the group stay inside the work-group's rows: masked below)
#pragma unroll
                    for (int c = 0; c < 4; c++) w[c] = *(const uint2*)(at + c * (D / 2));
                };
                fetch();
                while (__builtin_amdgcn_ballot_w64(hi > 0) != 0) {
                    uint2 v[4];
#pragma unroll
                    for (int c = 0; c < 4; c++) v[c] = w[c];
                    at += 8;
                    fetch();
                    const uint32_t live = hi > 0 ? (0xFFFFu >> (16 - min(hi, 16))) & (0xFFFFu << lo) : 0u;
                    // (dims of other groups become zeros, two at a time)
                    auto dim_bits = [&](int i) { return (uint32_t)((int32_t)(live << (31 - i)) >> 31); };
                    if (__builtin_amdgcn_ballot_w64(live != 0xFFFFu) != 0) {          // (uniform)
#pragma unroll
                        for (int c = 0; c < 4; c++) {
                            v[c].x &= __builtin_amdgcn_perm(dim_bits(c + 4), dim_bits(c), 0x05040100u);
                            v[c].y &= __builtin_amdgcn_perm(dim_bits(c + 12), dim_bits(c + 8), 0x05040100u);
                        }
                    }
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const half2v d = __builtin_bit_cast(half2v, i & 8 ? v[i & 3].y : v[i & 3].x);
                        const float x = (float)d[(i >> 2) & 1];
                        sum = __builtin_fmaf(x, x, sum);
                    }
                    lo = 0;
                    hi -= 16;
                }
                if (g < n_seg) {
                    const float n = __builtin_sqrtf(sum + 1e-30f);
                    finite = finite && n < INFINITY;
                    L.nrm[slot][g][li] = float2{n, 1.0f / n};
                }
            }
        }
        bool scalar_chain = !IS_V && __builtin_amdgcn_ballot_w64(!finite) != 0;           // (uniform)
        if (CS == 1 || IS_V) asm volatile("" ::: "memory");
        else scalar_chain = __syncthreads_or(scalar_chain) != 0;
        // ---- xhat.  (The contract divides by 1 where the norm is at most 1e-10, for V 1e-8: a non-zero fp16 value alone
        // makes it 6e-8, so those norms belong to rows of zeros, which stay zeros whatever they are divided by.  An
        // infinite or NaN norm of V makes every value of its row NaN, as the dense rotation would.)
        if constexpr (IS_V) {
#pragma unroll
            for (int q = 0; q < D / 32; q++) {
                load_a(q);
#pragma unroll
                for (int i = 0; i < 8; i++) A[8 * q + i] = div_by(A[8 * q + i], v_nrm);
            }
        } else {
#pragma unroll
            for (int q = 0; q < D / 32; q++) {
                load_a(q);
                // (addresses and masks that are the same for every block would be worked out ahead of the loop and spilled: with two
                // waves a block 166 moves of masks to lanes and back and 43 scratch accesses in the kernel, 42 and 2 this way;
                // 18.4 -> 17.5 us for K of 8 heads of 2001 tokens)
                uint32_t segs = seg_of[q];
                asm volatile("" : "+v"(segs));
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const int kk = 8 * q + i;
                    A[kk] = div_by(A[kk], L.nrm[slot][(segs >> (4 * i)) & 15u][li]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (n_zero) {                                     // (uniform) 0-bit dims come first
                int zeros = n_zero - lg;
                asm volatile("" : "+v"(zeros));
#pragma unroll
                for (int kk = 0; kk < D / 4; kk++) A[kk] = 4 * kk < zeros ? 0.f : A[kk];
            }
        }
        // codes of rows 4 lg .. + 3 from the values of column j
        auto quantise = [&](const float4v& y, int j, int g) -> uint32_t {
            uint32_t code[4] = {0, 0, 0, 0};
            if (a.quant_mode == BGTQ_QUANT_EXACT) {
                const int nb = g >= 0 ? (1 << L.hdr[H_BW + g]) - 1 : 0;
#pragma unroll 1
                for (int b = 0; b < nb; b++)
#pragma unroll
                    for (int r = 0; r < 4; r++) code[r] += P.k_boundaries[g][b] < y[r] ? 1u : 0u;
            } else {
                const float off = L.bin[j].x, scale = L.bin[j].y;
                const uint8_t* lut = &L.lut[max(g, 0) * BGTQ_LUT_BINS];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float t = (y[r] - off) * scale;
                    t = fminf(fmaxf(t, 0.0f), (float)(BGTQ_LUT_BINS - 1));
                    code[r] = lut[(int)t];
                }
                if (n_zero) {                                 // (uniform)
#pragma unroll
                    for (int r = 0; r < 4; r++) code[r] = g < 0 ? 0u : code[r];
                }
            }
            return code[0] | (code[1] << 8) | (code[2] << 16) | (code[3] << 24);
        };
        uint32_t odd_codes[D / 16 / CS];                      // of a block with infinities or NaNs: scalar chains over the raw rows
        if (!IS_V && scalar_chain) {
#pragma unroll 1
            for (int c = 0; c < D / 16 / CS; c++) {
                const int j = 16 * (part * (D / 16 / CS) + c) + li;
                const int4 dim = *(const int4*)P.enc_dim[j];
                float4v y = {0, 0, 0, 0};
#pragma unroll 1
                for (int r = 0; r < 4; r++) {
                    const int row = 4 * lg + r;
                    const float n = L.nrm[slot][max(dim.x, 0)][row].x, safe = n > 1e-10f ? n : 1.0f;
                    float t = 0.f;
                    for (int k = dim.w & 0xFF ? j : dim.y; dim.x >= 0 && k < (dim.w & 0xFF ? j + 1 : dim.z); k++) {
                        const float x = bgtq_h2f(*(const uint16_t*)(raw + row * RROW + ((k & 3) * (D / 4) + (k >> 2)) * 2)) / safe;
                        t = dim.w & 0xFF ? x : __builtin_fmaf(x, P.k_rot_T[k * D + j], t);
                    }
                    y[r] = t;
                }
                odd_codes[c] = quantise(y, j, dim.x);
            }
        }
        // ---- rotate and quantise 16 columns at a time; codes of rows 4 lg .. + 3, column 16 cb + li
        uint32_t codes[D / 16 / CS];
        // V: the cell search of 16 columns (the number of boundaries below a value) goes under the next 16 columns' products:
        // behind its own, all waves of a SIMD would come to it together and leave the matrix core alone.  3 compares, 4 selects
        // and 3 additions with carry for a value of 3 bits (7 and 7 before).  Operands are read eight steps ahead.
        auto columns = [&](auto bits) {
            constexpr int BITS = decltype(bits)::value, NC = D / 16 / CS;
            const float* rot = &L.rot[0][16 * part * NC + li][lg];
            float R[2][8];
            auto fetch = [&](int at) {                        // eight steps: columns at / 4, steps 8 (at % 4) ..
#pragma unroll
                for (int i = 0; i < 8; i++) R[at & 1][i] = rot[(at >> 2) * 64 + (8 * (at & 3) + i) * 4 * D];
            };
            fetch(0);
            // number of boundaries below x, its bits from the highest down, under the bits of `below`
            auto search = [&](float x, uint32_t below) {
                float cand[(1 << BITS) - 1];                  // in-order: the boundaries still in question
#pragma unroll
                for (int b = 0; b < (1 << BITS) - 1; b++) cand[b] = bd[b];
#pragma unroll
                for (int n = (1 << BITS) - 1; n >= 1; n >>= 1) {
                    const bool up = x > cand[n >> 1];
                    const uint64_t carry = __builtin_amdgcn_ballot_w64(up);
                    asm("v_addc_co_u32 %0, vcc, %1, %1, %2" : "=v"(below) : "v"(below), "s"(carry) : "vcc");
#pragma unroll
                    for (int b = 0; b < n >> 1; b++) cand[b] = up ? cand[b + (n >> 1) + 1] : cand[b];
                }
                return below;
            };
            float4v y = {0, 0, 0, 0}, before = {0, 0, 0, 0};
            uint32_t cell = 0;
#pragma unroll
            for (int at = 0; at < 4 * NC; at++) {
                if (at + 1 < 4 * NC) fetch(at + 1);
                if ((at & 3) == 0) {
                    before = y;
                    y = (float4v){0, 0, 0, 0};
                }
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const int kk = 8 * (at & 3) + i;
                    y = __builtin_amdgcn_mfma_f32_16x16x4f32(A[kk], R[at & 1][i], y, 0, 0, 0);
                    if (at >= 4 && i == 0) cell = search(before[3 - (at & 3)], cell << (8 - BITS));
                }
                if (at >= 4 && (at & 3) == 3) codes[(at >> 2) - 1] = cell;
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int r = 3; r >= 0; r--) cell = search(y[r], cell << (8 - BITS));
            codes[NC - 1] = cell;
        };
        if constexpr (IS_V) {
            if (v_bits == 3) columns(std::integral_constant<int, 3>{});         // (uniform)
            else if (v_bits == 4) columns(std::integral_constant<int, 4>{});
            else if (v_bits == 2) columns(std::integral_constant<int, 2>{});
            else columns(std::integral_constant<int, 1>{});
        } else {
#pragma unroll
            for (int c = 0; c < D / 16 / CS; c++) {
                const int cb = part * (D / 16 / CS) + c;
                const int j = 16 * cb + li;
                float4v y = {0, 0, 0, 0};
                const float* rot = &L.rot[0][j][lg];          // + step * 4 D: two steps a read
                const int g = L.group[j];
                if (scalar_chain) {
                    codes[c] = odd_codes[c];
                    continue;
                }
                const uint32_t span = ((const uint32_t*)P.rot_span)[cb >> 2] >> ((cb & 3) * 8);
                const int q_lo = (int)(span & 15u), q_hi = (int)((span >> 4) & 15u);
#pragma unroll
                for (int q = 0; q < D / 16; q++)
                    if (q >= q_lo && q < q_hi) {              // (uniform)
#pragma unroll
                        for (int i = 0; i < 4; i++) y = __builtin_amdgcn_mfma_f32_16x16x4f32(A[4 * q + i], rot[(4 * q + i) * 4 * D], y, 0, 0, 0);
                    }
                codes[c] = quantise(y, j, g);
                __builtin_amdgcn_sched_barrier(0);            // (operands of later columns would be read ahead and spill)
            }
        }
        meet();                                               // (the raw rows are read)
#pragma unroll
        for (int c = 0; c < D / 16 / CS; c++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                raw[(4 * lg + r) * CROW + 16 * (part * (D / 16 / CS) + c) + li] = (uint8_t)(codes[c] >> (8 * r));
        meet();
        if (CS == 1) { if (more) __builtin_amdgcn_s_setprio(2); else __builtin_amdgcn_s_setprio(0); }
        // ---- norms to store
        auto store_norm = [&](int g, int row, float out) {
            const int64_t nd = L.ndst[slot][row];
            if (nd < 0) return;
            if (a.codes_out && !IS_V) { if (a.norms_f32_out && g < a.norm_width) a.norms_f32_out[nd * a.norm_width + g] = out; }
            else if (g < (IS_V ? 1 : a.norm_width) && a.norms) a.norms[nd + g] = bgtq_f2h(out);
        };
        if (part == 0 || (!IS_V && need_cent)) {
            if (need_cent) {
                if constexpr (IS_V) {                         // the centroids of all codes in two bursts
                    float4v sum = {0, 0, 0, 0};
#pragma unroll
                    for (int half = 0; half < 2; half++) {
                        float cen[D / 8];
#pragma unroll
                        for (int q = 0; q < D / 32; q++) {
                            const uint32_t* cw = (const uint32_t*)&raw[li * CROW + 64 * half + 16 * q];
#pragma unroll
                            for (int i = 0; i < 4; i++) cen[4 * q + i] = L.cent[(cw[i] >> (8 * lg)) & 15u];
                        }
#pragma unroll
                        for (int i = 0; i < D / 8; i++) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(cen[i], cen[i], sum, 0, 0, 0);
                    }
                    const float cn = __builtin_sqrtf(diagonal(sum) + 1e-20f);
                    if (diag) store_norm(0, li, v_nrm.x / (cn > 1e-10f ? cn : 1.0f));
                }
                if constexpr (!IS_V) {                        // the centroids' chains, lane = (row, group) as above
#pragma unroll 1
                    for (int p = part; p < 2; p += CS) {
                        const int g = 4 * p + lg, s = g < n_seg ? L.hdr[H_START + g] : 0, len = g < n_seg ? L.hdr[H_LEN + g] : 0;
                        const bool far = g < n_seg && L.hdr[H_BW + g] > 5;        // (its centroids are not in LDS)
                        const bool any_far = __builtin_amdgcn_ballot_w64(far) != 0;
                        const uint8_t* at = &raw[li * CROW + (s & ~3)];
                        const float* cent = &L.cent[(g & 7) * 32];
                        float sum = 0.f;
                        uint32_t w[3];                        // codes s .. s + 7 from byte s & 3 on
                        auto fetch = [&](int t) {
#pragma unroll
                            for (int i = 0; i < 3; i++) w[i] = *(const uint32_t*)(at + t + 4 * i);
                        };
                        fetch(0);
                        for (int t = 0; __builtin_amdgcn_ballot_w64(t < len) != 0; t += 8) {
                            const uint32_t lo = __builtin_amdgcn_alignbyte(w[1], w[0], s & 3), hi = __builtin_amdgcn_alignbyte(w[2], w[1], s & 3);
                            float c[8];
                            if (any_far) {                    // (uniform)
#pragma unroll
                                for (int i = 0; i < 8; i++) {
                                    const uint32_t code = ((i < 4 ? lo : hi) >> (8 * (i & 3))) & 0xFFu;
                                    c[i] = t + i >= len ? 0.f : far ? P.k_centroids[g][code] : cent[code & 31u];
                                }
                            } else {
#pragma unroll
                                for (int i = 0; i < 8; i++) c[i] = cent[((i < 4 ? lo : hi) >> (8 * (i & 3))) & 31u];
                            }
                            fetch(t + 8);
#pragma unroll
                            for (int i = 0; i < 8; i++) {
                                const float m = t + i < len ? c[i] : 0.f;
                                sum = __builtin_fmaf(m, m, sum);
                            }
                        }
                        store_norm(g, li, g < n_seg ? L.nrm[slot][g][li].x / fmaxf(__builtin_sqrtf(sum), 1e-10f) : 0.f);
                    }
                }
            } else {
                for (int i = lane; i < BGTQ_MAX_SEGMENTS * 16; i += 64) {
                    const int g = i & 7, row = i >> 3;
                    store_norm(g, row, g < n_seg ? L.nrm[slot][g][row].x : 0.f);
                }
            }
        }
        // ---- records
        if (a.codes_out) {
            for (int i = part * 64 + lane; i < 16 * (D / 4); i += 64 * CS) {
                const int64_t n = L.dst[slot][i >> 5];
                if (n >= 0) *(uint32_t*)&a.codes_out[n * D + 4 * (i & 31)] = *(const uint32_t*)&raw[(i >> 5) * CROW + 4 * (i & 31)];
            }
        } else if (4 * dw < a.row_width) {
            const int rows = 64 / lpr;
            uint4 make[4];                                    // (the stores could alias the table for all the compiler knows: read once)
#pragma unroll
            for (int i = 0; i < 4; i++) make[i] = L.pack[4 * dw + i];
#pragma unroll 2
            for (int r = lane / lpr + part * rows; r < 16; r += rows * CS) {
                const int64_t dst = L.dst[slot][r];
                if (dst < 0) continue;
                uint32_t byte[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint4 p = make[i];
                    const uint32_t* c = (const uint32_t*)&raw[r * CROW + (p.x & ~3u)];
                    const uint32_t c0 = c[0], c1 = c[1];
                    const uint32_t x = __builtin_amdgcn_alignbyte(c1, c0, p.x & 3u);
                    byte[i] = __builtin_amdgcn_udot4(x, p.z, __builtin_amdgcn_ubfe(x, p.y & 0xFFu, p.y >> 8), false);
                    if (two_dots) byte[i] += __builtin_amdgcn_udot4(__builtin_amdgcn_alignbyte(c[2], c1, p.x & 3u), p.w, 0u, false) << 4;
                }
                const uint32_t w = __builtin_amdgcn_perm(byte[1], byte[0], 0x0C0C0400u) | __builtin_amdgcn_perm(byte[3], byte[2], 0x04000C0Cu);
                if (dwords) *(uint32_t*)(a.packed + dst + 4 * dw) = w;
                else
                    for (int i = 0; i < 4; i++)
                        if (4 * dw + i < a.row_width) a.packed[dst + 4 * dw + i] = (uint8_t)(w >> (8 * i));
            }
        }
        meet();                                               // the next block's rows overwrite codes and offsets
    }
}

template <int CS>
__global__ __launch_bounds__(EncodeLds<CS>::NW * 64) void encode_blocks_kernel(TileArgs t) {
    __shared__ __align__(16) EncodeLds<CS> L;
    int bid = blockIdx.x;
    const int nv = t.v_groups * t.v.n_kv;                     // (V blocks, the longer ones, go out first)
    if (bid < nv) encode_blocks<CS, true>(t.v, bid % t.v.n_kv, bid / t.v.n_kv, t.v_groups, L);
    else {
        bid -= nv;
        encode_blocks<CS, false>(t.k, bid % t.k.n_kv, bid / t.k.n_kv, t.k_groups, L);
    }
}

// K and / or V rows in blocks; either pointer may be null
int launch_blocks(const EncodeArgs* k, const EncodeArgs* v, hipStream_t st) {
    const EncodeArgs& any = k ? *k : *v;
    const int64_t N = (int64_t)any.B * any.S;
    if (N > INT32_MAX - 64) return BGTQ_EINVAL;               // the kernels index rows with 32 bits
    const int kinds = (k ? 1 : 0) + (v ? 1 : 0);
    TileArgs t{};
    if (k) t.k = *k;
    if (v) t.v = *v;
    const int64_t blocks = (N + 15) / 16;
    if (blocks * any.n_kv * kinds <= 512) {                   // (two work-groups fit a compute unit: one round)
        t.k_groups = k ? (int)blocks : 0;
        t.v_groups = v ? (int)blocks : 0;
        hipLaunchKernelGGL(encode_blocks_kernel<4>, dim3((unsigned)(blocks * any.n_kv * kinds)), dim3(256), 0, st, t);
        return bgtq_launch_status();
    }
    // One work-group of up to 16 waves a compute unit, in equal shares over kinds and heads, each wave the same
    // number of blocks; with fewer than 16 blocks a work-group, that many waves; with at most 8, two waves a block (2600
    // tokens of 2 heads, 6 blocks: 25.9 us with six waves, 18.0 with twelve).
    const int64_t most = std::max<int64_t>(1, 256 / (any.n_kv * kinds));
    const int64_t share = (blocks + most - 1) / most, rounds = (share + 15) / 16;
    if (share <= 8) {
        const int groups = (int)((blocks + share - 1) / share);      // (of at least `share` blocks at a time: one round)
        t.k_groups = k ? groups : 0;
        t.v_groups = v ? groups : 0;
        hipLaunchKernelGGL(encode_blocks_kernel<2>, dim3((unsigned)(groups * kinds * any.n_kv)), dim3((unsigned)std::max<int64_t>(4, 2 * share) * 64), 0, st, t);
        return bgtq_launch_status();
    }
    const int nw = (int)std::max<int64_t>(4, (share + rounds - 1) / rounds);
    const int groups = (int)((blocks + nw * rounds - 1) / (nw * rounds));
    t.k_groups = k ? groups : 0;
    t.v_groups = v ? groups : 0;
    hipLaunchKernelGGL(encode_blocks_kernel<1>, dim3((unsigned)(groups * kinds * any.n_kv)), dim3(nw * 64), 0, st, t);
    return bgtq_launch_status();
}

template <bool IS_V>
int launch_encode(const EncodeArgs& a, hipStream_t st) {
    const int64_t N = (int64_t)a.B * a.S;
    if (N == 0 || a.n_kv == 0) return BGTQ_OK;
    // few rows (a decode append): one row a work-group, the shortest chain of dependent stages
    if (N > 32) return IS_V ? launch_blocks(nullptr, &a, st) : launch_blocks(&a, nullptr, st);
    hipLaunchKernelGGL(encode_kernel<IS_V>, dim3((unsigned)N, (unsigned)a.n_kv), dim3(NT), 0, st, a);
    return bgtq_launch_status();
}

// ---- query permute + rotate ---------------------------------------------------
struct RotQArgs {
    const bgtq_head_plan* plans;
    const uint16_t* q;  int64_t q_sr, q_sh;
    uint16_t* q_rot;    int64_t qr_sr, qr_sh;
    int n_rows, n_q, gqa;
    int group;          // query heads per work-group: 1 or 4
    int bf16;           // q holds bf16
};

// QG query heads (h_first ..) of one (row, KV head): the rotation is fetched and parked once for
// all of them, the rows come in with the same round of loads (un-permuted, so that their
// addresses do not wait for head_perm; the gather by head_perm then runs through LDS), and a
// batch of the rotation column read from LDS serves every row.  Each row's chain is the one
// written in the contract above; rows past the group's last head are zeros and are not stored.
template <int QG>
__device__ __forceinline__ void rotate_q_group(const RotQArgs& a, const int64_t row, const int h,
                                               const int h_first, float* rot_s) {
    __shared__ uint16_t qraw[QG][D];
    __shared__ float xs[QG + 1][D];                 // (one more row of zeros, see the compact chain below)
    const int j = threadIdx.x;
    const bgtq_head_plan& P = a.plans[h];
    // what thread j needs of the segment table comes ready-made (enc_dim), and so does its column of
    // the rotation where the plan holds it by columns (no rotated segment longer than BGTQ_ROT_COL)
    const int4 dim = *(const int4*)P.enc_dim[j];
    const int g = dim.x, s = dim.y, e = dim.z, ident = dim.w & 0xFF, src = dim.w >> 8;
    const bool compact = P.rot_compact[0] != 0;      // (uniform)
    rot_piece rst[D / 4];
    float rc[BGTQ_ROT_COL];
    if (compact) {
#pragma unroll
        for (int i = 0; i < BGTQ_ROT_COL / 4; i++) {
            const float4 v = *(const float4*)&P.k_rot_cols[j][4 * i];
            rc[4 * i] = v.x; rc[4 * i + 1] = v.y; rc[4 * i + 2] = v.z; rc[4 * i + 3] = v.w;
        }
    } else {
        fetch_rotation(P.k_rot_T, j, rst);
    }
    const int gqa = a.gqa;
#pragma unroll
    for (int r = 0; r < QG; r++)
        qraw[r][j] = h_first + r < gqa ? a.q[row * a.q_sr + (int64_t)(h * gqa + h_first + r) * a.q_sh + j] : (uint16_t)0;
    xs[QG][j] = 0.f;
    if (!compact) park_rotation(rot_s, j, rst);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < QG; r++) xs[r][j] = bgtq_h2f(bgtq_in16(qraw[r][src], a.bf16));
    __syncthreads();
    float acc[QG];
#pragma unroll
    for (int r = 0; r < QG; r++) acc[r] = 0.f;
    if (g >= 0) {
        if (ident) {
#pragma unroll
            for (int r = 0; r < QG; r++) acc[r] = xs[r][j];
        } else if (compact) {
            // the column is zero past the segment's end: BGTQ_ROT_COL terms for every dim, no length test
            // (a term x * 0 leaves the sum as it is; the values read past the row are finite)
            constexpr int CB = QG == 1 ? 16 : 8;
#pragma unroll
            for (int i0 = 0; i0 < BGTQ_ROT_COL; i0 += CB) {
                float xv[QG][CB];
#pragma unroll
                for (int i = 0; i < CB; i++)
#pragma unroll
                    for (int r = 0; r < QG; r++) xv[r][i] = (&xs[r][0])[s + i0 + i];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < CB; i++)
#pragma unroll
                    for (int r = 0; r < QG; r++) acc[r] = __builtin_fmaf(xv[r][i], rc[i0 + i], acc[r]);
            }
        } else {
            constexpr int CB = QG == 1 ? 16 : 8;    // LDS reads a batch ahead of the chains
            for (int k0 = s; k0 < e; k0 += CB) {
                float rk[CB], xv[QG][CB];
#pragma unroll
                for (int i = 0; i < CB; i++) {
                    const int k = min(k0 + i, e - 1);
                    rk[i] = rot_s[k * D + j];
#pragma unroll
                    for (int r = 0; r < QG; r++) xv[r][i] = xs[r][k];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < CB; i++)
                    if (k0 + i < e) {
#pragma unroll
                        for (int r = 0; r < QG; r++) acc[r] = __builtin_fmaf(xv[r][i], rk[i], acc[r]);
                    }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < QG; r++)
        if (h_first + r < gqa)
            a.q_rot[row * a.qr_sr + (int64_t)(h * gqa + h_first + r) * a.qr_sh + j] = bgtq_f2h(acc[r]);
}

// Query heads [part * a.group, ..) of one (row, KV head).  One head per
// work-group where that still leaves the chip partly idle (every work-group fetches the 64 KB
// rotation), four where the rows are many.
__device__ __forceinline__ void rotate_q_block(const RotQArgs& a, const int row, const int h, const int part, float* rot_s) {
    if (a.group == 1) rotate_q_group<1>(a, row, h, part, rot_s);
    else              rotate_q_group<4>(a, row, h, part * 4, rot_s);
}
__device__ __forceinline__ void rotate_q_block(const RotQArgs& a, const int bid, float* rot_s) {
    const int n_kv = a.n_q / a.gqa;
    const int per = (a.gqa + a.group - 1) / a.group;            // work-groups per (row, KV head)
    const int rowh = bid / per, part = bid - rowh * per;
    rotate_q_block(a, rowh / n_kv, rowh % n_kv, part, rot_s);
}
__host__ inline int rotate_q_group_size(int64_t n_rows, int n_q) { return n_rows * n_q > 256 ? 4 : 1; }
__host__ inline unsigned rotate_q_blocks(int64_t n_rows, int n_kv, int gqa, int group) {
    return (unsigned)(n_rows * n_kv * ((gqa + group - 1) / group));
}

__global__ __launch_bounds__(NT) void rotate_q_kernel(RotQArgs a) {
    __shared__ __align__(16) float rot_s[D * D];
    rotate_q_block(a, blockIdx.x, rot_s);
}

// ---- batch rows by falling length, for the attention launch that follows: lengths on the device, one work-group ----
struct RankArgs { const int32_t* lens; int32_t* order; int B; };      // order null: not asked for
static_assert(BGTQ_ONE_LAUNCH_ROWS <= NT, "a thread a row");

__device__ __forceinline__ void rank_rows(const RankArgs& r, const int tid, int* lens_s) {
    if (tid < r.B) lens_s[tid] = r.lens[tid];
    __syncthreads();
    if (tid < r.B) r.order[bgtq_row_rank(lens_s, r.B, tid)] = tid;
}

// ---- decode-step preparation: append-encode K and V and rotate the queries, one launch ----
// Work-groups [0, n) encode one V row of one head each (the longest chain of the three goes out first),
// [n, 2 n) one K row each, the rest rotate one or four query heads each.
__device__ __forceinline__ void prepare_part(const EncodeArgs& ak, const EncodeArgs& av, const RotQArgs& aq,
                                             const int rows, int bid, float* rot_s) {
    const int n = rows * ak.n_kv;
    if (bid < n) {
        encode_row<true>(av, bid % rows, bid / rows, threadIdx.x, rot_s);
    } else if (bid < 2 * n) {
        bid -= n;
        encode_row<false>(ak, bid % rows, bid / rows, threadIdx.x, rot_s);
    } else {
        rotate_q_block(aq, bid - 2 * n, rot_s);
    }
}
// (BF16: some input is; asking at run time costs the chains of fp16 inputs 0.2 of 5.0 us)
// Steps of one token whose rows need no rank, which is nearly all: the grid is (rows, KV heads, 2 + query parts), with no division
// on the way to a work-group's rows, and what the first loads need (plans, K and V rows) comes as arguments of its own ahead of
// the blocks: they are in scalar registers when a wave starts (kernarg preload), the blocks a trip to memory behind it.
// One row x 8 heads of 4k tokens 65.2 -> 63.0 us (4 layers), 4 rows x 2 heads of 8k 151.3 -> 146.7 (8), 12 ragged rows of 7-head
// groups 87.8 -> 86.1 (4), 8 x 2 of 32k 205.1 -> 202.2 (6).
template <bool BF16>
__global__ __launch_bounds__(NT) void prepare_token_kernel(const bgtq_head_plan* plans, const uint16_t* v, const uint16_t* k, uint32_t v_sb, uint32_t v_sh,
                                                           uint32_t k_sb, uint32_t k_sh, EncodeArgs ak, EncodeArgs av, RotQArgs aq) {
    __shared__ __align__(16) float rot_s[D * D];       // the work-group's rotation, whatever its role
    if (!BF16) ak.bf16 = av.bf16 = aq.bf16 = 0;
    ak.plans = av.plans = aq.plans = plans;
    av.x = v; av.x_sb = v_sb; av.x_sh = v_sh;
    ak.x = k; ak.x_sb = k_sb; ak.x_sh = k_sh;
    ak.S = av.S = 1;
    const int row = blockIdx.x, h = blockIdx.y, role = blockIdx.z;
    if (role == 0) encode_row<true>(av, row, h, threadIdx.x, rot_s);
    else if (role == 1) encode_row<false>(ak, row, h, threadIdx.x, rot_s);
    else rotate_q_block(aq, row, h, role - 2, rot_s);
}
// All others.  Rank: RankArgs of a first work-group that ranks the rows, or nothing.  (Behind the others it started when a place
// came free and ended last: 64 equal rows x 8 heads of 700 tokens 43.1 us a step as they come, 45.5 with a last one, 43.9 with a
// first.  One that finds nothing to rank and its arguments cost two new tokens of one row x 8 heads of 4k 1.1 %: 79.6 -> 80.6 us, 4
// layers; eight of 8 x 2 and four of 12 x 4 rows nothing.)
template <bool BF16, class... Rank>
__global__ __launch_bounds__(NT) void prepare_kernel(EncodeArgs ak, EncodeArgs av, RotQArgs aq, int rows, Rank... rank) {
    if (!BF16) ak.bf16 = av.bf16 = aq.bf16 = 0;
    __shared__ __align__(16) float rot_s[D * D];
    if constexpr (sizeof...(Rank) != 0)
        if (blockIdx.x == 0) {                         // (uniform)
            rank_rows(rank..., threadIdx.x, (int*)rot_s);
            return;
        }
    prepare_part(ak, av, aq, rows, (int)blockIdx.x - (int)sizeof...(Rank), rot_s);
}
// The same with the attention over the buffered tokens, which depends on none of it: the longer work-groups first, in
// the LDS that is a rotation's otherwise; then the token that leaves the buffer, K and V by the two halves of a
// work-group, then the queries by two waves (a barrier counts the waves that are left).  SWAP: the step's token enters the
// buffer here, put there by those who read the one that leaves.
// 32 rows x 8 heads x 4 queries over 132 buffered tokens: 4.9 (swap) + 11.1 + 13.3 us as launches of their own, 4.9 + 16.3
// with K and V a work-group each and the swap ahead of them (1024 work-groups, two of them at a time on a compute unit), 14 here.
template <bool SWAP, class... Rank>
__global__ __launch_bounds__(WINDOW_THREADS, 2) void prepare_window_kernel(EncodeArgs ak, EncodeArgs av, RotQArgs aq, WindowArgs w,
                                                                        RingArgs rk, RingArgs rv, int rows, int n_window, Rank... rank) {
    __shared__ __align__(16) float rot_s[D * D];
    static_assert(window_lds_floats<4>(WINDOW_RIDE_W) <= D * D, "a window's scores fit the rotation's place");
    static_assert(WINDOW_THREADS == 2 * NT, "");
    int bid = blockIdx.x;
    const int n_kv = ak.n_kv, tid = threadIdx.x;
    if constexpr (sizeof...(Rank) != 0)
        if (bid == (int)gridDim.x - 1) {               // (in front of the longer ones it cost the window case 0.6 of 103 us a layer)
            rank_rows(rank..., tid, (int*)rot_s);
            return;
        }
    if (bid < n_window) {
        window_attn_block<4, SWAP>(w, bid % n_kv, bid / n_kv, rot_s);
        return;
    }
    bid -= n_window;
    if (bid < rows * n_kv) {
        const int row = bid % rows, h = bid / rows;
        if (tid < NT) encode_row<true, true>(av, row, h, tid, rot_s, SWAP ? &rv : nullptr);
        else encode_row<false, true>(ak, row, h, tid - NT, rot_s, SWAP ? &rk : nullptr);
    } else if (tid < NT) {
        rotate_q_block(aq, bid - rows * n_kv, rot_s);
    }
}

// argument checks + EncodeArgs assembly shared by the separate and the fused entry points
int fill_k_args(EncodeArgs& a, const bgtq_head_plan* plans,
                const void* k, int64_t k_sb, int64_t k_sh, int64_t k_ss, int B, int n_kv, int S,
                void* k_packed, int64_t kp_sb, int64_t kp_sh, int64_t kp_st, int k_row_width,
                void* k_norms, int64_t kn_sb, int64_t kn_sh, int64_t kn_st, int norm_width,
                const int32_t* t_pos, int t_pos_scalar, int max_T, int k_layout, int quant_mode) {
    BGTQ_CHECK_ARG(plans && k && k_packed && k_norms);
    BGTQ_CHECK_ARG(k_row_width >= 0 && k_row_width <= NT);
    BGTQ_CHECK_ARG(norm_width >= 0 && norm_width <= BGTQ_MAX_SEGMENTS);
    BGTQ_CHECK_ARG(k_layout == BGTQ_K_BITPACKED || k_layout == BGTQ_K_MIXED);
    BGTQ_CHECK_ARG(quant_mode == BGTQ_QUANT_LUT256 || quant_mode == BGTQ_QUANT_EXACT);
    BGTQ_CHECK_ARG(t_pos || t_pos_scalar >= 0);
    BGTQ_CHECK_ARG(max_T >= 0);
    if (!t_pos && (int64_t)t_pos_scalar + S > max_T) return BGTQ_ELIMIT;   // would run past the cache
    a.max_T = max_T;
    a.plans = plans; a.x = (const uint16_t*)k; a.x_sb = k_sb; a.x_sh = k_sh; a.x_ss = k_ss;
    a.B = B; a.n_kv = n_kv; a.S = S;
    a.packed = (uint8_t*)k_packed; a.p_sb = kp_sb; a.p_sh = kp_sh; a.p_st = kp_st;
    a.row_width = k_row_width;
    a.norms = (uint16_t*)k_norms; a.n_sb = kn_sb; a.n_sh = kn_sh; a.n_st = kn_st;
    a.norm_width = norm_width;
    a.t_pos = t_pos; a.t_pos_scalar = t_pos_scalar;
    a.layout = k_layout; a.quant_mode = quant_mode;
    return BGTQ_OK;
}

int fill_v_args(EncodeArgs& a, const bgtq_head_plan* plans,
                const void* v, int64_t v_sb, int64_t v_sh, int64_t v_ss, int B, int n_kv, int S,
                void* v_packed, int64_t vp_sb, int64_t vp_sh, int64_t vp_st, int v_row_width,
                void* v_norms, int64_t vn_sb, int64_t vn_sh, int64_t vn_st,
                const int32_t* t_pos, int t_pos_scalar, int max_T, int v_layout) {
    BGTQ_CHECK_ARG(plans && v && v_packed && v_norms);
    BGTQ_CHECK_ARG(v_row_width >= 0 && v_row_width <= NT);
    BGTQ_CHECK_ARG(v_layout == BGTQ_V_BITPACKED || v_layout == BGTQ_V_NIBBLE);
    BGTQ_CHECK_ARG(t_pos || t_pos_scalar >= 0);
    BGTQ_CHECK_ARG(max_T >= 0);
    if (!t_pos && (int64_t)t_pos_scalar + S > max_T) return BGTQ_ELIMIT;
    a.max_T = max_T;
    a.plans = plans; a.x = (const uint16_t*)v; a.x_sb = v_sb; a.x_sh = v_sh; a.x_ss = v_ss;
    a.B = B; a.n_kv = n_kv; a.S = S;
    a.packed = (uint8_t*)v_packed; a.p_sb = vp_sb; a.p_sh = vp_sh; a.p_st = vp_st;
    a.row_width = v_row_width;
    a.norms = (uint16_t*)v_norms; a.n_sb = vn_sb; a.n_sh = vn_sh; a.n_st = vn_st;
    a.norm_width = 1;
    a.t_pos = t_pos; a.t_pos_scalar = t_pos_scalar;
    a.layout = v_layout;
    return BGTQ_OK;
}

int launch_rotate_q(const bgtq_head_plan* plans, const void* q, int64_t q_sr, int64_t q_sh, int bf16,
                    void* q_rot, int64_t qr_sr, int64_t qr_sh, int n_rows, int n_kv, int gqa, hipStream_t st) {
    const int group = rotate_q_group_size(n_rows, n_kv * gqa);
    RotQArgs a{plans, (const uint16_t*)q, q_sr, q_sh, (uint16_t*)q_rot, qr_sr, qr_sh, n_rows, n_kv * gqa, gqa, group, bf16};
    hipLaunchKernelGGL(rotate_q_kernel, dim3(rotate_q_blocks(n_rows, n_kv, gqa, group)), dim3(NT), 0, st, a);
    return bgtq_launch_status();
}

// K and V appended and (q not null) the queries rotated: one launch for the few rows of a decode step
int launch_prepare(const EncodeArgs& ak, const EncodeArgs& av, const void* q, int64_t q_sr, int64_t q_sh, int q_bf16,
                   void* q_rot, int64_t qr_sr, int64_t qr_sh, int gqa, const WindowArgs* window, const RankArgs& rank, hipStream_t st) {
    const int B = ak.B, n_kv = ak.n_kv;
    const int64_t N = (int64_t)B * ak.S;
    if (N > BGTQ_ONE_LAUNCH_ROWS) {          // prefill-sized append: the three stages are big enough on their own
        const int rc = launch_blocks(&ak, &av, st);
        if (rc != BGTQ_OK || !q) return rc;
        return launch_rotate_q(ak.plans, q, q_sr, q_sh, q_bf16, q_rot, qr_sr, qr_sh, B, n_kv, gqa, st);
    }
    const int group = rotate_q_group_size(B, n_kv * gqa);
    RotQArgs aq{ak.plans, (const uint16_t*)q, q_sr, q_sh, (uint16_t*)q_rot, qr_sr, qr_sh, B, n_kv * gqa, gqa, group, q_bf16};
    const int rows = (int)N;
    const unsigned blocks = (unsigned)(2 * rows * n_kv) + (q ? rotate_q_blocks(B, n_kv, gqa, group) : 0u) + (rank.order ? 1u : 0u);
    if (window) {
        const WindowArgs& w = *window;
        const dim3 grid(blocks - (unsigned)(rows * n_kv) + (unsigned)(B * n_kv));
        const RingArgs rk{w.swap.slot, (uint16_t*)w.kbuf, w.w_sb, w.w_sh, w.w_st, w.W, w.swap.k, w.swap.k_sb, w.swap.k_sh, w.bf16};
        const RingArgs rv{w.swap.slot, (uint16_t*)w.vbuf, w.w_sb, w.w_sh, w.w_st, w.W, w.swap.v, w.swap.v_sb, w.swap.v_sh, w.bf16};
        if (rank.order) {
            auto kern = w.swap.slot ? prepare_window_kernel<true, RankArgs> : prepare_window_kernel<false, RankArgs>;
            hipLaunchKernelGGL(kern, grid, dim3(WINDOW_THREADS), 0, st, ak, av, aq, w, rk, rv, rows, B * n_kv, rank);
        } else {
            auto kern = w.swap.slot ? prepare_window_kernel<true> : prepare_window_kernel<false>;
            hipLaunchKernelGGL(kern, grid, dim3(WINDOW_THREADS), 0, st, ak, av, aq, w, rk, rv, rows, B * n_kv);
        }
    } else {
        const bool bf16 = ak.bf16 || av.bf16 || (q && q_bf16);
        const int64_t strides[] = {av.x_sb, av.x_sh, ak.x_sb, ak.x_sh};
        bool token = !rank.order && ak.S == 1;
        for (int64_t each : strides) token = token && each >= 0 && each < (int64_t)1 << 32;
        if (token) {
            auto kern = bf16 ? prepare_token_kernel<true> : prepare_token_kernel<false>;
            const dim3 grid((unsigned)rows, (unsigned)n_kv, 2u + (q ? (unsigned)((gqa + group - 1) / group) : 0u));
            hipLaunchKernelGGL(kern, grid, dim3(NT), 0, st, ak.plans, av.x, ak.x, (uint32_t)av.x_sb, (uint32_t)av.x_sh,
                               (uint32_t)ak.x_sb, (uint32_t)ak.x_sh, ak, av, aq);
        } else if (blocks == 0) {
            return BGTQ_OK;                            // (no tokens and no queries)
        } else if (rank.order) {
            auto kern = bf16 ? prepare_kernel<true, RankArgs> : prepare_kernel<false, RankArgs>;
            hipLaunchKernelGGL(kern, dim3(blocks), dim3(NT), 0, st, ak, av, aq, rows, rank);
        } else {
            auto kern = bf16 ? prepare_kernel<true> : prepare_kernel<false>;
            hipLaunchKernelGGL(kern, dim3(blocks), dim3(NT), 0, st, ak, av, aq, rows);
        }
    }
    return bgtq_launch_status();
}

int fill_step_args(const bgtq_step& s, EncodeArgs& ak, EncodeArgs& av) {
    BGTQ_CHECK_ARG(s.x_dtype == BGTQ_X_FP16 || s.x_dtype == BGTQ_X_BF16);
    int rc = fill_k_args(ak, s.plans, s.k, s.k_sb, s.k_sh, s.k_ss, s.B, s.n_kv, s.S, s.k_packed, s.kp_sb, s.kp_sh, s.kp_st,
                         s.k_row_width, s.k_norms, s.kn_sb, s.kn_sh, s.kn_st, s.norm_width, s.t_pos, s.t_pos_scalar, s.max_T,
                         s.k_layout, s.quant_mode);
    if (rc != BGTQ_OK) return rc;
    rc = fill_v_args(av, s.plans, s.v, s.v_sb, s.v_sh, s.v_ss, s.B, s.n_kv, s.S, s.v_packed, s.vp_sb, s.vp_sh, s.vp_st,
                     s.v_row_width, s.v_norms, s.vn_sb, s.vn_sh, s.vn_st, s.t_pos, s.t_pos_scalar, s.max_T,
                     s.v_layout == BGTQ_V_NIBBLE4 ? BGTQ_V_NIBBLE : s.v_layout);
    ak.bf16 = av.bf16 = s.x_dtype == BGTQ_X_BF16;
    return rc;
}

}  // namespace

int bgtq_step_prepare(const bgtq_step& s, bool kv_fp16, const WindowArgs* window, int32_t* order, hipStream_t st) {
    EncodeArgs ak{}, av{};
    const int rc = fill_step_args(s, ak, av);
    if (rc != BGTQ_OK) return rc;
    const int q_bf16 = ak.bf16;
    if (kv_fp16) ak.bf16 = av.bf16 = 0;
    return launch_prepare(ak, av, s.q_rot ? s.q : nullptr, s.q_sb, s.q_sh, q_bf16, s.q_rot,
                          (int64_t)s.n_kv * s.gqa * D, D, s.gqa, window, RankArgs{s.seq_lens, order, s.B}, st);
}

extern "C" {

int bgtq_encode_kv(const bgtq_step* step, void* stream) {
    BGTQ_CHECK_ARG(step && step->B >= 0 && step->n_kv >= 0 && step->S >= 0);
    if (step->B == 0 || step->n_kv == 0 || step->S == 0) return BGTQ_OK;
    EncodeArgs ak{}, av{};
    const int rc = fill_step_args(*step, ak, av);
    if (rc != BGTQ_OK) return rc;
    return launch_prepare(ak, av, nullptr, 0, 0, 0, nullptr, 0, 0, 1, nullptr, RankArgs{}, (hipStream_t)stream);
}

int bgtq_encode_k(const bgtq_head_plan* plans,
                  const void* k, int64_t k_sb, int64_t k_sh, int64_t k_ss,
                  int B, int n_kv, int S,
                  void* k_packed, int64_t kp_sb, int64_t kp_sh, int64_t kp_st, int k_row_width,
                  void* k_norms, int64_t kn_sb, int64_t kn_sh, int64_t kn_st, int norm_width,
                  const int32_t* t_pos, int t_pos_scalar, int max_T,
                  int k_layout, int quant_mode, void* stream) {
    BGTQ_CHECK_ARG(B >= 0 && n_kv >= 0 && S >= 0);
    if (B == 0 || n_kv == 0 || S == 0) return BGTQ_OK;     // nothing to encode
    EncodeArgs a{};
    int rc = fill_k_args(a, plans, k, k_sb, k_sh, k_ss, B, n_kv, S, k_packed, kp_sb, kp_sh, kp_st, k_row_width,
                         k_norms, kn_sb, kn_sh, kn_st, norm_width, t_pos, t_pos_scalar, max_T, k_layout, quant_mode);
    if (rc != BGTQ_OK) return rc;
    return launch_encode<false>(a, (hipStream_t)stream);
}

int bgtq_encode_v(const bgtq_head_plan* plans,
                  const void* v, int64_t v_sb, int64_t v_sh, int64_t v_ss,
                  int B, int n_kv, int S,
                  void* v_packed, int64_t vp_sb, int64_t vp_sh, int64_t vp_st, int v_row_width,
                  void* v_norms, int64_t vn_sb, int64_t vn_sh, int64_t vn_st,
                  const int32_t* t_pos, int t_pos_scalar, int max_T,
                  int v_layout, void* stream) {
    BGTQ_CHECK_ARG(B >= 0 && n_kv >= 0 && S >= 0);
    if (B == 0 || n_kv == 0 || S == 0) return BGTQ_OK;
    EncodeArgs a{};
    int rc = fill_v_args(a, plans, v, v_sb, v_sh, v_ss, B, n_kv, S, v_packed, vp_sb, vp_sh, vp_st, v_row_width,
                         v_norms, vn_sb, vn_sh, vn_st, t_pos, t_pos_scalar, max_T, v_layout);
    if (rc != BGTQ_OK) return rc;
    return launch_encode<true>(a, (hipStream_t)stream);
}

int bgtq_compress_k_codes(const bgtq_head_plan* plan, const void* k, int64_t N,
                          void* codes, float* norms, int norm_width,
                          int corrected, int quant_mode, void* stream) {
    BGTQ_CHECK_ARG(plan && k && codes && norms);
    BGTQ_CHECK_ARG(N >= 0 && N < (int64_t)1 << 31);
    BGTQ_CHECK_ARG(norm_width >= 1 && norm_width <= BGTQ_MAX_SEGMENTS);
    BGTQ_CHECK_ARG(quant_mode == BGTQ_QUANT_LUT256 || quant_mode == BGTQ_QUANT_EXACT);
    EncodeArgs a{};
    a.plans = plan; a.x = (const uint16_t*)k; a.x_sb = 0; a.x_sh = 0; a.x_ss = D;
    a.B = 1; a.n_kv = 1; a.S = (int)N;
    a.codes_out = (uint8_t*)codes; a.norms_f32_out = norms; a.norm_width = norm_width;
    a.corrected = corrected; a.layout = BGTQ_K_BITPACKED; a.quant_mode = quant_mode;
    return launch_encode<false>(a, (hipStream_t)stream);
}

int bgtq_compress_v_codes(const bgtq_head_plan* plan, const void* v, int64_t N,
                          void* codes, void* norms_f16, void* stream) {
    BGTQ_CHECK_ARG(plan && v && codes && norms_f16);
    BGTQ_CHECK_ARG(N >= 0 && N < (int64_t)1 << 31);
    EncodeArgs a{};
    a.plans = plan; a.x = (const uint16_t*)v; a.x_sb = 0; a.x_sh = 0; a.x_ss = D;
    a.B = 1; a.n_kv = 1; a.S = (int)N;
    a.codes_out = (uint8_t*)codes; a.norms = (uint16_t*)norms_f16; a.norm_width = 1;
    return launch_encode<true>(a, (hipStream_t)stream);
}

int bgtq_rotate_q(const bgtq_head_plan* plans,
                  const void* q, int64_t q_sr, int64_t q_sh,
                  void* q_rot, int64_t qr_sr, int64_t qr_sh,
                  int n_rows, int n_kv, int gqa, void* stream) {
    BGTQ_CHECK_ARG(plans && q && q_rot);
    BGTQ_CHECK_ARG(n_rows >= 0 && n_kv >= 0 && gqa >= 1);
    if (n_rows == 0 || n_kv == 0) return BGTQ_OK;
    return launch_rotate_q(plans, q, q_sr, q_sh, 0, q_rot, qr_sr, qr_sh, n_rows, n_kv, gqa, (hipStream_t)stream);
}

int bgtq_decode_prepare(const bgtq_head_plan* plans,
                        const void* k, int64_t k_sb, int64_t k_sh, int64_t k_ss,
                        const void* v, int64_t v_sb, int64_t v_sh, int64_t v_ss,
                        int B, int n_kv, int S,
                        void* k_packed, int64_t kp_sb, int64_t kp_sh, int64_t kp_st, int k_row_width,
                        void* k_norms, int64_t kn_sb, int64_t kn_sh, int64_t kn_st, int norm_width,
                        void* v_packed, int64_t vp_sb, int64_t vp_sh, int64_t vp_st, int v_row_width,
                        void* v_norms, int64_t vn_sb, int64_t vn_sh, int64_t vn_st,
                        const int32_t* t_pos, int t_pos_scalar, int max_T,
                        int k_layout, int v_layout, int quant_mode,
                        const void* q, int64_t q_sr, int64_t q_sh,
                        void* q_rot, int64_t qr_sr, int64_t qr_sh, int gqa, void* stream) {
    BGTQ_CHECK_ARG(B >= 0 && n_kv >= 0 && S >= 0 && gqa >= 1);
    if (B == 0 || n_kv == 0) return BGTQ_OK;
    EncodeArgs ak{}, av{};
    int rc = fill_k_args(ak, plans, k, k_sb, k_sh, k_ss, B, n_kv, S, k_packed, kp_sb, kp_sh, kp_st, k_row_width,
                         k_norms, kn_sb, kn_sh, kn_st, norm_width, t_pos, t_pos_scalar, max_T, k_layout, quant_mode);
    if (rc != BGTQ_OK) return rc;
    rc = fill_v_args(av, plans, v, v_sb, v_sh, v_ss, B, n_kv, S, v_packed, vp_sb, vp_sh, vp_st, v_row_width,
                     v_norms, vn_sb, vn_sh, vn_st, t_pos, t_pos_scalar, max_T, v_layout);
    if (rc != BGTQ_OK) return rc;
    BGTQ_CHECK_ARG((q == nullptr) == (q_rot == nullptr));     // both, or neither (queries rotated elsewhere)
    return launch_prepare(ak, av, q, q_sr, q_sh, 0, q_rot, qr_sr, qr_sh, gqa, nullptr, RankArgs{}, (hipStream_t)stream);
}


}  // extern "C"
