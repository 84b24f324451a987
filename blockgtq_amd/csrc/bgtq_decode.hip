// Fused unpack + dequant + split-T decode attention, the partition merge, and
// the dense fp16 window partial, for gfx950.
//
// decode_generic_kernel is the layout-agnostic path: any segment table, both K
// layouts, both V layouts, any row stride.  One work-group of 256 threads owns
// one partition of one (batch row, KV head).  Per 256-token tile the packed K
// rows, K norms, packed V rows and V norms are staged into LDS with coalesced
// loads; thread t then scores token t against all query heads of the group
// (codes pulled out of the staged record with shift/mask, codebooks and the
// rotated queries read from LDS), the tile maximum is reduced across the
// work-group, and thread (d, half) accumulates output dim d for one half of
// the query heads over the tile's tokens.
#include "bgtq_common.h"
#include <algorithm>
#include <cmath>
#include <mutex>

#include "bgtq_decode.h"
#include "bgtq_window.h"

namespace {

constexpr int D = BGTQ_D;
constexpr int GT = 256;          // threads == tokens per tile of the generic kernel
constexpr int ROW_PAD = 4;       // slack bytes so a 2-byte window never leaves the tile


// code of width `bw` at absolute bit `bit` of a staged record
__device__ inline unsigned take_bits(const uint8_t* row, int bit, int bw) {
    int byte = bit >> 3;
    unsigned w = (unsigned)row[byte] | ((unsigned)row[byte + 1] << 8);
    return (w >> (bit & 7)) & ((1u << bw) - 1u);
}

template <int GQA_MAX>
__global__ __launch_bounds__(GT) void decode_generic_kernel(DecodeArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x;
    const int c = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
    const bgtq_head_plan& P = a.plans[h];
    const int gqa = a.gqa;

    // (a length beyond the capacity the caller stated reads nothing past it)
    const int T = a.seq_lens ? min(max(a.seq_lens[b], 0), a.T) : a.T;
    const int chunk = (T + a.n_splits - 1) / a.n_splits;
    const int t0 = min(c * chunk, T);
    const int t1 = min(t0 + chunk, T);

    // ---- LDS carve-up ------------------------------------------------------
    const int krow = (a.k_row_width + ROW_PAD + 3) & ~3;
    const int vrow = (a.v_row_width + ROW_PAD + 3) & ~3;
    float* q_s = (float*)smem;                               // [GQA_MAX][D]
    float* cb_s = q_s + GQA_MAX * D;                         // [8][256]
    float* vlut_s = cb_s + BGTQ_MAX_SEGMENTS * BGTQ_MAX_CENTROIDS;  // [16]
    float* p_s = vlut_s + 16;                                // [GQA_MAX][GT]
    float* red_s = p_s + GQA_MAX * GT;                       // [GQA_MAX][4]
    float* alpha_s = red_s + GQA_MAX * 4;                    // [GQA_MAX] rescale of the tile
    float* fin_s = alpha_s + GQA_MAX;                        // [2][GQA_MAX] final m, l
    float* kn_s = fin_s + 2 * GQA_MAX;                       // [GT][8]
    float* vn_s = kn_s + GT * BGTQ_MAX_SEGMENTS;             // [GT]
    uint32_t* dim_s = (uint32_t*)(vn_s + GT);                // [D] bit | bw<<16 | seg<<24
    uint8_t* krow_s = (uint8_t*)(dim_s + D);                 // [GT][krow]
    uint8_t* vrow_s = krow_s + (size_t)GT * krow;            // [GT][vrow]

    // ---- static tables -----------------------------------------------------
    for (int i = tid; i < gqa * D; i += GT) {
        int hq = i / D, d = i - hq * D;
        q_s[i] = bgtq_h2f(a.q[b * a.q_sb + (h * gqa + hq) * a.q_sh + d]);
    }
    for (int i = tid; i < BGTQ_MAX_SEGMENTS * BGTQ_MAX_CENTROIDS; i += GT)
        cb_s[i] = bgtq_h2f(P.k_codebook_f16[i >> 8][i & 255]);
    if (tid < 16) vlut_s[tid] = bgtq_h2f(P.v_lut_f16[tid]);
    if (tid < D) {
        int g = P.group_of[tid];
        uint32_t e = 0xFFFFFFFFu;
        if (g >= 0) {
            int bw = P.seg_bw[g], rel = tid - P.seg_start[g];
            int bit, xbw;
            if (a.k_layout == BGTQ_K_MIXED) {
                if (bw <= 4) { bit = (tid - P.n_zero_dims) * 4; xbw = 4; }
                else         { bit = (P.seg_mixed_off[g] + rel) * 8; xbw = 8; }
            } else {
                if (bw <= 4) { bit = P.seg_pack_off[g] * 8 + rel * bw; xbw = bw; }
                else         { bit = (P.seg_pack_off[g] + rel) * 8; xbw = 8; }
            }
            e = (uint32_t)bit | ((uint32_t)xbw << 16) | ((uint32_t)g << 24);
        }
        dim_s[tid] = e;
    }
    const int n_seg = P.n_seg;
    const int kbytes = min((a.k_layout == BGTQ_K_MIXED) ? P.k_mixed_bytes : P.k_row_bytes,
                           a.k_row_width);
    const int vbw = (a.v_layout == BGTQ_V_BITPACKED) ? P.v_bits : 4;
    const int vbytes = min(bgtq_seg_bytes(vbw, D), a.v_row_width);

    const uint8_t* kp_base = a.kp + b * a.kp_sb + h * a.kp_sh;
    const uint16_t* kn_base = a.kn + b * a.kn_sb + h * a.kn_sh;
    const uint8_t* vp_base = a.vp + b * a.vp_sb + h * a.vp_sh;
    const uint16_t* vn_base = a.vn + b * a.vn_sb + h * a.vn_sh;

    // running softmax state (replicated in every thread) and output accumulators
    float m_run[GQA_MAX], l_run[GQA_MAX];
    const int hhalf = (GQA_MAX + 1) / 2;         // heads per PV thread
    float acc[(GQA_MAX + 1) / 2];
#pragma unroll
    for (int i = 0; i < GQA_MAX; i++) { m_run[i] = -INFINITY; l_run[i] = 0.f; }
#pragma unroll
    for (int i = 0; i < hhalf; i++) acc[i] = 0.f;
    const int pv_d = tid & (D - 1);
    const int pv_h0 = (tid >> 7) * hhalf;

    for (int tile = t0; tile < t1; tile += GT) {
        const int nt = min(GT, t1 - tile);
        __syncthreads();   // previous tile fully consumed (also orders the static tables)
        // ---- stage the tile -----------------------------------------------
        for (int i = tid; i < nt * kbytes; i += GT) {
            int t = i / kbytes, o = i - t * kbytes;
            krow_s[t * krow + o] = kp_base[(int64_t)(tile + t) * a.kp_st + o];
        }
        for (int i = tid; i < nt * vbytes; i += GT) {
            int t = i / vbytes, o = i - t * vbytes;
            vrow_s[t * vrow + o] = vp_base[(int64_t)(tile + t) * a.vp_st + o];
        }
        for (int i = tid; i < nt * n_seg; i += GT) {
            int t = i / n_seg, g = i - t * n_seg;
            kn_s[t * BGTQ_MAX_SEGMENTS + g] = bgtq_h2f(kn_base[(int64_t)(tile + t) * a.kn_st + g]);
        }
        if (tid < nt) vn_s[tid] = bgtq_h2f(vn_base[(int64_t)(tile + tid) * a.vn_st]);
        __syncthreads();

        // ---- scores: thread = token ------------------------------------------
        float logit[GQA_MAX];
#pragma unroll
        for (int i = 0; i < GQA_MAX; i++) logit[i] = -INFINITY;
        if (tid < nt) {
            const uint8_t* row = krow_s + tid * krow;
            float tot[GQA_MAX], part[GQA_MAX];
#pragma unroll
            for (int i = 0; i < GQA_MAX; i++) { tot[i] = 0.f; part[i] = 0.f; }
            int cur = -1;
            for (int d = P.n_zero_dims; d < D; d++) {
                uint32_t e = dim_s[d];
                int g = (int)(e >> 24);
                if (g != cur) {
                    if (cur >= 0) {
                        float n = kn_s[tid * BGTQ_MAX_SEGMENTS + cur];
#pragma unroll
                        for (int i = 0; i < GQA_MAX; i++) { tot[i] += part[i] * n; part[i] = 0.f; }
                    }
                    cur = g;
                }
                unsigned code = take_bits(row, (int)(e & 0xFFFFu), (int)((e >> 16) & 0xFFu));
                float cv = cb_s[g * BGTQ_MAX_CENTROIDS + code];
#pragma unroll
                for (int i = 0; i < GQA_MAX; i++)
                    if (i < gqa) part[i] += q_s[i * D + d] * cv;
            }
            if (cur >= 0) {
                float n = kn_s[tid * BGTQ_MAX_SEGMENTS + cur];
#pragma unroll
                for (int i = 0; i < GQA_MAX; i++) tot[i] += part[i] * n;
            }
#pragma unroll
            for (int i = 0; i < GQA_MAX; i++) logit[i] = tot[i] * a.scale;
        }

        // ---- tile maximum per head (work-group reduce) -------------------------
#pragma unroll
        for (int i = 0; i < GQA_MAX; i++) {
            float m = wave_max(logit[i]);
            if ((tid & 63) == 0) red_s[i * 4 + (tid >> 6)] = m;
        }
        __syncthreads();
        float alpha[GQA_MAX];
#pragma unroll
        for (int i = 0; i < GQA_MAX; i++) {
            float m = fmaxf(fmaxf(red_s[i * 4], red_s[i * 4 + 1]),
                            fmaxf(red_s[i * 4 + 2], red_s[i * 4 + 3]));
            float m_new = fmaxf(m_run[i], m);
            alpha[i] = (m_run[i] == -INFINITY) ? 0.f : __expf(m_run[i] - m_new);
            m_run[i] = m_new;
            float p = (tid < nt && i < gqa) ? __expf(logit[i] - m_new) : 0.f;
            p_s[i * GT + tid] = p * ((tid < nt) ? vn_s[tid] : 0.f);   // V norm folded into p
            logit[i] = p;
            if (tid == 0) alpha_s[i] = alpha[i];
        }
        __syncthreads();   // red_s consumed, p_s visible
#pragma unroll
        for (int i = 0; i < GQA_MAX; i++) {
            float s = wave_sum(logit[i]);
            if ((tid & 63) == 0) red_s[i * 4 + (tid >> 6)] = s;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < GQA_MAX; i++) {
            float s = red_s[i * 4] + red_s[i * 4 + 1] + red_s[i * 4 + 2] + red_s[i * 4 + 3];
            l_run[i] = l_run[i] * alpha[i] + s;
        }

        // ---- values: thread = (dim, half of the heads) ------------------------
#pragma unroll
        for (int i = 0; i < hhalf; i++)
            if (pv_h0 + i < GQA_MAX) acc[i] *= alpha_s[pv_h0 + i];
        for (int t = 0; t < nt; t++) {
            unsigned code = take_bits(vrow_s + t * vrow, pv_d * vbw, vbw);
            float val = vlut_s[code];
#pragma unroll
            for (int i = 0; i < hhalf; i++)
                if (pv_h0 + i < GQA_MAX) acc[i] += p_s[(pv_h0 + i) * GT + t] * val;
        }
    }

    // ---- partition result --------------------------------------------------------
    __syncthreads();
    if (tid == 0) {
#pragma unroll
        for (int i = 0; i < GQA_MAX; i++) { fin_s[i] = m_run[i]; fin_s[GQA_MAX + i] = l_run[i]; }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < hhalf; i++) {
        int hq = pv_h0 + i;
        if (hq < gqa) {
            float l = fin_s[GQA_MAX + hq];
            float o = (t1 > t0) ? acc[i] / l : 0.f;
            size_t row = ((size_t)b * a.n_kv * gqa + (size_t)h * gqa + hq) * a.n_splits + c;
            a.part_out[row * D + pv_d] = o;
        }
    }
    if (tid < gqa) {
        float lse = (t1 > t0) ? fin_s[tid] + __logf(fin_s[GQA_MAX + tid]) : -INFINITY;
        size_t row = ((size_t)b * a.n_kv * gqa + (size_t)h * gqa + tid) * a.n_splits + c;
        a.part_lse[row] = lse;
    }
}

size_t generic_smem_bytes(int gqa_max, int krow_bytes, int vrow_bytes) {
    size_t krow = (size_t)((krow_bytes + ROW_PAD + 3) & ~3);
    size_t vrow = (size_t)((vrow_bytes + ROW_PAD + 3) & ~3);
    size_t f = (size_t)gqa_max * D + BGTQ_MAX_SEGMENTS * BGTQ_MAX_CENTROIDS + 16 +
               (size_t)gqa_max * GT + (size_t)gqa_max * 7 + (size_t)GT * BGTQ_MAX_SEGMENTS + GT + D;
    return f * 4 + (size_t)GT * (krow + vrow) + 16;
}

template <int GQA_MAX>
int launch_generic(const DecodeArgs& a, hipStream_t st) {
    size_t smem = generic_smem_bytes(GQA_MAX, a.k_row_width, a.v_row_width);
    auto kern = decode_generic_kernel<GQA_MAX>;
    if (smem > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)kern,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
        if (e != hipSuccess) return (int)e;
    }
    dim3 grid((unsigned)a.n_splits, (unsigned)a.n_kv, (unsigned)a.B);
    hipLaunchKernelGGL(kern, grid, dim3(GT), smem, st, a);
    return bgtq_launch_status();
}

// ---- partition merge + V un-rotation ------------------------------------------
// One work-group of RT_THREADS threads per (batch row, query head).  Its loads are 16 bytes a lane
// and contiguous across the wave: thread t holds columns 4(t & 31) .. +3 of the rows
// r = t >> 5 (mod RT_THREADS / 32) of the partial vectors and of the un-rotation, sums over its own
// rows, and the RT_THREADS / 32 row classes are added through LDS (in a fixed order, so the result
// does not depend on timing).  What depends on no computed value is asked for up front: the log-sum-exps,
// 16 partial vectors and the whole un-rotation.  Partitions behind the first 16 cost a round of loads each
// RT_THREADS / 32 of them.  512 threads (16 classes: 8 rows of the un-rotation a thread instead of 32) where the
// launch has at most one work-group per compute unit, 128 threads where work-groups queue up.
// Grid (heads of a group, KV heads, rows): no division on the way to the un-rotation.  The arguments up to n_extra fill 13 of the
// 14 scalar registers that hold them when a wave starts (kernarg preload): the first loads go out at once.  One row x 32 heads of
// 4k tokens 66.8 -> 65.2 us (4 layers), 4 x 16 of 8k 152.8 -> 151.2 (8), 12 x 28 ragged 88.2 -> 87.3 (4).
// MANY: how the weights of the partitions come about.  Up to merge_held() of them every wave works out maximum and denominator by
// itself, 16 lanes beside each other over log-sum-exps that they hold, and a thread the weights of its own row class: no trip through
// LDS and two barriers less.  Behind the first round of vectors it reads a log-sum-exp and then a vector, two trips; more partitions
// are therefore weighed once by the whole work-group, in LDS.  us a launch (repeated in a graph), held and by the work-group:
//   512 threads, 1 row x 4 heads: 24 partitions 2.74, 3.22; 48 3.20, 3.46; 64 3.52, 3.64; 85 4.27, 3.94; 128 5.33, 4.37; 256 8.62, 5.80
//                1 row x 32 heads: 24 2.82, 3.27; 64 3.60, 3.71; 85 4.41, 4.03; 128 5.48, 4.44 (past 64 with loops over the rest)
//   128 threads, 9 rows x 32 heads: 18 4.17, 4.22; 20 4.19, 4.25; 22 4.64, 4.63; 24 4.88, 4.71; 32 6.08, 5.46
//                32 rows x 32 heads: 18 6.19, 6.28; 20 6.39, 6.29; 22 6.83, 6.73; 24 6.90, 6.77; 32 7.97, 7.19; 64 16.2, 12.5
// (one row x 32 heads of 4k tokens, 32 partitions: 63.0 -> 61.5 us for 4 layers, 4 x 16 of 8k 146.7 -> 144.3 for 8, 12 x 28 ragged
// 85.2 -> 84.4 for 4; one row x 4 heads of 65k, 256 partitions, a layer: 25.9 us held, 20.1 by the work-group)
constexpr int merge_held(int threads) { return threads == 512 ? 64 : 20; }
static_assert(offsetof(bgtq_head_plan, v_rot) % 16 == 0 && sizeof(bgtq_head_plan) % 16 == 0,
              "the un-rotation is read 16 bytes at a time");
template <int RT_THREADS, bool MANY>
__global__ __launch_bounds__(RT_THREADS) void lse_reduce_kernel(
    const bgtq_head_plan* plans, const float* part_out, const float* part_lse, const float* extra_lse, int n_splits, int n_q,
    int gqa, int unrotate, int n_extra, const float* extra_out, uint16_t* out, int64_t o_sb, int64_t o_sh, float* lse_out) {
    constexpr int RT_CLASSES = RT_THREADS / 32;
    __shared__ __align__(16) float cls_sum[RT_CLASSES][D];
    __shared__ float vec[D];
    const int j = threadIdx.x;
    const int cls = j >> 5, c4 = (j & 31) * 4;
    const int h = blockIdx.y, hq = h * gqa + blockIdx.x, b = blockIdx.z;
    const size_t row = (size_t)b * n_q + hq;
    const float* pl = part_lse + row * n_splits;
    const float* el = extra_lse ? extra_lse + row * n_extra : nullptr;
    const float* R = plans[h].v_rot;
    const float* po = part_out + row * n_splits * D + c4;

    // loads land in issue order: the partitions' log-sum-exps go first
    constexpr int NB = 16 / RT_CLASSES;        // rounds of partial vectors fetched before anything else (16 vectors)
    constexpr int NL = MANY ? 1 : (merge_held(RT_THREADS) + 15) / 16;      // log-sum-exps a lane holds of all of them
    const int s16 = j & 15;
    float l_all[NL], l_own[NB];
    __shared__ float wgt[MANY ? BGTQ_MAX_SPLITS : 1], red[RT_THREADS / 64], dsum[RT_CLASSES];
    if constexpr (MANY) {
        l_all[0] = j < n_splits ? pl[j] : -INFINITY;
    } else {
#pragma unroll
        for (int i = 0; i < NL; i++) l_all[i] = s16 + 16 * i < n_splits ? pl[s16 + 16 * i] : -INFINITY;
#pragma unroll
        for (int i = 0; i < NB; i++) l_own[i] = RT_CLASSES * i + cls < n_splits ? pl[RT_CLASSES * i + cls] : -INFINITY;
    }
    float4 pv[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) pv[i] = *(const float4*)(po + (size_t)min(RT_CLASSES * i + cls, n_splits - 1) * D);
    const float x0 = n_extra && j < D ? extra_out[row * n_extra * D + j] : 0.f;
    float4 rv[D / RT_CLASSES];                 // rows 16 i + cls of the un-rotation, this thread's four columns
    if (unrotate) {
#pragma unroll
        for (int i = 0; i < D / RT_CLASSES; i++) rv[i] = *(const float4*)(R + (RT_CLASSES * i + cls) * D + c4);
    }

    float m;
    if constexpr (MANY) {
        m = l_all[0];
        if (j < n_splits) wgt[j] = m;
        for (int c = j + RT_THREADS; c < n_splits; c += RT_THREADS) { const float l = pl[c]; wgt[c] = l; m = fmaxf(m, l); }
        m = wave_max(m);
        if ((j & 63) == 0) red[j >> 6] = m;
        __syncthreads();
        m = red[0];
#pragma unroll
        for (int i = 1; i < RT_THREADS / 64; i++) m = fmaxf(m, red[i]);
    } else {
        m = l_all[0];
#pragma unroll
        for (int i = 1; i < NL; i++) m = fmaxf(m, l_all[i]);
        m = row16_max(m);
    }
    for (int e = 0; e < n_extra; e++) m = fmaxf(m, el[e]);
    if (m == -INFINITY) {                      // nothing visible at all (the same in every thread)
        if (j < D) out[b * o_sb + hq * o_sh + j] = 0;
        if (lse_out && j == 0) lse_out[row] = -INFINITY;
        return;
    }
    // weights: exp(lse - m), 0 for empty partitions (their vectors are undefined)
    auto weight = [&](float l) { return l == -INFINITY ? 0.f : __expf(l - m); };
    float den = 0.f, dcl = 0.f;                // (dcl: weights of this thread's row class)
    float4 a4 = {0.f, 0.f, 0.f, 0.f};
    auto add = [&](float w, const float4& v) {
        if constexpr (MANY) dcl += w;
        if (w != 0.f) { a4.x += w * v.x; a4.y += w * v.y; a4.z += w * v.z; a4.w += w * v.w; }
    };
    if constexpr (MANY) {
        for (int c = j; c < n_splits; c += RT_THREADS) wgt[c] = weight(wgt[c]);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NB; i++) add(wgt[RT_CLASSES * i + cls], pv[i]);      // (more than 16 partitions)
        for (int c = RT_CLASSES * NB + cls; c < n_splits; c += RT_CLASSES) add(wgt[c], *(const float4*)(po + (size_t)c * D));
        if ((j & 31) == 0) dsum[cls] = dcl;
    } else {
#pragma unroll
        for (int i = 0; i < NL; i++) den += weight(l_all[i]);
        den = row16_sum(den);
#pragma unroll
        for (int i = 0; i < NB; i++) add(weight(l_own[i]), pv[i]);
        for (int c = RT_CLASSES * NB + cls; c < n_splits; c += RT_CLASSES) add(weight(pl[c]), *(const float4*)(po + (size_t)c * D));
    }
    *(float4*)&cls_sum[cls][c4] = a4;
    float acce = 0.f;
    if (j < D)
        for (int e = 0; e < n_extra; e++) {
            float l = el[e];
            if (l == -INFINITY) continue;
            float w = __expf(l - m);
            den += w;
            acce += w * (e == 0 ? x0 : extra_out[(row * n_extra + e) * D + j]);
        }
    __syncthreads();
    // the classes are added pairwise in a fixed order
    auto fold = [&](const float (*t)[D], int col) {
        float s[RT_CLASSES];
#pragma unroll
        for (int i = 0; i < RT_CLASSES; i++) s[i] = t[i][col];
#pragma unroll
        for (int w = RT_CLASSES / 2; w >= 1; w >>= 1)
#pragma unroll
            for (int i = 0; i < w; i++) s[i] = s[2 * i] + s[2 * i + 1];
        return s[0];
    };
    float res = 0.f;
    if (j < D) {
        if constexpr (MANY) {
            float ds[RT_CLASSES];
#pragma unroll
            for (int i = 0; i < RT_CLASSES; i++) ds[i] = dsum[i];
#pragma unroll
            for (int w = RT_CLASSES / 2; w >= 1; w >>= 1)
#pragma unroll
                for (int i = 0; i < w; i++) ds[i] = ds[2 * i] + ds[2 * i + 1];
            den += ds[0];
        }
        res = fold(cls_sum, j);
    }
    if (unrotate) {
        if (j < D) vec[j] = res;
        __syncthreads();                       // also: every read of cls_sum above is done
        float4 r4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < D / RT_CLASSES; i++) {
            const float x = vec[RT_CLASSES * i + cls];
            r4.x += x * rv[i].x; r4.y += x * rv[i].y; r4.z += x * rv[i].z; r4.w += x * rv[i].w;
        }
        *(float4*)&cls_sum[cls][c4] = r4;
        __syncthreads();
        if (j < D) res = fold(cls_sum, j);
    }
    if (j < D) {
        out[b * o_sb + hq * o_sh + j] = bgtq_f2h((res + acce) / den);
        if (lse_out && j == 0) lse_out[row] = m + __logf(den);
    }
}


// ---- dense fp16 partial over the sink + recent-window tokens ------------------
constexpr int WT = WINDOW_THREADS;
__global__ __launch_bounds__(WT) void window_attn_generic_kernel(
    const uint16_t* q, int64_t q_sb, int64_t q_sh, int bf16,
    const uint16_t* kbuf, const uint16_t* vbuf, int64_t w_sb, int64_t w_sh, int64_t w_st,
    const int32_t* lens, int W, int n_q, int gqa, float scale, float* part_out, float* part_lse) {
    extern __shared__ float wlog[];            // [W] logits, then weights
    __shared__ float q_s[D];
    __shared__ float red[WT / 64];
    const int tid = threadIdx.x;
    const int hq = blockIdx.x, b = blockIdx.y, h = hq / gqa;
    const int n = lens ? min(lens[b], W) : W;
    const size_t row = (size_t)b * n_q + hq;
    if (tid < D) q_s[tid] = bgtq_h2f(bgtq_in16(q[b * q_sb + hq * q_sh + tid], bf16));
    __syncthreads();
    const uint16_t* kb = kbuf + b * w_sb + h * w_sh;
    const uint16_t* vb = vbuf + b * w_sb + h * w_sh;
    float m = -INFINITY;
    for (int t = tid; t < n; t += WT) {
        const uint16_t* kr = kb + (int64_t)t * w_st;
        float acc = 0.f;
        for (int d = 0; d < D; d++) acc += q_s[d] * bgtq_h2f(kr[d]);
        acc *= scale;
        wlog[t] = acc;
        m = fmaxf(m, acc);
    }
    m = wave_max(m);
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    __syncthreads();
    float l = 0.f;
    for (int t = tid; t < n; t += WT) {
        float p = __expf(wlog[t] - m);
        wlog[t] = p;
        l += p;
    }
    l = wave_sum(l);
    if ((tid & 63) == 0) red[tid >> 6] = l;
    __syncthreads();
    l = red[0] + red[1] + red[2] + red[3];
    if (tid < D) {
        float acc = 0.f;
        for (int t = 0; t < n; t++) acc += wlog[t] * bgtq_h2f(vb[(int64_t)t * w_st + tid]);
        part_out[row * D + tid] = n > 0 ? acc / l : 0.f;
    }
    if (tid == 0) part_lse[row] = n > 0 ? m + __logf(l) : -INFINITY;
}


// The same partial for buffers whose rows start on 16-byte boundaries (window_attn_block)
template <int HG>
__global__ __launch_bounds__(WT) void window_attn_kernel(WindowArgs a) {
    extern __shared__ float lds[];
    window_attn_block<HG>(a, blockIdx.x, blockIdx.y, lds);
}

// ---- with-buffer append: the token in ring slot slot[b] leaves, this step's token enters -----
// One work-group per (KV head, batch row), thread j moves dim j of K and of V.  A slot outside
// [0, W) moves nothing and leaves zeros in the outputs.
__global__ __launch_bounds__(D) void window_swap_kernel(
    uint16_t* kbuf, uint16_t* vbuf, int64_t w_sb, int64_t w_sh, int64_t w_st,
    const uint16_t* new_k, const uint16_t* new_v, int64_t nk_sb, int64_t nk_sh, int64_t nv_sb, int64_t nv_sh, int bf16,
    const int32_t* slot, int W, int n_kv, uint16_t* old_k, uint16_t* old_v) {
    const int j = threadIdx.x, h = blockIdx.x, b = blockIdx.y;
    const int sl = slot[b];
    const int64_t o = ((int64_t)b * n_kv + h) * D + j;
    if (sl < 0 || sl >= W) { old_k[o] = 0; old_v[o] = 0; return; }
    const int64_t at = b * w_sb + h * w_sh + (int64_t)sl * w_st + j;
    const uint16_t nk = bgtq_in16(new_k[b * nk_sb + h * nk_sh + j], bf16), nv = bgtq_in16(new_v[b * nv_sb + h * nv_sh + j], bf16);
    old_k[o] = kbuf[at];
    old_v[o] = vbuf[at];
    kbuf[at] = nk;
    vbuf[at] = nv;
}

int launch_window_attn(const WindowArgs& a, int B, int n_kv, hipStream_t st) {
    const int64_t gqa = a.gqa;
    if (!window_wide(a)) {
        hipLaunchKernelGGL(window_attn_generic_kernel, dim3((unsigned)(n_kv * gqa), (unsigned)B), dim3(WT), (size_t)std::max(a.W, 1) * sizeof(float), st,
                           a.q, a.q_sb, a.q_sh, a.bf16, a.kbuf, a.vbuf, a.w_sb, a.w_sh, a.w_st, a.lens, a.W, a.n_q, a.gqa, a.scale, a.part_out, a.part_lse);
        return bgtq_launch_status();
    }
    const dim3 grid((unsigned)n_kv, (unsigned)B);
    if (window_rides(a))
        hipLaunchKernelGGL(window_attn_kernel<4>, grid, dim3(WT), window_lds_floats<4>(a.W) * sizeof(float), st, a);
    else
        hipLaunchKernelGGL(window_attn_kernel<1>, grid, dim3(WT), window_lds_floats<1>(a.W) * sizeof(float), st, a);
    return bgtq_launch_status();
}

int launch_window_swap(void* kbuf, void* vbuf, int64_t w_sb, int64_t w_sh, int64_t w_st,
                       const void* new_k, const void* new_v, int64_t nk_sb, int64_t nk_sh, int64_t nv_sb, int64_t nv_sh,
                       int bf16, const int32_t* slot, int W, int B, int n_kv, void* old_k, void* old_v, hipStream_t st) {
    hipLaunchKernelGGL(window_swap_kernel, dim3((unsigned)n_kv, (unsigned)B), dim3(D), 0, st,
                       (uint16_t*)kbuf, (uint16_t*)vbuf, w_sb, w_sh, w_st, (const uint16_t*)new_k, (const uint16_t*)new_v,
                       nk_sb, nk_sh, nv_sb, nv_sh, bf16, slot, W, n_kv, (uint16_t*)old_k, (uint16_t*)old_v);
    return bgtq_launch_status();
}

}  // namespace

static int g_decode_path = 0;
static int g_last_path = 0;      // kernel the last attention call ran: 1 layout-agnostic, 2 MFMA

// ---- partition results of bgtq_decode_attend_static ------------------------------------------
// The partial vectors and log-sum-exps of the entry point that allocates nothing live in
// this array: one copy per GPU the library runs on, held until the process ends.  Host code
// never uses the array's name as an address; it asks the runtime once per device for the
// device address of that GPU's copy and passes that to the kernels.
static __device__ __align__(256) unsigned char scratch[BGTQ_STATIC_SCRATCH_BYTES];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[MAX_DEVICES];        // device address of `scratch` on device i, once known

// Device address of the current device's scratch array (asked for on the first call on
// that device, with that device current).
int scratch_of_current_device(void** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= MAX_DEVICES) return BGTQ_ELIMIT;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return (int)e;
        if (!p) return BGTQ_EINVAL;
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return BGTQ_OK;
}
// Partitions per (row, KV head).  A work-group keeps a compute unit busy, so what a launch takes is its rounds of 256
// work-groups times (set-up and merge + tiles of a partition), in units of one tile at a work-group's full rate
// (0.4 to 0.5 us); set-up and merge are worth 12 of them.  Only counts that just fill some number of rounds are
// looked at, and a partition has at least 128 tokens.  The merge takes 0.01 to 0.02 us a partition (512 threads), 0.1 to 0.2 where
// 128-thread work-groups queue up; two fifths or two thirds of MERGE choose alike for all but 15 of 24 000 shapes.  One work-group too
// many costs a round:
//   12 rows x 4 heads, 3001 tokens: 6 partitions (288 work-groups) 32.6 us a step, 5 (240) 26.0
//   20 rows x 8 heads, 8k tokens:   2 (320) 105 us, 3 (480, two full rounds) 81
// Rows of different lengths (the lengths are on the device): half of the longest on average, and where there are several
// rounds the long partitions stick out behind the last one by some 0.65 of their length.
//   8 rows x 2 heads, up to 32k tokens: 64 partitions (four rounds) 48.7 us a step, 16 33.0
//   32 rows x 8 heads, up to 16k: 1 (one round) 144, 3 124, 4 121, 8 140; up to 4k: 1 50, 4 61
int pick_splits(int B, int n_kv, int max_T, bool ragged) {
    if (B <= 0 || n_kv <= 0 || max_T <= 0) return 1;
    constexpr float FIXED = 12.f, MEAN = 0.53f, TAIL = 0.65f, MERGE = 1.f / 16.f;
    const int64_t pairs = (int64_t)B * n_kv;
    const int tiles = max_T / 64 + (max_T % 64 != 0);
    const int most = std::min(max_T / 128 + (max_T % 128 != 0), (int)BGTQ_MAX_SPLITS);
    int best = 1;
    float best_cost = INFINITY;
    for (int round = 1; round <= 8; round++) {
        const int n = (int)std::max<int64_t>(1, std::min<int64_t>(most, 256 * round / pairs));
        const int64_t rounds = (pairs * n + 255) / 256;
        const float part = (float)((tiles + n - 1) / n);
        const float cost = MERGE * n + (!ragged || rounds == 1 ? rounds * (FIXED + part) : rounds * (FIXED + MEAN * part) + TAIL * part);
        if (cost < best_cost) { best = n; best_cost = cost; }
    }
    return best;
}

int decode_attn(const bgtq_head_plan* plans,
                const void* q_rot, int64_t q_sb, int64_t q_sh,
                const void* k_packed, int64_t kp_sb, int64_t kp_sh, int64_t kp_st, int k_row_width,
                const void* k_norms, int64_t kn_sb, int64_t kn_sh, int64_t kn_st,
                const void* v_packed, int64_t vp_sb, int64_t vp_sh, int64_t vp_st, int v_row_width,
                const void* v_norms, int64_t vn_sb, int64_t vn_sh, int64_t vn_st,
                const int32_t* seq_lens, int T,
                int B, int n_kv, int gqa, int n_splits,
                float* partial_out, float* partial_lse,
                int k_layout, int v_layout, float scale, const int32_t* row_order, void* stream) {
    BGTQ_CHECK_ARG(plans && q_rot && k_packed && k_norms && v_packed && v_norms);
    BGTQ_CHECK_ARG(partial_out && partial_lse);
    BGTQ_CHECK_ARG(B >= 0 && n_kv >= 0 && T >= 0);
    BGTQ_CHECK_ARG(gqa >= 1 && gqa <= BGTQ_MAX_GQA);
    BGTQ_CHECK_ARG(k_layout == BGTQ_K_BITPACKED || k_layout == BGTQ_K_MIXED);
    BGTQ_CHECK_ARG(v_layout == BGTQ_V_BITPACKED || v_layout == BGTQ_V_NIBBLE || v_layout == BGTQ_V_NIBBLE4);
    if (n_splits > BGTQ_MAX_SPLITS) return BGTQ_ELIMIT;
    BGTQ_CHECK_ARG(n_splits >= 1);
    if (B == 0 || n_kv == 0) return BGTQ_OK;
    DecodeArgs a{};
    a.plans = plans;
    a.q = (const uint16_t*)q_rot; a.q_sb = q_sb; a.q_sh = q_sh;
    a.kp = (const uint8_t*)k_packed; a.kp_sb = kp_sb; a.kp_sh = kp_sh; a.kp_st = kp_st;
    a.kn = (const uint16_t*)k_norms; a.kn_sb = kn_sb; a.kn_sh = kn_sh; a.kn_st = kn_st;
    a.vp = (const uint8_t*)v_packed; a.vp_sb = vp_sb; a.vp_sh = vp_sh; a.vp_st = vp_st;
    a.vn = (const uint16_t*)v_norms; a.vn_sb = vn_sb; a.vn_sh = vn_sh; a.vn_st = vn_st;
    a.seq_lens = seq_lens; a.T = T;
    a.B = B; a.n_kv = n_kv; a.gqa = gqa; a.n_splits = n_splits;
    a.part_out = partial_out; a.part_lse = partial_lse;
    a.k_layout = k_layout; a.v_layout = v_layout; a.scale = scale;
    BGTQ_CHECK_ARG(k_row_width >= 1 && k_row_width <= BGTQ_D);
    BGTQ_CHECK_ARG(v_row_width >= 1 && v_row_width <= BGTQ_D / 2);
    a.k_row_width = k_row_width; a.v_row_width = v_row_width;
    hipStream_t st = (hipStream_t)stream;
    if (g_decode_path != 1) {
        int rc = bgtq_launch_decode_seg(a, row_order, st);
        if (rc != BGTQ_EUNSUPPORTED) { g_last_path = 2; return rc; }
        if (g_decode_path == 2) return rc;        // forced fast path: report why it refused
    }
    g_last_path = 1;
    if (gqa <= 4) return launch_generic<4>(a, st);
    if (gqa <= 8) return launch_generic<8>(a, st);
    return launch_generic<16>(a, st);
}

}  // namespace

extern "C" {

int bgtq_last_decode_path(void) { return g_last_path; }

int bgtq_set_decode_path(int path) {
    if (path < 0 || path > 2) return BGTQ_EINVAL;
    g_decode_path = path;
    return BGTQ_OK;
}

size_t bgtq_workspace_bytes(int B, int n_q, int n_splits) {
    if (B <= 0 || n_q <= 0 || n_splits <= 0) return 0;
    return (size_t)B * n_q * n_splits * (D + 1) * sizeof(float);
}

int bgtq_default_splits(int B, int n_kv, int max_T) { return pick_splits(B, n_kv, max_T, false); }

int bgtq_ragged_splits(int B, int n_kv, int max_T) { return pick_splits(B, n_kv, max_T, true); }

int bgtq_decode_attn(const bgtq_head_plan* plans,
                     const void* q_rot, int64_t q_sb, int64_t q_sh,
                     const void* k_packed, int64_t kp_sb, int64_t kp_sh, int64_t kp_st, int k_row_width,
                     const void* k_norms, int64_t kn_sb, int64_t kn_sh, int64_t kn_st,
                     const void* v_packed, int64_t vp_sb, int64_t vp_sh, int64_t vp_st, int v_row_width,
                     const void* v_norms, int64_t vn_sb, int64_t vn_sh, int64_t vn_st,
                     const int32_t* seq_lens, int T,
                     int B, int n_kv, int gqa, int n_splits,
                     float* partial_out, float* partial_lse,
                     int k_layout, int v_layout, float scale, void* stream) {
    return decode_attn(plans, q_rot, q_sb, q_sh, k_packed, kp_sb, kp_sh, kp_st, k_row_width, k_norms, kn_sb, kn_sh, kn_st,
                       v_packed, vp_sb, vp_sh, vp_st, v_row_width, v_norms, vn_sb, vn_sh, vn_st, seq_lens, T, B, n_kv, gqa,
                       n_splits, partial_out, partial_lse, k_layout, v_layout, scale, nullptr, stream);
}

int bgtq_lse_reduce(const bgtq_head_plan* plans,
                    const float* partial_out, const float* partial_lse, int n_splits,
                    const float* extra_out, const float* extra_lse, int n_extra,
                    int B, int n_kv, int gqa, int unrotate,
                    void* out, int64_t o_sb, int64_t o_sh,
                    float* lse_out, void* stream) {
    BGTQ_CHECK_ARG(plans && partial_out && partial_lse && out);
    BGTQ_CHECK_ARG(B >= 0 && n_kv >= 0 && gqa >= 1 && n_splits >= 1 && n_extra >= 0);
    BGTQ_CHECK_ARG(n_extra == 0 || (extra_out && extra_lse));
    // the kernel reads the partial vectors and the plan 16 bytes at a time
    BGTQ_CHECK_ARG(((uintptr_t)partial_out & 15) == 0 && ((uintptr_t)plans & 15) == 0);
    if (n_splits > BGTQ_MAX_SPLITS) return BGTQ_ELIMIT;
    if (B == 0 || n_kv == 0) return BGTQ_OK;
    const bool few = (int64_t)B * n_kv * gqa <= 256, many = n_splits > merge_held(few ? 512 : 128);
    auto kern = few ? (many ? lse_reduce_kernel<512, true> : lse_reduce_kernel<512, false>)
                    : (many ? lse_reduce_kernel<128, true> : lse_reduce_kernel<128, false>);
    hipLaunchKernelGGL(kern, dim3((unsigned)gqa, (unsigned)n_kv, (unsigned)B),
                       dim3(few ? 512 : 128), 0, (hipStream_t)stream, plans, partial_out, partial_lse, n_extra ? extra_lse : nullptr,
                       n_splits, n_kv * gqa, gqa, unrotate, n_extra, n_extra ? extra_out : nullptr, (uint16_t*)out, o_sb, o_sh, lse_out);
    return bgtq_launch_status();
}

int bgtq_decode_attend_static(const bgtq_head_plan* plans,
                              const void* q_rot, int64_t q_sb, int64_t q_sh,
                              const void* k_packed, int64_t kp_sb, int64_t kp_sh, int64_t kp_st, int k_row_width,
                              const void* k_norms, int64_t kn_sb, int64_t kn_sh, int64_t kn_st,
                              const void* v_packed, int64_t vp_sb, int64_t vp_sh, int64_t vp_st, int v_row_width,
                              const void* v_norms, int64_t vn_sb, int64_t vn_sh, int64_t vn_st,
                              const int32_t* seq_lens, int T,
                              int B, int n_kv, int gqa, int n_splits,
                              int k_layout, int v_layout, float scale, int unrotate,
                              void* out, int64_t o_sb, int64_t o_sh, float* lse_out, void* stream) {
    BGTQ_CHECK_ARG(out);
    BGTQ_CHECK_ARG(B >= 0 && n_kv >= 0 && gqa >= 1 && gqa <= BGTQ_MAX_GQA);
    if (n_splits <= 0) {
        n_splits = bgtq_default_splits(B, n_kv, T > 0 ? T : 1);
        // (no more than one round of them where more would not fit the array)
        const int64_t pairs = (int64_t)B * n_kv;
        if (n_splits > 1 && pairs > 0 && bgtq_workspace_bytes(B, n_kv * gqa, n_splits) > (size_t)BGTQ_STATIC_SCRATCH_BYTES)
            n_splits = (int)std::min<int64_t>(n_splits, std::max<int64_t>(1, 256 / pairs));
    }
    if (n_splits > BGTQ_MAX_SPLITS) return BGTQ_ELIMIT;
    if (B == 0 || n_kv == 0) return BGTQ_OK;
    const size_t rows = (size_t)B * n_kv * gqa * n_splits;         // (batch row, query head, partition)
    if (bgtq_workspace_bytes(B, n_kv * gqa, n_splits) > (size_t)BGTQ_STATIC_SCRATCH_BYTES) return BGTQ_ELIMIT;
    void* base = nullptr;
    int rc = scratch_of_current_device(&base);
    if (rc != BGTQ_OK) return rc;
    float* part_out = (float*)base;                                 // [rows][128], 16-byte aligned
    float* part_lse = part_out + rows * D;                          // [rows]
    rc = bgtq_decode_attn(plans, q_rot, q_sb, q_sh, k_packed, kp_sb, kp_sh, kp_st, k_row_width,
                          k_norms, kn_sb, kn_sh, kn_st, v_packed, vp_sb, vp_sh, vp_st, v_row_width,
                          v_norms, vn_sb, vn_sh, vn_st, seq_lens, T, B, n_kv, gqa, n_splits,
                          part_out, part_lse, k_layout, v_layout, scale, stream);
    if (rc != BGTQ_OK) return rc;
    return bgtq_lse_reduce(plans, part_out, part_lse, n_splits, nullptr, nullptr, 0,
                           B, n_kv, gqa, unrotate, out, o_sb, o_sh, lse_out, stream);
}

int bgtq_window_attn(const void* q, int64_t q_sb, int64_t q_sh,
                     const void* kbuf, const void* vbuf,
                     int64_t w_sb, int64_t w_sh, int64_t w_st,
                     const int32_t* lens, int W,
                     int B, int n_kv, int gqa, float scale,
                     float* part_out, float* part_lse, void* stream) {
    BGTQ_CHECK_ARG(q && kbuf && vbuf && part_out && part_lse);
    BGTQ_CHECK_ARG(B >= 0 && n_kv >= 0 && gqa >= 1 && W >= 0);
    if (W > 8192) return BGTQ_ELIMIT;
    if (B == 0 || n_kv == 0) return BGTQ_OK;
    const WindowArgs a{(const uint16_t*)q, q_sb, q_sh, 0, (const uint16_t*)kbuf, (const uint16_t*)vbuf, w_sb, w_sh, w_st,
                       lens, W, n_kv * gqa, gqa, scale, part_out, part_lse, {}};
    return launch_window_attn(a, B, n_kv, (hipStream_t)stream);
}

int bgtq_window_swap(void* kbuf, void* vbuf, int64_t w_sb, int64_t w_sh, int64_t w_st,
                     const void* new_k, const void* new_v, int64_t n_sb, int64_t n_sh,
                     const int32_t* slot, int W, int B, int n_kv,
                     void* old_k, void* old_v, void* stream) {
    BGTQ_CHECK_ARG(kbuf && vbuf && new_k && new_v && slot && old_k && old_v);
    BGTQ_CHECK_ARG(B >= 0 && n_kv >= 0 && W >= 1);
    if (B == 0 || n_kv == 0) return BGTQ_OK;
    return launch_window_swap(kbuf, vbuf, w_sb, w_sh, w_st, new_k, new_v, n_sb, n_sh, n_sb, n_sh, 0, slot, W, B, n_kv,
                              old_k, old_v, (hipStream_t)stream);
}

int bgtq_decode_step(const bgtq_step* step, void* stream) {
    BGTQ_CHECK_ARG(step);
    bgtq_step s = *step;
    hipStream_t st = (hipStream_t)stream;
    BGTQ_CHECK_ARG(s.B >= 0 && s.n_kv >= 0 && s.S >= 0 && s.gqa >= 1 && s.q && s.out);
    if (s.B == 0 || s.n_kv == 0) return BGTQ_OK;
    const int n_q = s.n_kv * s.gqa;
    const bool windowed = s.win_k != nullptr;
    WindowArgs window{};
    if (windowed) {
        BGTQ_CHECK_ARG(s.S == 1 && s.q_rot && s.win_v && s.win_slot && s.win_lens && s.win_old && s.win_out && s.win_lse);
        BGTQ_CHECK_ARG(s.k && s.v && s.win_W >= 1);
        if (s.win_W > 8192) return BGTQ_ELIMIT;
        window = WindowArgs{(const uint16_t*)s.q, s.q_sb, s.q_sh, s.x_dtype == BGTQ_X_BF16, (const uint16_t*)s.win_k, (const uint16_t*)s.win_v,
                            s.w_sb, s.w_sh, s.w_st, s.win_lens, s.win_W, n_q, s.gqa, s.scale, s.win_out, s.win_lse, {}};
        // small batches: the buffer's partial in the preparation's launch, and the swap as well where the new tokens can be
        // read in the place of their slot
        const WindowSwap swap{s.win_slot, (const uint16_t*)s.k, (const uint16_t*)s.v, s.k_sb, s.k_sh, s.v_sb, s.v_sh};
        const bool rides = s.B <= BGTQ_ONE_LAUNCH_ROWS && window_rides(window);
        uint16_t *old_k = (uint16_t*)s.win_old, *old_v = old_k + (size_t)s.B * s.n_kv * D;
        if (rides && window_swaps(swap)) {
            window.swap = swap;
        } else {
            const int rc = launch_window_swap(s.win_k, s.win_v, s.w_sb, s.w_sh, s.w_st, s.k, s.v, s.k_sb, s.k_sh, s.v_sb, s.v_sh,
                                              s.x_dtype == BGTQ_X_BF16, s.win_slot, s.win_W, s.B, s.n_kv, old_k, old_v, st);
            if (rc != BGTQ_OK) return rc;
        }
        if (!rides) {
            const int rc = launch_window_attn(window, s.B, s.n_kv, st);
            if (rc != BGTQ_OK) return rc;
            window.q = nullptr;
        }
        s.k = old_k; s.v = old_v;
        s.k_sb = s.v_sb = (int64_t)s.n_kv * D; s.k_sh = s.v_sh = D; s.k_ss = s.v_ss = D;
    }
    int32_t* order = bgtq_orders_rows(s.B, s.n_kv, s.S, s.T, s.n_splits, s.seq_lens != nullptr) && bgtq_order_fits(*step) ? (int32_t*)s.out : nullptr;
    int rc = bgtq_step_prepare(s, windowed && s.x_dtype == BGTQ_X_BF16, window.q ? &window : nullptr, order, st);
    if (rc != BGTQ_OK) return rc;
    const void* q = s.q_rot ? s.q_rot : s.q;
    rc = decode_attn(s.plans, q, s.q_rot ? (int64_t)n_q * D : s.q_sb, s.q_rot ? D : s.q_sh,
                          s.k_packed, s.kp_sb, s.kp_sh, s.kp_st, s.k_row_width, s.k_norms, s.kn_sb, s.kn_sh, s.kn_st,
                          s.v_packed, s.vp_sb, s.vp_sh, s.vp_st, s.v_row_width, s.v_norms, s.vn_sb, s.vn_sh, s.vn_st,
                          s.seq_lens, s.T, s.B, s.n_kv, s.gqa, s.n_splits, s.partial_out, s.partial_lse,
                          s.k_layout, s.v_layout, s.scale, order, stream);
    if (rc != BGTQ_OK) return rc;
    return bgtq_lse_reduce(s.plans, s.partial_out, s.partial_lse, s.n_splits, windowed ? s.win_out : nullptr,
                           windowed ? s.win_lse : nullptr, windowed ? 1 : 0, s.B, s.n_kv, s.gqa, 1,
                           s.out, (int64_t)n_q * D, D, nullptr, stream);
}

size_t bgtq_plan_sizeof(void) { return sizeof(bgtq_head_plan); }
int bgtq_abi_version(void) { return 8; }
int bgtq_decode_kernel_revision(void) { return 12; }

const char* bgtq_strerror(int code) {
    switch (code) {
    case BGTQ_OK: return "ok";
    case BGTQ_EINVAL: return "invalid argument";
    case BGTQ_EUNSUPPORTED: return "not supported by this build";
    case BGTQ_ELIMIT: return "size beyond a documented maximum";
    default: return code > 0 ? hipGetErrorString((hipError_t)code) : "unknown error";
    }
}


}  // extern "C"
