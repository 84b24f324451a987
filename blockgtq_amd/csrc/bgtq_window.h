// Dense fp16 attention partial over the sink and recent-window tokens: one work-group's part, shared by the kernel of its
// own (bgtq_decode.hip) and the launch that prepares a decode step (bgtq_encode.hip).
#pragma once
#include "bgtq_common.h"

constexpr int WINDOW_THREADS = 256;

__device__ inline float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ inline float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// sum over the 16 lanes of a row, in every lane of it (rotations within the row: no LDS traffic)
__device__ __forceinline__ float row16_sum(float x) {
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x128, 0xf, 0xf, false));
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x124, 0xf, 0xf, false));
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x122, 0xf, 0xf, false));
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x121, 0xf, 0xf, false));
    return x;
}

struct WindowArgs {
    const uint16_t* q; int64_t q_sb, q_sh; int bf16;
    const uint16_t *kbuf, *vbuf; int64_t w_sb, w_sh, w_st;
    const int32_t* lens; int W, n_q, gqa; float scale;
    float *part_out, *part_lse;
};

// LDS floats of one work-group: sums, maxima and denominators, then HG rows of W scores
template <int HG>
constexpr size_t window_lds_floats(size_t W) { return (size_t)(WINDOW_THREADS / 64) * HG * BGTQ_D + 2 * HG + HG * W; }

// rows and query vectors on 16-byte boundaries
inline bool window_wide(const WindowArgs& a) {
    return (((uintptr_t)a.q | (uintptr_t)a.kbuf | (uintptr_t)a.vbuf) & 15) == 0 && ((a.q_sb | a.q_sh | a.w_sb | a.w_sh | a.w_st) & 7) == 0;
}
// four heads at a time, in at most 57 KB of LDS
constexpr int WINDOW_RIDE_W = 3072;
inline bool window_rides(const WindowArgs& a) { return window_wide(a) && a.gqa > 1 && a.W <= WINDOW_RIDE_W; }

// For buffers whose rows start on 16-byte boundaries (the manager's do): one
// work-group per (batch row, KV head) serves all its query heads, HG at a time, so the window is
// read once per HG heads, and every load is contiguous across the wave.  Scores: 16 lanes share a
// token (8 dims each, one 16-byte load), 4 tokens per wave instruction; values: a wave covers
// one token row per load (2 dims a lane), the four waves take every fourth token and their sums
// meet in LDS.  wlog holds HG rows of W scores, then weights.
template <int HG>
__device__ __forceinline__ void window_attn_block(const WindowArgs& a, const int h, const int b, float* lds) {
#pragma clang fp contract(fast)
    constexpr int D = BGTQ_D, WT = WINDOW_THREADS, NW = WT / 64;
    float (*osum)[HG][D] = (float (*)[HG][D])lds;
    float *red_m = lds + NW * HG * D, *red_l = red_m + HG, *wlog = red_l + HG;      // wlog [HG][W]
    const uint16_t* q = a.q;
    const int64_t q_sb = a.q_sb, q_sh = a.q_sh, w_sb = a.w_sb, w_sh = a.w_sh, w_st = a.w_st;
    const int bf16 = a.bf16, W = a.W, n_q = a.n_q, gqa = a.gqa;
    const int32_t* lens = a.lens;
    const uint16_t *kbuf = a.kbuf, *vbuf = a.vbuf;
    const float scale = a.scale;
    float *part_out = a.part_out, *part_lse = a.part_lse;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lens ? min(lens[b], W) : W;
    const uint16_t* kb = kbuf + b * w_sb + h * w_sh;
    const uint16_t* vb = vbuf + b * w_sb + h * w_sh;
    const int sub = lane & 15, tq = lane >> 4;  // scores: dim chunk and token within a wave load
    // Loads run one batch ahead of the arithmetic that uses them (a batch waited for on the spot
    // costs a trip to memory each); small batches in rolled loops measured as fast as large
    // unrolled ones.
    constexpr int SB = 3;                       // score passes (4 tokens per wave each) per batch
    constexpr int PB = 8;                       // value rows per batch
    auto fetch_k = [&](uint4 (&k4)[SB], const int t0) {
#pragma unroll
        for (int u = 0; u < SB; u++) {
            const int t = t0 + u * 4 * NW + tq;
            k4[u] = uint4{0, 0, 0, 0};
            if (t < n) k4[u] = *(const uint4*)(kb + (int64_t)t * w_st + sub * 8);
        }
    };
    auto fetch_v = [&](uint32_t (&vv)[PB], const int t0) {
#pragma unroll
        for (int u = 0; u < PB; u++) {
            const int t = t0 + u * NW;
            vv[u] = t < n ? *(const uint32_t*)(vb + (int64_t)t * w_st + 2 * lane) : 0u;
        }
    };
    for (int g0 = 0; g0 < gqa; g0 += HG) {
        const int ng = min(HG, gqa - g0);
        // ---- scores: 16 lanes share a token ------------------------------------------------
        float qf[HG][8];
#pragma unroll
        for (int g = 0; g < HG; g++) {
            uint4 w4 = {0, 0, 0, 0};
            if (g < ng) w4 = *(const uint4*)(q + b * q_sb + (int64_t)(h * gqa + g0 + g) * q_sh + sub * 8);
            const uint32_t ws[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                qf[g][2 * i] = bgtq_h2f(bgtq_in16((uint16_t)(ws[i] & 0xFFFFu), bf16)) * scale;
                qf[g][2 * i + 1] = bgtq_h2f(bgtq_in16((uint16_t)(ws[i] >> 16), bf16)) * scale;
            }
        }
        uint4 kc[SB], kn[SB];
        uint32_t vc[PB], vn[PB];
        fetch_k(kc, wave * 4);
        fetch_v(vc, wave);                      // the first value rows do not wait for the scores
#pragma unroll 1
        for (int t0 = wave * 4; t0 < n; t0 += SB * 4 * NW) {
            fetch_k(kn, t0 + SB * 4 * NW);
#pragma unroll
            for (int u = 0; u < SB; u++) {
                const int t = t0 + u * 4 * NW + tq;
                const uint32_t ks[4] = {kc[u].x, kc[u].y, kc[u].z, kc[u].w};
                float kf[8];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    kf[2 * i] = bgtq_h2f((uint16_t)(ks[i] & 0xFFFFu));
                    kf[2 * i + 1] = bgtq_h2f((uint16_t)(ks[i] >> 16));
                }
#pragma unroll
                for (int g = 0; g < HG; g++) {
                    float acc = 0.f;
#pragma unroll
                    for (int i = 0; i < 8; i++) acc += qf[g][i] * kf[i];
                    acc = row16_sum(acc);
                    if (sub == 0 && t < n && g < ng) wlog[g * W + t] = acc;
                }
            }
#pragma unroll
            for (int u = 0; u < SB; u++) kc[u] = kn[u];
        }
        __syncthreads();
        // ---- softmax weights: wave w owns heads w, w + 4, ... ----------------------------------
        for (int g = wave; g < ng; g += NW) {
            float mm = -INFINITY;
            for (int t = lane; t < n; t += 64) mm = fmaxf(mm, wlog[g * W + t]);
            mm = wave_max(mm);
            float ll = 0.f;
            for (int t = lane; t < n; t += 64) {
                const float p = __expf(wlog[g * W + t] - mm);
                wlog[g * W + t] = p;
                ll += p;
            }
            ll = wave_sum(ll);
            if (lane == 0) { red_m[g] = mm; red_l[g] = ll; }
        }
        __syncthreads();
        // ---- values: wave w takes tokens w, w + 4, ...; lane = dims 2 lane, 2 lane + 1 -------
        float o0[HG], o1[HG];
#pragma unroll
        for (int g = 0; g < HG; g++) o0[g] = o1[g] = 0.f;
#pragma unroll 1
        for (int t0 = wave; t0 < n; t0 += PB * NW) {
            fetch_v(vn, t0 + PB * NW);
            float pw[PB][HG];                   // the batch's weights, read together
#pragma unroll
            for (int u = 0; u < PB; u++)
#pragma unroll
                for (int g = 0; g < HG; g++) {
                    const int t = min(t0 + u * NW, n - 1);
                    pw[u][g] = wlog[min(g, ng - 1) * W + t];
                }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < PB; u++) {
                const bool live = t0 + u * NW < n;
                const float v0 = bgtq_h2f((uint16_t)(vc[u] & 0xFFFFu)), v1 = bgtq_h2f((uint16_t)(vc[u] >> 16));
#pragma unroll
                for (int g = 0; g < HG; g++) {
                    const float p = (g < ng && live) ? pw[u][g] : 0.f;
                    o0[g] += p * v0;
                    o1[g] += p * v1;
                }
            }
#pragma unroll
            for (int u = 0; u < PB; u++) vc[u] = vn[u];
        }
#pragma unroll
        for (int g = 0; g < HG; g++) { osum[wave][g][2 * lane] = o0[g]; osum[wave][g][2 * lane + 1] = o1[g]; }
        __syncthreads();
        for (int i = tid; i < ng * D; i += WT) {
            const int g = i / D, d = i - g * D;
            const float acc = (osum[0][g][d] + osum[1][g][d]) + (osum[2][g][d] + osum[3][g][d]);
            const size_t row = (size_t)b * n_q + h * gqa + g0 + g;
            const float mg = red_m[g], lg = red_l[g];
            part_out[row * D + d] = n > 0 ? acc / lg : 0.f;
            if (d == 0) {                      // (ln lg = log2 lg * ln 2 with ln 2 in two parts; spelled out, so that both files round alike)
                const float y = __builtin_amdgcn_logf(lg);
                part_lse[row] = n > 0 ? mg + __builtin_fmaf(y, 0.693147182f, y * -1.90465430e-9f) : -INFINITY;
            }
        }
        __syncthreads();                        // wlog, red_* and osum are reused by the next heads
    }
}

