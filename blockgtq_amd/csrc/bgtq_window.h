// Dense fp16 attention partial over the sink and recent-window tokens: one work-group's part, shared by the kernel of its
// own (bgtq_decode.hip) and the launch that prepares a decode step (bgtq_encode.hip).
#pragma once
#include <type_traits>

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

__device__ __forceinline__ float row16_max(float x) {
    x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x128, 0xf, 0xf, false)));
    x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x124, 0xf, 0xf, false)));
    x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x122, 0xf, 0xf, false)));
    x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x121, 0xf, 0xf, false)));
    return x;
}

// The token that enters the buffer in this step (slot[b], nothing where that lies outside [0, W)), where the launch itself
// puts it there: the attention takes that row from the new tokens whatever the slot holds by then.
struct WindowSwap {
    const int32_t* slot;
    const uint16_t *k, *v; int64_t k_sb, k_sh, v_sb, v_sh;      // of the type of q
};

struct WindowArgs {
    const uint16_t* q; int64_t q_sb, q_sh; int bf16;
    const uint16_t *kbuf, *vbuf; int64_t w_sb, w_sh, w_st;
    const int32_t* lens; int W, n_q, gqa; float scale;
    float *part_out, *part_lse;
    WindowSwap swap;         // slot null: the buffer holds the new token already
};

// LDS floats of one work-group: sums, maxima and denominators, then HG rows of W scores
template <int HG>
constexpr size_t window_lds_floats(size_t W) { return (size_t)(WINDOW_THREADS / 64) * HG * BGTQ_D + 2 * HG + HG * W; }

// rows and query vectors on 16-byte boundaries, rows of a (batch row, head) within 32 bits
inline bool window_wide(const WindowArgs& a) {
    return (((uintptr_t)a.q | (uintptr_t)a.kbuf | (uintptr_t)a.vbuf) & 15) == 0 && ((a.q_sb | a.q_sh | a.w_sb | a.w_sh | a.w_st) & 7) == 0 &&
           a.w_st >= 0 && a.w_st * (a.W + 4) < (int64_t)1 << 32;
}
// four heads at a time, in at most 57 KB of LDS
constexpr int WINDOW_RIDE_W = 3072;
inline bool window_rides(const WindowArgs& a) { return window_wide(a) && a.gqa > 1 && a.W <= WINDOW_RIDE_W; }
// new tokens that the attention can read in the place of their slot
inline bool window_swaps(const WindowSwap& s) {
    return (((uintptr_t)s.k | (uintptr_t)s.v) & 15) == 0 && ((s.k_sb | s.k_sh | s.v_sb | s.v_sh) & 7) == 0;
}

// For buffers whose rows start on 16-byte boundaries (the manager's do): one
// work-group per (batch row, KV head) serves all its query heads, HG at a time, so the window is
// read once per HG heads, and every load is contiguous across the wave.  Scores: 16 lanes share a
// token (8 dims each, one 16-byte load), 4 tokens per wave instruction; values: a wave covers
// one token row per load (2 dims a lane), the four waves take every fourth token and their sums
// meet in LDS.  wlog holds HG scores a token, then weights.
// SWAP: a.swap names this step's tokens.
template <int HG, bool SWAP = false>
__device__ __forceinline__ void window_attn_block(const WindowArgs& a, const int h, const int b, float* lds) {
#pragma clang fp contract(fast)
    constexpr int D = BGTQ_D, WT = WINDOW_THREADS, NW = WT / 64;
    float (*osum)[HG][D] = (float (*)[HG][D])lds;
    float *red_m = lds + NW * HG * D, *red_l = red_m + HG, *wlog = red_l + HG;      // wlog [W][HG]
    const uint16_t* q = a.q;
    const int64_t q_sb = a.q_sb, q_sh = a.q_sh, w_sb = a.w_sb, w_sh = a.w_sh, w_st = a.w_st;
    const int bf16 = a.bf16, W = a.W, n_q = a.n_q, gqa = a.gqa;
    const int32_t* lens = a.lens;
    const uint16_t *kbuf = a.kbuf, *vbuf = a.vbuf;
    const float scale = a.scale;
    float *part_out = a.part_out, *part_lse = a.part_lse;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lens ? min(lens[b], W) : W;
    const uint16_t* kb = kbuf + b * w_sb + h * w_sh;
    const uint16_t* vb = vbuf + b * w_sb + h * w_sh;
    const int slot = SWAP ? a.swap.slot[b] : -1;              // (outside [0, W): never a token's number)
    const int sub = lane & 15, tq = lane >> 4;  // scores: dim chunk and token within a wave load
    // Loads run two batches ahead of the arithmetic that uses them, in three sets of registers that take turns (moving
    // a batch from one to another waits for it): with one batch ahead every batch cost a trip to memory, 5.6 of a
    // work-group's 13.3 us for the values of 132 tokens and 4.7 for the scores beside 768 work-groups that load as well.
    constexpr int SB = 3;                       // score passes (4 tokens per wave each) per batch
    constexpr int PB = 12;                      // value rows per batch
    // (rows are uniform across the wave: scalar addresses, one lane offset.  The first row's number is opaque, or every
    // row of three batches would become a pointer of its own that lives through the loop)
    const uint32_t step = (uint32_t)w_st, k_lane = (uint32_t)tq * step + sub * 8;
    auto fetch_k = [&](uint4 (&k4)[SB], int t0) {
        asm volatile("" : "+s"(t0));
#pragma unroll
        for (int u = 0; u < SB; u++) {
            const int t = t0 + u * 4 * NW;
            k4[u] = uint4{0, 0, 0, 0};
            if (t + tq < n) k4[u] = *(const uint4*)(kb + (uint32_t)t * step + k_lane);
        }
    };
    auto fetch_v = [&](uint32_t (&vv)[PB], int t0) {
        asm volatile("" : "+s"(t0));
#pragma unroll
        for (int u = 0; u < PB; u++) {
            const int t = t0 + u * NW;
            vv[u] = t < n ? *(const uint32_t*)(vb + (uint32_t)t * step + 2 * lane) : 0u;
        }
    };
    // SWAP: this lane's part of the new token's rows; what is read from its slot (the old token or the new one) is not used
    uint32_t own_k[4] = {0, 0, 0, 0}, own_v = 0;
    if constexpr (SWAP) {
        const uint4 k4 = *(const uint4*)(a.swap.k + b * a.swap.k_sb + h * a.swap.k_sh + sub * 8);
        own_k[0] = k4.x; own_k[1] = k4.y; own_k[2] = k4.z; own_k[3] = k4.w;
        own_v = *(const uint32_t*)(a.swap.v + b * a.swap.v_sb + h * a.swap.v_sh + 2 * lane);
        auto as16 = [&](uint32_t x) { return (uint32_t)bgtq_in16((uint16_t)x, bf16) | ((uint32_t)bgtq_in16((uint16_t)(x >> 16), bf16) << 16); };
#pragma unroll
        for (int i = 0; i < 4; i++) own_k[i] = as16(own_k[i]);
        own_v = as16(own_v);
    }
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
        constexpr int SSTEP = SB * 4 * NW, PSTEP = PB * NW;
        uint4 kr[3][SB];
        uint32_t vr[3][PB];
#pragma unroll
        for (int i = 0; i < 2; i++) fetch_k(kr[i], wave * 4 + i * SSTEP);
#pragma unroll
        for (int i = 0; i < 2; i++) fetch_v(vr[i], wave + i * PSTEP);      // the first value rows do not wait for the scores
        auto scores = [&](const uint4 (&kc)[SB], const int t0) {
#pragma unroll
            for (int u = 0; u < SB; u++) {
                const int t = t0 + u * 4 * NW + tq;
                uint32_t ks[4] = {kc[u].x, kc[u].y, kc[u].z, kc[u].w};
                if (SWAP && slot - (t - tq) >= 0 && slot - (t - tq) < 4) {          // (uniform)
#pragma unroll
                    for (int i = 0; i < 4; i++) ks[i] = t == slot ? own_k[i] : ks[i];
                }
                float kf[8];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    kf[2 * i] = bgtq_h2f((uint16_t)(ks[i] & 0xFFFFu));
                    kf[2 * i + 1] = bgtq_h2f((uint16_t)(ks[i] >> 16));
                }
                float acc[HG];
#pragma unroll
                for (int g = 0; g < HG; g++) {
                    acc[g] = 0.f;
#pragma unroll
                    for (int i = 0; i < 8; i++) acc[g] += qf[g][i] * kf[i];
                    acc[g] = row16_sum(acc[g]);
                }
                if (sub == 0 && t < n)
#pragma unroll
                    for (int g = 0; g < HG; g++) wlog[t * HG + g] = acc[g];        // (of heads past the last: not looked at)
            }
        };
#pragma unroll 1
        for (int t0 = wave * 4; t0 < n; t0 += 3 * SSTEP)
#pragma unroll
            for (int i = 0; i < 3; i++) {
                fetch_k(kr[(i + 2) % 3], t0 + (i + 2) * SSTEP);
                __builtin_amdgcn_sched_barrier(0);
                if (t0 + i * SSTEP < n) scores(kr[i], t0 + i * SSTEP);     // (uniform)
                __builtin_amdgcn_sched_barrier(0);
            }
        __syncthreads();
        // ---- softmax weights: wave w owns heads w, w + 4, ... ----------------------------------
        for (int g = wave; g < ng; g += NW) {
            float mm = -INFINITY;
            for (int t = lane; t < n; t += 64) mm = fmaxf(mm, wlog[t * HG + g]);
            mm = wave_max(mm);
            float ll = 0.f;
            for (int t = lane; t < n; t += 64) {
                const float p = __expf(wlog[t * HG + g] - mm);
                wlog[t * HG + g] = p;
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
        auto values = [&](uint32_t (&vc)[PB], const int t0) {
            // (uniform; a row behind the visible ones stays zeros: what is masked below is a product with it)
            if (SWAP && slot >= t0 && slot < min(t0 + PSTEP, n) && (slot - t0) % NW == 0) {
#pragma unroll
                for (int u = 0; u < PB; u++) vc[u] = t0 + u * NW == slot ? own_v : vc[u];
            }
            // (FULL: a wave alone issues an instruction every ten clocks or so; what is not masked is a third less of them)
            auto add = [&](auto full) {
                constexpr bool FULL = decltype(full)::value;
                float pw[PB][HG];                   // the batch's weights, read together
#pragma unroll
                for (int u = 0; u < PB; u++)
#pragma unroll
                    for (int g = 0; g < HG; g++) pw[u][g] = wlog[(FULL ? t0 + u * NW : min(t0 + u * NW, n - 1)) * HG + g];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < PB; u++) {
                    const bool live = FULL || t0 + u * NW < n;
                    const float v0 = bgtq_h2f((uint16_t)(vc[u] & 0xFFFFu)), v1 = bgtq_h2f((uint16_t)(vc[u] >> 16));
#pragma unroll
                    for (int g = 0; g < HG; g++) {
                        const float p = FULL || (g < ng && live) ? pw[u][g] : 0.f;
                        o0[g] += p * v0;
                        o1[g] += p * v1;
                    }
                }
            };
            if (ng == HG && t0 + (PB - 1) * NW < n) add(std::true_type{}); else add(std::false_type{});
        };
#pragma unroll 1
        for (int t0 = wave; t0 < n; t0 += 3 * PSTEP)
#pragma unroll
            for (int i = 0; i < 3; i++) {
                fetch_v(vr[(i + 2) % 3], t0 + (i + 2) * PSTEP);
                __builtin_amdgcn_sched_barrier(0);
                if (t0 + i * PSTEP < n) values(vr[i], t0 + i * PSTEP);     // (uniform)
                __builtin_amdgcn_sched_barrier(0);
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

