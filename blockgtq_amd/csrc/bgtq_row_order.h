// Rows of a decode step by falling length: when a step sends them out so, a row's place, where the order lies meanwhile.
// No device types: it compiles for the CPU alone as well.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include "../../include/bgtq.h"

// Rows (batch x new tokens) up to which a step's append and query rotation are one launch
constexpr int BGTQ_ONE_LAUNCH_ROWS = 64;

// Whether a step sends rows of different lengths out by falling length (ranked in the launch that prepares the step): where
// there is more than one round of work-groups, the long partitions first and the short ones into the places that come free.
// The same partitions, the same results.  us a step (captured), rows as they come and in order; lengths even from T / 16 to T, and all T:
//   64 rows x 8 heads, T 3000, 1 partition:  65.3, 54.8; 68.5, 69.1     64 x 8, 1500, 1: 50.7, 48.4; 52.8, 53.4
//   64 x 2, 12000, 4:                        51.7, 42.1; 56.1, 56.5     24 x 8, 6000, 4: 52.3, 50.0; 57.6, 58.2
//   40 x 4, 3000, 3:                         33.0, 30.9; 34.6, 35.4     24 x 4, 6000, 5: 35.0, 32.8; 37.0, 37.8
// The ranking and a dependent read at every work-group's start cost 0 to 1 us, which equal rows do not get back.  Short partitions
// give too little for it: 40 x 8, 700 (11 tiles) 32.3, 31.6; 36.0, 36.3, but 40 x 8, 300 (5 tiles) 24.4, 24.6; 25.3, 25.6, so these
// go as they come.  (Fewer partitions would do for rows in order, 32 x 8 of up to 16k 90.2 us with two for 94.5 with four; other
// partitions mean other roundings.)
inline bool bgtq_orders_rows(int B, int n_kv, int S, int T, int n_splits, bool ragged) {
    constexpr int64_t SHORTEST = 8, TILE = 64;
    // (a step without new tokens is a launch of any number of rows)
    return ragged && B > 1 && S >= 1 && (int64_t)B * S <= BGTQ_ONE_LAUNCH_ROWS && (int64_t)B * n_kv * n_splits > 256 &&
           T > (SHORTEST - 1) * TILE * n_splits;
}

// Place of row i of n by falling length, equal rows as they come
__host__ __device__ inline int bgtq_row_rank(const int* lens, int n, int i) {
    int rank = 0;
    for (int j = 0; j < n; j++) rank += lens[j] > lens[i] || (lens[j] == lens[i] && j < i) ? 1 : 0;
    return rank;
}

// The order lies at the start of the step's output, which nothing else writes before the partitions are merged.  It is written
// while the step's inputs and scratch are in use, and the attention takes what it finds there for batch rows: not where any other
// buffer of the step has a byte there (`out` over the queries or over scratch is allowed, the merge is the last to use them), nor
// where that is not plain (strides that run backwards), nor where the order would not be aligned.
inline bool bgtq_order_fits(const bgtq_step& s) {
    const int64_t B = s.B, n_kv = s.n_kv, n_q = n_kv * s.gqa, D = BGTQ_HEAD_DIM;
    const uintptr_t lo = (uintptr_t)s.out, hi = lo + (size_t)B * sizeof(int32_t);
    auto apart = [&](const void* p, int64_t bytes) { return !p || bytes <= 0 || (uintptr_t)p >= hi || (uintptr_t)p + (size_t)bytes <= lo; };
    // B x n x m rows of `last` elements
    auto rows_apart = [&](const void* p, int64_t size, int64_t sb, int64_t n, int64_t sh, int64_t m, int64_t ss, int64_t last) {
        return sb >= 0 && sh >= 0 && ss >= 0 && apart(p, m < 1 ? 0 : ((B - 1) * sb + (n - 1) * sh + (m - 1) * ss + last) * size);
    };
    const int64_t rows = s.T > s.max_T ? s.T : s.max_T;
    if ((lo & 3) != 0 || !apart(s.plans, n_kv * (int64_t)sizeof(bgtq_head_plan))) return false;
    if (!rows_apart(s.q, 2, s.q_sb, n_q, s.q_sh, 1, 0, D) || !rows_apart(s.k, 2, s.k_sb, n_kv, s.k_sh, s.S, s.k_ss, D) ||
        !rows_apart(s.v, 2, s.v_sb, n_kv, s.v_sh, s.S, s.v_ss, D) || !apart(s.q_rot, B * n_q * D * 2)) return false;
    if (!rows_apart(s.k_packed, 1, s.kp_sb, n_kv, s.kp_sh, rows, s.kp_st, s.k_row_width) ||
        !rows_apart(s.k_norms, 2, s.kn_sb, n_kv, s.kn_sh, rows, s.kn_st, s.norm_width) ||
        !rows_apart(s.v_packed, 1, s.vp_sb, n_kv, s.vp_sh, rows, s.vp_st, s.v_row_width) ||
        !rows_apart(s.v_norms, 2, s.vn_sb, n_kv, s.vn_sh, rows, s.vn_st, 1)) return false;
    if (!apart(s.t_pos, B * 4) || !apart(s.seq_lens, B * 4) || !apart(s.partial_out, B * n_q * s.n_splits * D * 4) ||
        !apart(s.partial_lse, B * n_q * s.n_splits * 4)) return false;
    if (!s.win_k) return true;                                // (the other fields of the buffer are not read then)
    return rows_apart(s.win_k, 2, s.w_sb, n_kv, s.w_sh, s.win_W, s.w_st, D) && rows_apart(s.win_v, 2, s.w_sb, n_kv, s.w_sh, s.win_W, s.w_st, D) &&
           apart(s.win_slot, B * 4) && apart(s.win_lens, B * 4) && apart(s.win_old, 2 * B * n_kv * D * 2) &&
           apart(s.win_out, B * n_q * D * 4) && apart(s.win_lse, B * n_q * 4);
}
