// Prompt-phase attention with a workspace (gfx950): records staged once, then a plain matrix-core attention.
//
// bgtq_prefill_attn dequantises every tile in every work-group that sees it, 128 times over for an 8k prompt of 8
// query heads a KV head, and that is half of its time.  Here three kernels share the work:
//
//   stage   every 64-token tile is dequantised once into 32 KB of the workspace, already in the order in which
//           the attention's waves read their matrix operands (a fragment is 64 lanes x 16 bytes that follow each
//           other), so that a tile travels to LDS as it lies and every LDS read is a contiguous kilobyte.  The
//           query rotation and the value un-rotation of a head are split here into fp16 (bf16 for bf16 queries)
//           parts in operand order, too.
//   attend  NW waves, 32 query rows each: 32 NW / gqa tokens of every query head of the group.  The rows
//           are rotated at the start and un-rotated at the end inside the kernel, on the same matrix cores.
//           S^T = K Q^T puts one query in each lane, so softmax statistics stay in the lane, and P goes from the
//           score registers straight into O^T = V^T P^T.  Where an accumulator serves as an operand again (rotated
//           queries, probabilities, outputs), the contraction index is permuted: slot 16 s + 8 g + e of a 32-block
//           holds index 16 s + 8 (e / 4) + 4 g + e % 4, which is where half-wave g keeps its register 8 s + e.
//   merge   only where a few query rows meet a long context: the tiles of a query block are dealt to several
//           work-groups, whose unnormalised sums this kernel adds and un-rotates.
//
// Arithmetic: fp16(centroid * norm) records, fp16 rotated queries and probabilities, fp32 sums (the denominator from
// the fp32 exponentials).  The query rotation counts with its fp32 values whole: three 16-bit parts of an entry add up to
// it, their products with 16-bit queries are exact and summed in fp32.  The un-rotation takes two fp16 parts of either
// factor, as bgtq_prefill_attn does: an error of 2^-22 of the largest terms, ahead of a rounding to fp16 (2^-11).
//
// Reference behaviour: blockgtq/prefill.py:66-101, blockgtq/kernels/fused_packed_attention.py:1876-2594.
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "bgtq_dequant_tile.h"

namespace {

typedef float float16v __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int D = BGTQ_D;
constexpr int MT = DQ_MT;
constexpr int PROMPT_BIG = 2048;             // work-groups of 256 rows from which on they are taken
constexpr int MAX_GQA_ROWS = 128;            // query rows of the smaller work-group, the most query heads of a group
constexpr int TILE = 2 * MT * D * 2;         // bytes of a staged tile: K fragments, then V fragments
constexpr int PART = D * D * 2;              // bytes of one 16-bit part of a rotation
constexpr float REFRESH = 4.0f;

// rotation parts of a head: the query rotation (3 parts in the type of the queries), then the un-rotation (2 fp16 parts)
constexpr int Q_PARTS = 3, HEAD_PARTS = Q_PARTS + 2;
// fp16 has no exponents for what a head leaves over (an entry of 0.01 and its remainders span 2^-7 to 2^-31): every
// remainder is held 2^11 times as large as it is, which is about the size of the head
constexpr float F16_STEP = 2048.f;

__device__ __forceinline__ uint32_t cvt_pk_f16(float lo, float hi) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    h2 r = {(_Float16)lo, (_Float16)hi};
    return __builtin_bit_cast(uint32_t, r);
}

// ---- stage ------------------------------------------------------------------------------------------------
struct StageArgs {
    const bgtq_head_plan* plans;
    const uint8_t* kp;  int64_t kp_sb, kp_sh;
    const uint16_t* kn; int64_t kn_sb, kn_sh; int kn_st;
    const uint8_t* vp;  int64_t vp_sb, vp_sh;
    const uint16_t* vn; int64_t vn_sb, vn_sh;
    int n_kv, pairs, T, n_tiles, per_wg;     // (row, head) pairs, tiles of one, how many of them a work-group takes
    int k_layout, v_layout, k_row_width, v_stride;
    int kt, knr, vnr, vt;                    // raw tile areas in LDS
    int bf16, rotate_q;                      // parts of the query rotation: bf16 / fp16, or none
    uint8_t *rot, *tiles;
};

__host__ __device__ inline int raw_bytes(int krow, int vstride, int kn_st, int& kt, int& knr, int& vnr, int& vt) {
    kt = (MT * krow + 32 + 15) & ~15;
    knr = (MT * kn_st * 2 + 16 + 15) & ~15;
    vnr = MT * 2 + 16;
    vt = (MT * vstride + 32 + 15) & ~15;
    return kt + knr + vnr + vt;
}
constexpr int ROT_WGS = D * D / 8 / DQ_THR;   // work-groups per head that split its rotations, the first of the launch
constexpr int RAW_OFF = BGTQ_VLUT_BYTES + BGTQ_LUT_IMAGE_BYTES;

// One head's rotation parts.  A fragment (rows 32 ob .., step kk) holds, for lane (li, lg), row 32 ob + li and
// slots 16 kk + 8 lg + e.  Query rotation: row = packed dim, slot = original dim.  Un-rotation: row = output dim,
// slot s = rotated dim in the permuted order.
__device__ __forceinline__ void stage_rotations(const StageArgs& a, int wg, int tid, uint8_t* smem) {
    const int h = wg / ROT_WGS;
    const bgtq_head_plan& P = a.plans[h];
    int* inv = (int*)smem;                   // original dim -> packed dim
    if (tid < D) inv[P.head_perm[tid]] = tid;
    __syncthreads();
    uint8_t* dst = a.rot + (size_t)h * HEAD_PARTS * PART;
    {
        const int i = (wg - h * ROT_WGS) * DQ_THR + tid;           // piece of 8 slots
        const int lane = i & 63, kk = (i >> 6) & 7, ob = i >> 9, li = lane & 31, lg = lane >> 5;
        const int row = 32 * ob + li;
        if (a.rotate_q) {
            uint16_t part[Q_PARTS][8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                float x = P.k_rot_T[inv[16 * kk + 8 * lg + e] * D + row];
#pragma unroll
                for (int p = 0; p < Q_PARTS; p++) {              // (differences and powers of two: exact)
                    if (a.bf16) {
                        const __bf16 v = (__bf16)x;
                        part[p][e] = __builtin_bit_cast(uint16_t, v);
                        x -= (float)v;
                    } else {
                        const _Float16 v = (_Float16)x;
                        part[p][e] = __builtin_bit_cast(uint16_t, v);
                        x = (x - (float)v) * F16_STEP;
                    }
                }
            }
#pragma unroll
            for (int p = 0; p < Q_PARTS; p++) *(uint4v*)(dst + p * PART + i * 16) = *(const uint4v*)part[p];
        }
        uint16_t hi[8], lo[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float x = P.v_rot[(16 * kk + 8 * (e >> 2) + 4 * lg + (e & 3)) * D + row];
            const _Float16 p0 = (_Float16)x, p1 = (_Float16)(x - (float)p0);
            hi[e] = __builtin_bit_cast(uint16_t, p0);
            lo[e] = __builtin_bit_cast(uint16_t, p1);
        }
        *(uint4v*)(dst + Q_PARTS * PART + i * 16) = *(const uint4v*)hi;
        *(uint4v*)(dst + (Q_PARTS + 1) * PART + i * 16) = *(const uint4v*)lo;
    }
}

// One set of raw records: two work-groups share a compute unit (at most 78 KB of LDS each) and one's loads run under the
// other's lookups.  With two sets a work-group was alone there, and 292 of them (4100 records of 8 heads) took two rounds.
// 4100 records of 8 heads: 19.9 -> 12.2 us, 4 x 8192 of 2 heads 26.9 -> 18.2 (a large copy or merge in front of each).
// Bound by the loads and lookups of a tile, one behind the other.  Work-groups are numbered as the attention's are, (row, head)
// fastest: with 8 pairs an XCD then writes the tiles it will read, and that it read in the call before.  Tiles that lie in
// the L2 of another XCD, from a call just ended in the same workspace, made it 16.0 us (12.6 with 66 MB copied in between, which
// drives them out); 11.1 now, 11.4 behind the copy.
__global__ __launch_bounds__(DQ_THR) void prompt_stage_kernel(StageArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n_rot = ROT_WGS * a.n_kv;
    if ((int)blockIdx.x < n_rot) { stage_rotations(a, (int)blockIdx.x, tid, smem); return; }
    const int part = ((int)blockIdx.x - n_rot) / a.pairs, pair = (int)blockIdx.x - n_rot - part * a.pairs;
    const int tile0 = part * a.per_wg, tile1 = min(tile0 + a.per_wg, a.n_tiles);
    const int b = pair / a.n_kv, h = pair - b * a.n_kv;
    const bgtq_head_plan& P = a.plans[h];
    const bool vnib = a.v_layout == BGTQ_V_NIBBLE;
    const int krow = a.k_row_width, vrow = a.v_stride, kn_st = a.kn_st;
    const uint32_t voff = (uint32_t)lane * 16;
    const uint32_t kraw = RAW_OFF, knraw = kraw + a.kt, vnraw = knraw + a.knr, vraw = vnraw + a.vnr, ktile = vraw + a.vt, vtile = ktile + MT * DQ_KROW;
    const uint8_t* kp_base = a.kp + b * a.kp_sb + h * a.kp_sh;
    const uint8_t* vp_base = a.vp + b * a.vp_sb + h * a.vp_sh;
    const uint8_t* kn_base = (const uint8_t*)(a.kn + b * a.kn_sb + h * a.kn_sh);
    const uint8_t* vn_base = (const uint8_t*)(a.vn + b * a.vn_sb + h * a.vn_sh);
    const uint32_t kph = (uint32_t)((uintptr_t)kp_base & 15), vph = (uint32_t)((uintptr_t)vp_base & 15);
    const uint32_t knph = (uint32_t)((uintptr_t)kn_base & 15), vnph = (uint32_t)((uintptr_t)vn_base & 15);
    // wave 0 fetches the K records, wave 1 the V records, wave 2 both norm arrays
    auto issue = [&](int tile) {
        const int t = tile * MT, nt = min(MT, a.T - t);
        if (wave == 0) {
            dma_region<9>(kp_base - kph + (int64_t)t * krow, kraw, dma_shape((int)kph + nt * krow, voff), voff);
        } else if (wave == 1) {
            dma_region<9>(vp_base - vph + (int64_t)t * vrow, vraw, dma_shape((int)vph + nt * vrow, voff), voff);
        } else if (wave == 2) {
            dma_region<2>(kn_base - knph + (int64_t)t * kn_st * 2, knraw, dma_shape((int)knph + nt * kn_st * 2, voff), voff);
            dma_region<1>(vn_base - vnph + (int64_t)t * 2, vnraw, dma_shape((int)vnph + nt * 2, voff), voff);
        }
    };
    issue(tile0);
    dq_load_tables(P, a.k_layout, vnib, vnib ? 4 : (int)P.v_bits, wave, voff);
    TileDequant dq;
    dq.init(P, a.k_layout, vnib, tid);
    // the K tile's columns of 0-bit dims are never written: zero them once
    const int n_zero = min(max(P.n_zero_dims, 0), D);
    for (int i = tid; i < MT * (n_zero / 2); i += DQ_THR) {
        const int t = i / (n_zero / 2), c = i - t * (n_zero / 2);
        lds_put<uint32_t>(ktile + (uint32_t)t * DQ_KROW + c * 4, 0u);
    }
    const int li = lane & 31, lg = lane >> 5;
    uint8_t* out = a.tiles + (size_t)pair * a.n_tiles * TILE + voff;
    for (int tile = tile0; tile < tile1; tile++) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();                     // raw tile (and tables) complete; the tile buffers have been read
        dq.run(kraw + kph + (uint32_t)lane * krow, knraw + knph + (uint32_t)lane * kn_st * 2, vnraw + vnph, vraw + vph, vrow,
               min(MT, a.T - tile * MT), ktile, vtile);
        __syncthreads();
        if (tile + 1 < tile1) issue(tile + 1);                   // (the raw tile has been read)
        uint8_t* o = out + (size_t)tile * TILE;
#pragma unroll
        for (int c = 0; c < 2; c++) {        // K fragment (token block tb, step kk = wave); dims in the permuted order
            const uint32_t src = ktile + (uint32_t)(32 * c + li) * DQ_KROW + (uint32_t)(16 * wave + 4 * lg) * 2;
            const uint2v x0 = lds_at<uint2v>(src), x1 = lds_at<uint2v>(src + 16);
            *(uint4v*)(o + (8 * c + wave) * 1024) = (uint4v){x0.x, x0.y, x1.x, x1.y};
        }
#pragma unroll
        for (int c = 0; c < 2; c++) {        // V fragment f = (16-token group f / 4, dims 32 (f % 4) ..)
            const int f = 2 * wave + c;
            *(uint4v*)(o + 16384 + f * 1024) = lds_at<uint4v>(vtile + (uint32_t)(32 * (f & 3) + li) * DQ_VTROW + (uint32_t)(16 * (f >> 2) + 8 * lg) * 2);
        }
    }
}

// ---- attend -----------------------------------------------------------------------------------------------
struct PromptArgs {
    const uint8_t *rot, *tiles;
    const uint16_t* q; int64_t q_sb, q_sh, q_ss;
    int n_kv, gqa, S, T, n_tiles, q_pos_offset, causal, n_splits;
    float scale;
    int rotate_q, unrotate;
    int rows, n_qb;                          // query rows per work-group (32 a wave), blocks of them
    float *part_o, *part_ml;                 // n_splits > 1: sums [wg][wave][register / 4][lane][4], (reference, denominator) [wg][wave][row]
    uint16_t* out; int64_t o_sb, o_sh, o_ss;
};

// LDS of four waves' attention: two staged tiles; two parts of a rotation take their place before and after the walk
constexpr size_t PROMPT_LDS = 2 * TILE;
static_assert(2 * PART <= PROMPT_LDS, "");

// Which rows a wave holds: row r = wave * 32 + (lane & 31) of the block is head r / BQ, token s0 + r % BQ.
struct RowOf {
    int hq, sq, s0;
    bool ok;
    __device__ __forceinline__ RowOf(const PromptArgs& a, int qb, int wave, int lane) {
        const int BQ = a.rows / a.gqa, row = wave * 32 + (lane & 31);
        s0 = qb * BQ;
        hq = row / BQ;
        sq = s0 + row - hq * BQ;
        ok = hq < a.gqa && sq < a.S;
    }
};

// n consecutive rotation parts from the workspace to LDS address dst: each wave its share
template <int NW>                                               // (waves that take part, `wave` counts through them)
__device__ __forceinline__ void load_parts(const uint8_t* src, int n, int wave, uint32_t voff, uint32_t dst = 0) {
    for (int c = wave; c < n * (PART / 4096); c += NW) dma_full<4>(voff, uniform_ptr(src + c * 4096), dst + (uint32_t)c * 4096);
}

// Normalise, un-rotate (out^T = R^T O^T: both factors split into fp16 head and remainder, the product of the
// remainders left out) and store.  The parts lie in LDS.
__device__ __forceinline__ void finish_rows(const PromptArgs& a, float16v (&O)[4], float l_tot, const RowOf& row, int b, int h, int lane) {
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
#pragma unroll
    for (int db = 0; db < 4; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) O[db][r] *= inv;
    const int lg = lane >> 5;
    uint32_t frag = (uint32_t)lane * 16;
    asm("" : "+v"(frag));
    if (a.unrotate) {
        half8 Bh[8], Bl[8];
#pragma unroll
        for (int db = 0; db < 4; db++)
#pragma unroll
            for (int s = 0; s < 2; s++) {
                uint32_t hi[4], lo[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float x0 = O[db][8 * s + 2 * j], x1 = O[db][8 * s + 2 * j + 1];
                    const _Float16 h0 = (_Float16)x0, h1 = (_Float16)x1;
                    hi[j] = cvt_pk_f16((float)h0, (float)h1);
                    lo[j] = cvt_pk_f16(x0 - (float)h0, x1 - (float)h1);
                }
                Bh[2 * db + s] = __builtin_bit_cast(half8, (uint4v){hi[0], hi[1], hi[2], hi[3]});
                Bl[2 * db + s] = __builtin_bit_cast(half8, (uint4v){lo[0], lo[1], lo[2], lo[3]});
            }
#pragma unroll
        for (int ob = 0; ob < 4; ob++) O[ob] = (float16v){0};
#pragma unroll
        for (int st = 0; st < 8; st++) {                       // four independent accumulators per pass
            half8 Ah[4], Al[4];
#pragma unroll
            for (int ob = 0; ob < 4; ob++) {
                Ah[ob] = lds_at<half8>(frag + (8 * ob + st) * 1024);
                Al[ob] = lds_at<half8>(frag + PART + (8 * ob + st) * 1024);
            }
#pragma unroll
            for (int ob = 0; ob < 4; ob++) O[ob] = __builtin_amdgcn_mfma_f32_32x32x16_f16(Ah[ob], Bh[st], O[ob], 0, 0, 0);
#pragma unroll
            for (int ob = 0; ob < 4; ob++) O[ob] = __builtin_amdgcn_mfma_f32_32x32x16_f16(Al[ob], Bh[st], O[ob], 0, 0, 0);
#pragma unroll
            for (int ob = 0; ob < 4; ob++) O[ob] = __builtin_amdgcn_mfma_f32_32x32x16_f16(Ah[ob], Bl[st], O[ob], 0, 0, 0);
        }
    }
    if (row.ok) {
        uint16_t* orow = a.out + b * a.o_sb + ((int64_t)h * a.gqa + row.hq) * a.o_sh + (int64_t)row.sq * a.o_ss;
#pragma unroll
        for (int ob = 0; ob < 4; ob++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint2v w = {cvt_pk_f16(O[ob][4 * j], O[ob][4 * j + 1]), cvt_pk_f16(O[ob][4 * j + 2], O[ob][4 * j + 3])};
                *(uint2v*)(orow + 32 * ob + 8 * j + 4 * lg) = w;
            }
    }
}

// TEAMS 2: two teams of NW waves hold the same rows and walk one half of the partition's tiles each, in LDS of their own;
// their sums meet in LDS.  That takes the place of two work-groups on a compute unit with a partition each, and of a launch
// that reads their sums back (33 MB and 14 us for 1000 queries over 4100 records of 8 heads; the attention itself takes longer,
// since its first and last part wait for the slower team: the call 97.5 -> 96.4 us).
// Turns: with one barrier a tile the two waves of a SIMD fell into step, both at their exponentials and then both at the value
// products.  A second barrier after the exponentials, and one team (one half of eight waves) half a tile behind: the same
// 1000 queries 96.4 -> 94.2 us, 28 heads of 1000 queries 39.1 -> 37.8 (43.2 with partitions and a merge), 4 x 8k prompts
// 1113 -> 1100 (the clock is down to 1.75 GHz there: the matrix cores are busy 60 % of the cycles).
constexpr int prompt_ring(int nw) { return nw == 8 ? 4 : 2; }    // tiles in LDS, for each team
constexpr size_t prompt_lds(int nw, int teams) { return teams * prompt_ring(nw) * TILE + (teams > 1 ? nw * 64 * 8 : 0); }
template <bool BF16, int NW, int TEAMS>
__global__ __launch_bounds__(64 * NW * TEAMS, 2) void prompt_attn_kernel(PromptArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6), team = TEAMS == 1 ? 0 : wave_all / NW, wave = wave_all - team * NW;
    const uint32_t lds0 = (uint32_t)team * (uint32_t)PROMPT_LDS;
    const int h = blockIdx.x, b = blockIdx.y;
    // the query block that sees most tokens first, so that the short blocks fill the tail of the launch
    const int nz = (int)gridDim.z - 1 - (int)blockIdx.z, qb = nz / a.n_splits, c = nz - qb * a.n_splits;
    const RowOf row(a, qb, wave, lane);
    const int lg = lane >> 5;
    const int s_last = min(row.s0 + a.rows / a.gqa, a.S) - 1;
    const int t_end = a.causal ? min(a.T, a.q_pos_offset + s_last + 1) : a.T;
    const int n_all = (t_end + MT - 1) / MT;
    const int parts = a.n_splits * TEAMS, mine = c * TEAMS + team;
    const int tile0 = (int)((int64_t)n_all * mine / parts), tile1 = (int)((int64_t)n_all * (mine + 1) / parts);
    const int n_full = min(tile1, (a.causal ? min(a.T, a.q_pos_offset + row.s0 + 1) : a.T) / MT);   // tiles before this one are seen whole by every row
    const int lim = !row.ok ? a.T : a.causal ? min(a.T, a.q_pos_offset + row.sq + 1) : a.T;    // tokens t < lim are visible to this row
    const bool live = __builtin_amdgcn_ballot_w64(row.ok) != 0;                              // (a wave without rows only moves data)
    // the two waves of a SIMD take turns: while one computes scores and exponentials, the other, `late` by half a tile, adds up values.
    // The half of eight waves that is not late moves the tiles, into the third and fourth place while the late ones read two.
    constexpr bool TURNS = TEAMS > 1 || NW == 8;
    constexpr int RING = prompt_ring(NW), MOVERS = TEAMS == 1 && NW == 8 ? NW / 2 : NW;
    const bool late = TURNS && (TEAMS > 1 ? team == 1 : wave >= NW / 2), mover = MOVERS == NW || !late;

    const uint32_t voff = (uint32_t)lane * 16;
    const uint8_t* rot_h = a.rot + (size_t)h * HEAD_PARTS * PART;
    const uint8_t* tiles = a.tiles + (size_t)(b * a.n_kv + h) * a.n_tiles * TILE + wave * (TILE / 2 / MOVERS);
    // this wave's share of a tile's K or V fragments; tile t lies in place t % RING of the LDS
    auto issue = [&](int tile, int part) {
        constexpr int N = TILE / 2 / MOVERS / 1024;
        if (mover && tile < tile1) dma_full<N>(voff, uniform_ptr(tiles + (size_t)tile * TILE + part), lds0 + (uint32_t)(tile & (RING - 1)) * TILE + part + wave * (TILE / 2 / MOVERS));
    };
    constexpr int K_PART = 0, V_PART = TILE / 2;

    // ---- queries as B operands of S^T = K Q^T, in the permuted order of the staged dims
    half8 Qb[8];
    const uint16_t* qrow = a.q + b * a.q_sb + ((int64_t)h * a.gqa + (row.ok ? row.hq : 0)) * a.q_sh + (int64_t)(row.ok ? row.sq : 0) * a.q_ss;
    if (a.rotate_q) {
        // two parts fit LDS at a time: the remainders first; the head takes the last one's place under the products of the other
        // (1000 fp16 queries over 4100 records of 8 heads: this kernel 74 us with two parts and a denominator from fp16 values, 78 now)
        if (TEAMS == 1) load_parts<NW>(rot_h + PART, 2, wave, voff);
        else load_parts<NW * TEAMS>(rot_h, 3, wave_all, voff);   // (two teams' room holds all three)
        uint4v qv[8];                                            // lane: dims 16 kk + 8 lg .. + 7 of its query
#pragma unroll
        for (int kk = 0; kk < 8; kk++) {
            qv[kk] = (uint4v){0, 0, 0, 0};
            if (row.ok) qv[kk] = *(const uint4v*)(qrow + 16 * kk + 8 * lg);
        }
        float16v R[4];                                           // packed dims 32 ob ..
#pragma unroll
        for (int ob = 0; ob < 4; ob++) R[ob] = (float16v){0};
        auto add_part = [&](uint32_t at) {
            asm("" : "+v"(at));
#pragma unroll
            for (int kk = 0; kk < 8; kk++)
#pragma unroll
                for (int ob = 0; ob < 4; ob++) {
                    if constexpr (BF16)
                        R[ob] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lds_at<bf16x8>(at + (8 * ob + kk) * 1024), __builtin_bit_cast(bf16x8, qv[kk]), R[ob], 0, 0, 0);
                    else
                        R[ob] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lds_at<half8>(at + (8 * ob + kk) * 1024), __builtin_bit_cast(half8, qv[kk]), R[ob], 0, 0, 0);
                }
        };
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        auto step = [&]() {                                      // sums of a part in units of the next larger one
            if constexpr (!BF16) {
#pragma unroll
                for (int ob = 0; ob < 4; ob++)
#pragma unroll
                    for (int r = 0; r < 16; r++) R[ob][r] *= 1.f / F16_STEP;
            }
        };
        if constexpr (TEAMS == 1) {
            if (live) { add_part(PART + voff); step(); }
            __syncthreads();
            load_parts<NW>(rot_h, 1, wave, voff, PART);
            if (live) { add_part(voff); step(); }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (live) add_part(PART + voff);
        } else if (live) {
            add_part(2 * PART + voff);
            step();
            add_part(PART + voff);
            step();
            add_part(voff);
        }
        __syncthreads();
        issue(tile0, K_PART); issue(tile0, V_PART);
#pragma unroll
        for (int ob = 0; ob < 4; ob++)
#pragma unroll
            for (int s = 0; s < 2; s++)
                Qb[2 * ob + s] = __builtin_bit_cast(half8, (uint4v){cvt_pk_f16(R[ob][8 * s], R[ob][8 * s + 1]), cvt_pk_f16(R[ob][8 * s + 2], R[ob][8 * s + 3]),
                                                                    cvt_pk_f16(R[ob][8 * s + 4], R[ob][8 * s + 5]), cvt_pk_f16(R[ob][8 * s + 6], R[ob][8 * s + 7])});
    } else {
#pragma unroll
        for (int kk = 0; kk < 8; kk++) {
            uint2v x0 = {0, 0}, x1 = {0, 0};
            if (row.ok) { x0 = *(const uint2v*)(qrow + 16 * kk + 4 * lg); x1 = *(const uint2v*)(qrow + 16 * kk + 8 + 4 * lg); }
            Qb[kk] = __builtin_bit_cast(half8, (uint4v){x0.x, x0.y, x1.x, x1.y});
        }
        issue(tile0, K_PART); issue(tile0, V_PART);
    }

    const float c2 = a.scale * 1.44269504088896340736f;        // scores in log2 units
    float16v O[4];                                              // O^T: block db = dims 32 db .., reg r -> dim 32 db + 8 (r / 4) + 4 lg + r % 4
#pragma unroll
    for (int db = 0; db < 4; db++) O[db] = (float16v){0};
    float m_ref = -INFINITY, l_part = 0.f, mx = -INFINITY;       // per query (this half's share of the denominator; maximum of the tile at hand)

    // The walk is one tile deep: while a tile's scores become probabilities on the vector unit, the matrix core
    // works on the scores of the next one, and the maximum of those is taken under the value product.  (4 x 8k prompts
    // 1186 -> 1167 us, 1000 queries over 4100 records 122 -> 119, against the same parts one after the other; that was before
    // the two waves of a SIMD took turns, with the matrix cores busy 53 % of the cycles at 1.9 GHz.  The clock gives way to
    // more: 60 % at 1.75 GHz with turns, 980 TFLOP/s, where the library's bf16 product of 8192 x 8192 matrices reaches 1290
    // on the same card.)
    auto frags = [&](int tile) __attribute__((always_inline)) {
        uint32_t at = lds0 + (uint32_t)(tile & (RING - 1)) * TILE + voff;
        asm("" : "+v"(at));                                      // (fragments at immediate offsets: left alone, every address gets an instruction)
        return at;
    };
    // S^T = K Q^T for the wave's 32 queries: 2 token blocks x 8 steps of 16 dims
    auto k_frag = [&](uint32_t at, int i) __attribute__((always_inline)) { return lds_at<half8>(at + (8 * (i & 1) + (i >> 1)) * 1024); };
    // scores past a row's last token go to -inf
    auto mask = [&](float16v (&S)[2], int tile) __attribute__((always_inline)) {
        const int rest = lim - tile * MT - 4 * lg;
#pragma unroll
        for (int tb = 0; tb < 2; tb++)
#pragma unroll
            for (int r = 0; r < 16; r++)                         // reg r of block tb is token t0 + 32 tb + 8 (r / 4) + 4 lg + r % 4
                if (32 * tb + 8 * (r >> 2) + (r & 3) >= rest) S[tb][r] = -INFINITY;
    };
    auto enter = [&](int tile) __attribute__((always_inline)) {
        if (TURNS || tile1 - tile0 > 1) {                        // (a tile alone is complete already)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");    // this wave's share of V of this tile and K of the next
            __syncthreads();                                     // they are complete; everyone is done with the tile before
        }
        issue(tile + 2, K_PART);
        issue(tile + 1, V_PART);
        if (live && __builtin_amdgcn_ballot_w64(mx > m_ref)) {           // wave-uniform, rare after the first tiles
            const float top = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float m_new = top > m_ref ? top + REFRESH : m_ref;
            const float alpha = (m_ref == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m_ref - m_new);
            l_part *= alpha;
#pragma unroll
            for (int db = 0; db < 4; db++)
#pragma unroll
                for (int r = 0; r < 16; r++) O[db][r] *= alpha;
            m_ref = m_new;
        }
    };
    auto change_phase = [&]() __attribute__((always_inline)) {
        if constexpr (TURNS) {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // One straight line of code.  S: scores of this tile, N: those of the next (NEXT: there is one; CUT: it needs the mask)
    auto products = [&](auto NEXT, auto CUT, float16v (&S)[2], float16v (&N)[2], int tile) __attribute__((always_inline)) {
        constexpr bool next = decltype(NEXT)::value;
        // rows that have seen no record yet keep every exponential at 0 (no inf - inf)
        const float mneg = m_ref == -INFINITY ? 0.f : -m_ref;
        const uint32_t kf = frags(tile + 1), vf = frags(tile) + V_PART;
        constexpr int AHEAD = 4;                                  // operands are read so many products before their use
        half8 A[16], V[16];
        uint32_t Pw[16];                                          // fp16 pairs: Pw[j] = regs 2j, 2j + 1 of block j / 8
        if (next) {
#pragma unroll
            for (int i = 0; i < AHEAD; i++) A[i] = k_frag(kf, i);
            N[0] = N[1] = (float16v){0};
        }
        // ---- probabilities (raw scores stay in the registers; the scale goes into the exponent's multiply-add) under the
        // products of the next scores: a pair of exponentials, and the packing of the pair before, with every product
        // (The denominator adds the exponentials as they are: below 2^-14 the rounded ones keep less than 11 bits, and a long
        // tail of those can be a per cent of it.  Tile by tile, because one of them alone vanishes beside the whole sum.)
        float p0 = 0.f, p1 = 0.f, l_tile = 0.f;
        auto pack = [&](int j) __attribute__((always_inline)) {
            Pw[j] = cvt_pk_f16(p0, p1);
            l_tile += p0 + p1;
        };
#pragma unroll
        for (int i = 0; i < 16; i++) {
            if (next) {
                if (i + AHEAD < 16) A[i + AHEAD] = k_frag(kf, i + AHEAD);
            }
            if (i + AHEAD >= 16) V[i + AHEAD - 16] = lds_at<half8>(vf + (i + AHEAD - 16) * 1024);
            if (next) N[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[i], Qb[i >> 1], N[i & 1], 0, 0, 0);
            if (i > 0) pack(i - 1);
            p0 = __builtin_amdgcn_exp2f(fmaf(S[i >> 3][2 * (i & 7)], c2, mneg));
            p1 = __builtin_amdgcn_exp2f(fmaf(S[i >> 3][2 * (i & 7) + 1], c2, mneg));
            if (next) __builtin_amdgcn_sched_barrier(0);
        }
        pack(15);
        l_part += l_tile;
        change_phase();
        // ---- O^T += V^T P^T: 16-token group 2 tb + hf; the maximum of the next scores underneath
        float m = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            if (i + AHEAD < 16) V[i + AHEAD] = lds_at<half8>(vf + (i + AHEAD) * 1024);
            const int g = i >> 2;
            O[i & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(V[i], __builtin_bit_cast(half8, (uint4v){Pw[4 * g], Pw[4 * g + 1], Pw[4 * g + 2], Pw[4 * g + 3]}), O[i & 3], 0, 0, 0);
            if (next) {
                if (i == 3 && decltype(CUT)::value) mask(N, tile + 1);
                if (i >= 4) {
#pragma unroll
                    for (int r = (i - 4) * 4 / 3; r < (i - 3) * 4 / 3; r++) m = fmaxf(fmaxf(m, N[0][r]), N[1][r]);
                    asm volatile("" : "+v"(m));                  // (keeps its place under the products)
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (next) mx = m * c2;                                   // c2 > 0: the maximum commutes with the scale
    };
    if (tile0 < tile1) {
        float16v Sa[2], Sb[2];
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();                                         // the first tile
        issue(tile0 + 1, K_PART);
        Sa[0] = Sa[1] = Sb[0] = Sb[1] = (float16v){0};
        if (live) {
            const uint32_t kf = frags(tile0);
#pragma unroll
            for (int i = 0; i < 16; i++) Sa[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(k_frag(kf, i), Qb[i >> 1], Sa[i & 1], 0, 0, 0);
            mask(Sa, tile0);
#pragma unroll
            for (int r = 0; r < 16; r++) mx = fmaxf(fmaxf(mx, Sa[0][r]), Sa[1][r]);
            mx *= c2;
        }
        if (late) change_phase();
        int tile = tile0;
        if (TURNS && !live) {
            for (; tile + 1 < tile1; tile++) { enter(tile); change_phase(); }
        }
        while ((!TURNS || live) && tile + 2 < n_full) {          // two tiles a round: the two sets of scores change places
            enter(tile);
            if (TURNS || live) products(std::true_type{}, std::false_type{}, Sa, Sb, tile);
            enter(++tile);
            if (TURNS || live) products(std::true_type{}, std::false_type{}, Sb, Sa, tile);
            ++tile;
        }
        for (; tile + 1 < tile1; tile++) {                       // (a wave without rows is past them)
            enter(tile);
            if (TURNS || live) products(std::true_type{}, std::true_type{}, Sa, Sb, tile);
            Sa[0] = Sb[0];
            Sa[1] = Sb[1];
        }
        enter(tile);
        if (live) products(std::false_type{}, std::false_type{}, Sa, Sb, tile);
        else change_phase();
        if (TURNS && !late) change_phase();
    }

    float l_tot = l_part + __shfl_xor(l_part, 32, 64);
    if constexpr (TEAMS > 1) {
        static_assert(TEAMS == 2 && NW * 64 * 64 * 4 <= PROMPT_LDS, "a team's sums fit its tiles");
        // both teams meet as many barriers as the longer walk has (two a tile, and two)
        const int n = tile1 - tile0, longest = (n_all + parts - 1) / parts;
        for (int i = n > 0 ? 2 * n + 2 : 0; i < 2 * longest + 2; i++) __syncthreads();
        __syncthreads();                                         // every wave is done with the tiles
        // the second team's sums in the place of its tiles, [wave][register][lane], (reference, denominator) behind both teams'
        float* sums = (float*)(smem + PROMPT_LDS) + wave * 64 * 64 + lane;
        float2* ml = (float2*)(smem + 2 * PROMPT_LDS) + wave * 64 + lane;
        if (team == 1) {
#pragma unroll
            for (int r = 0; r < 64; r++) sums[r * 64] = O[r >> 4][r & 15];
            *ml = float2{m_ref, l_tot};
        }
        if (a.n_splits == 1 && a.unrotate) {                     // ... the un-rotation in the place of the first team's
            load_parts<NW * TEAMS>(rot_h + Q_PARTS * PART, 2, wave_all, voff);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        __syncthreads();
        if (team == 1) return;
        const float2 y = *ml;
        const float m = fmaxf(m_ref, y.x);
        const float f0 = m_ref == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_ref - m), f1 = y.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(y.x - m);
        l_tot = fmaf(f1, y.y, f0 * l_tot);
#pragma unroll
        for (int r = 0; r < 64; r++) O[r >> 4][r & 15] = fmaf(f1, sums[r * 64], f0 * O[r >> 4][r & 15]);
        m_ref = m;
    }
    if (a.n_splits == 1) {
        if (TEAMS == 1 && a.unrotate) {
            __syncthreads();                                     // every wave is done with the tiles
            load_parts<NW>(rot_h + Q_PARTS * PART, 2, wave, voff);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
        if (live) finish_rows(a, O, l_tot, row, b, h, lane);
    } else if (live) {
        const size_t wg = ((size_t)(b * a.n_kv + h) * a.n_qb + qb) * a.n_splits + c;
        float4* po = (float4*)(a.part_o + (wg * NW + wave) * 64 * 64) + lane;
#pragma unroll
        for (int i = 0; i < 16; i++) po[i * 64] = float4{O[i >> 2][4 * (i & 3)], O[i >> 2][4 * (i & 3) + 1], O[i >> 2][4 * (i & 3) + 2], O[i >> 2][4 * (i & 3) + 3]};
        if (lane < 32) *(float2*)(a.part_ml + ((wg * NW + wave) * 32 + lane) * 2) = float2{m_ref, l_tot};
    }
}

// ---- merge ------------------------------------------------------------------------------------------------
// The partial sums of 32 rows (one wave of the attention) are added by PER waves.  Eight where few rows meet many
// partitions: each wave takes every eighth of them, then the eight meet in LDS.  (One wave walking all of them took 43 us
// for 62 partitions.)  One, and four groups of rows to a work-group, where the groups alone fill the chip and partitions
// are few: 2 partitions of 1024 groups 28.9 us with eight waves a group (four rounds of work-groups that each fetch the
// un-rotation and keep six waves waiting), 13.6 with one.
constexpr int merge_waves(int per) { return per == 1 ? 4 : per; }
constexpr size_t merge_lds(int per) { return 2 * PART + (per == 1 ? 0 : per / 2 * (64 * 64 + 64) * sizeof(float)); }
template <int PER>
__global__ __launch_bounds__(64 * merge_waves(PER)) void prompt_merge_kernel(PromptArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    constexpr int WAVES = merge_waves(PER);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = a.rows / 32;
    const int h = blockIdx.x, b = blockIdx.y;
    const int group = min((int)blockIdx.z * (WAVES / PER) + wave / PER, a.n_qb * nw - 1);   // (a wave past the last group repeats it and stores nothing)
    const bool mine = (int)blockIdx.z * (WAVES / PER) + wave / PER < a.n_qb * nw;
    const int qb = group / nw, w = group - qb * nw, part = wave % PER;
    const RowOf row(a, qb, w, lane);
    if (PER == WAVES && __builtin_amdgcn_ballot_w64(row.ok) == 0) return;                    // (uniform over the work-group)
    if (a.unrotate) load_parts<WAVES>(a.rot + ((size_t)h * HEAD_PARTS + Q_PARTS) * PART, 2, wave, (uint32_t)lane * 16);
    const size_t wg0 = ((size_t)(b * a.n_kv + h) * a.n_qb + qb) * a.n_splits;
    float16v O[4];
#pragma unroll
    for (int db = 0; db < 4; db++) O[db] = (float16v){0};
    float l_tot = 0.f, m = -INFINITY;
    const float2* ml = (const float2*)a.part_ml + (wg0 * nw + w) * 32 + (lane & 31);
    for (int c = 0; c < a.n_splits; c++) m = fmaxf(m, ml[(size_t)c * nw * 32].x);
    for (int c = part; c < a.n_splits; c += PER) {
        const float4* po = (const float4*)(a.part_o + ((wg0 + c) * nw + w) * 64 * 64) + lane;
        float4 x[16];
#pragma unroll
        for (int i = 0; i < 16; i++) x[i] = po[i * 64];
        const float2 y = ml[(size_t)c * nw * 32];
        const float f = y.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(y.x - m);
        l_tot += f * y.y;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            O[i >> 2][4 * (i & 3)] = fmaf(f, x[i].x, O[i >> 2][4 * (i & 3)]);
            O[i >> 2][4 * (i & 3) + 1] = fmaf(f, x[i].y, O[i >> 2][4 * (i & 3) + 1]);
            O[i >> 2][4 * (i & 3) + 2] = fmaf(f, x[i].z, O[i >> 2][4 * (i & 3) + 2]);
            O[i >> 2][4 * (i & 3) + 3] = fmaf(f, x[i].w, O[i >> 2][4 * (i & 3) + 3]);
        }
    }
    float* meet = (float*)(smem + 2 * PART);                     // [PER / 2][64 registers, denominator][lane]
#pragma unroll
    for (int half = PER / 2; half >= 1; half >>= 1) {
        float* at = meet + (part & (half - 1)) * 65 * 64 + lane;
        if (part >= half && part < 2 * half) {
#pragma unroll
            for (int r = 0; r < 64; r++) at[r * 64] = O[r >> 4][r & 15];
            at[64 * 64] = l_tot;
        }
        __syncthreads();
        if (part < half) {
#pragma unroll
            for (int r = 0; r < 64; r++) O[r >> 4][r & 15] += at[r * 64];
            l_tot += at[64 * 64];
        }
        __syncthreads();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // this wave's share of the un-rotation
    __syncthreads();
    if (part == 0 && mine) finish_rows(a, O, l_tot, row, b, h, lane);
}

// Rows of a work-group.  256 (one work-group a compute unit) fetch every tile for twice as many rows, which counts
// where the chip is full and limited by power: 8k prompts 5 % faster.  128 (two a compute unit) fill the chip with half the rows and end with shorter tails: 1k to 2k prompts 5 to 20 % faster.
int prompt_rows(int B, int n_kv, int gqa, int S) {
    return gqa > MAX_GQA_ROWS || (int64_t)B * n_kv * gqa * S >= (int64_t)PROMPT_BIG * 256 ? 256 : 128;
}
// Two teams to a work-group where that deals the tiles into as many parts as work-groups of one team would: 128 rows, and
// twice the partitions that fill the compute units once.  (With an odd number, say 3 partitions of 160 blocks, teams would
// leave compute units idle that the partitions use; where a short context makes fewer, each partition has one to itself.)
int prompt_teams(int64_t wgs, int rows, int ns) { return rows == 128 && ns >= 2 && ns == 2 * (256 / wgs) ? 2 : 1; }
// Tiles of one query block dealt to several work-groups where the blocks alone leave compute units idle, four
// tiles or more each (below that set-up and merge cost more than the walk)
int prompt_splits(int B, int n_kv, int gqa, int S, int T) {
    const int rows = prompt_rows(B, n_kv, gqa, S), BQ = rows / gqa;
    const int64_t wgs = (int64_t)B * n_kv * ((S + BQ - 1) / BQ), room = rows == 256 ? 256 : 512;
    const int64_t want = std::max<int64_t>(1, room / std::max<int64_t>(wgs, 1));
    const int64_t tiles = (T + MT - 1) / MT;
    return (int)std::max<int64_t>(1, std::min(want, tiles / 4));
}

}  // namespace

extern "C" {

size_t bgtq_prompt_workspace_bytes(int B, int n_kv, int gqa, int S, int T) {
    if (B <= 0 || n_kv <= 0 || gqa <= 0 || gqa > 256 || S <= 0 || T <= 0) return 0;
    const int ns = prompt_splits(B, n_kv, gqa, S, T), rows = prompt_rows(B, n_kv, gqa, S), BQ = rows / gqa;
    const size_t blocks = (size_t)B * n_kv * ((S + BQ - 1) / BQ), ng = ns / prompt_teams((int64_t)blocks, rows, ns);
    return (size_t)n_kv * HEAD_PARTS * PART + (size_t)B * n_kv * ((T + MT - 1) / MT) * TILE +
           (ng > 1 ? blocks * ns * (rows / 32) * (64 * 64 + 64) * sizeof(float) : 0);   // (ns: never less than fewer records need)
}

int bgtq_prompt_attn(const bgtq_head_plan* plans,
                     const void* q, int x_dtype, int rotate_q, int64_t q_sb, int64_t q_sh, int64_t q_ss,
                     const void* k_packed, int64_t kp_sb, int64_t kp_sh, int64_t kp_st, int k_row_width,
                     const void* k_norms, int64_t kn_sb, int64_t kn_sh, int64_t kn_st,
                     const void* v_packed, int64_t vp_sb, int64_t vp_sh, int64_t vp_st, int v_row_width,
                     const void* v_norms, int64_t vn_sb, int64_t vn_sh, int64_t vn_st,
                     int B, int n_kv, int gqa, int S, int T, int q_pos_offset, int is_causal,
                     int k_layout, int v_layout, float scale, int unrotate,
                     void* workspace, size_t workspace_bytes,
                     void* out, int64_t o_sb, int64_t o_sh, int64_t o_ss, void* stream) {
    BGTQ_CHECK_ARG(plans && q && k_packed && k_norms && v_packed && v_norms && out);
    BGTQ_CHECK_ARG(B >= 0 && n_kv > 0 && gqa > 0 && S >= 0 && T >= 0 && q_pos_offset >= 0);
    BGTQ_CHECK_ARG(x_dtype == BGTQ_X_FP16 || (x_dtype == BGTQ_X_BF16 && rotate_q));
    if (B == 0 || S == 0) return BGTQ_OK;            // no query rows: nothing to write
    BGTQ_CHECK_ARG(k_layout == BGTQ_K_BITPACKED || k_layout == BGTQ_K_MIXED);
    BGTQ_CHECK_ARG(v_layout == BGTQ_V_BITPACKED || v_layout == BGTQ_V_NIBBLE);
    // layout requirements, those of bgtq_prefill_attn
    if (!(scale > 0.f) || T == 0) return BGTQ_EUNSUPPORTED;
    if (gqa > 256) return BGTQ_EUNSUPPORTED;
    if ((kp_st & 3) || (kp_sb & 3) || (kp_sh & 3) || ((uintptr_t)k_packed & 3)) return BGTQ_EUNSUPPORTED;
    if ((vp_st & 3) || (vp_sb & 3) || (vp_sh & 3) || ((uintptr_t)v_packed & 3)) return BGTQ_EUNSUPPORTED;
    if (kp_st != k_row_width || k_row_width < 4 || k_row_width > 128) return BGTQ_EUNSUPPORTED;
    if (vn_st != 1 || kn_st < 1 || kn_st > BGTQ_MAX_SEGMENTS) return BGTQ_EUNSUPPORTED;
    if (v_row_width != 16 && v_row_width != 32 && v_row_width != 48 && v_row_width != 64) return BGTQ_EUNSUPPORTED;
    if (vp_st < v_row_width || vp_st > v_row_width + 4) return BGTQ_EUNSUPPORTED;
    if (v_layout == BGTQ_V_NIBBLE && v_row_width != 64) return BGTQ_EUNSUPPORTED;
    if ((q_ss & 7) || (q_sh & 7) || (q_sb & 7) || ((uintptr_t)q & 15)) return BGTQ_EUNSUPPORTED;           // 16-byte query loads
    if ((o_ss & 3) || (o_sh & 3) || (o_sb & 3) || ((uintptr_t)out & 7)) return BGTQ_EUNSUPPORTED;          // 8-byte output stores
    BGTQ_CHECK_ARG(workspace && ((uintptr_t)workspace & 15) == 0);
    if (is_causal) T = (int)std::min<int64_t>(T, (int64_t)q_pos_offset + S);                               // no row sees a record past the last query's position
    if (workspace_bytes < bgtq_prompt_workspace_bytes(B, n_kv, gqa, S, T)) return BGTQ_EINVAL;
    const int rows = prompt_rows(B, n_kv, gqa, S), BQ = rows / gqa, n_qb = (S + BQ - 1) / BQ, all_parts = prompt_splits(B, n_kv, gqa, S, T);
    const int teams = prompt_teams((int64_t)B * n_kv * n_qb, rows, all_parts), ns = all_parts / teams;
    // a grid dimension holds 65535 query blocks (the bound of bgtq_prefill_attn: blocks of fewer rows are only taken below
    // 2^19 rows); with partitions there are at most 256 blocks, and as many groups of 32 rows as the merge's grid takes
    if (n_qb > 65535 || B > 65535) return BGTQ_EUNSUPPORTED;
    static std::atomic<int> ready{0};
    if (ready.load(std::memory_order_acquire) == 0) {
        // offsets into the dynamic LDS block are used as LDS addresses: holds only without static LDS
        int ok = 1;
        for (const void* f : {(const void*)prompt_stage_kernel, (const void*)prompt_attn_kernel<false, 4, 1>, (const void*)prompt_attn_kernel<true, 4, 1>,
                              (const void*)prompt_attn_kernel<false, 4, 2>, (const void*)prompt_attn_kernel<true, 4, 2>,
                              (const void*)prompt_attn_kernel<false, 8, 1>, (const void*)prompt_attn_kernel<true, 8, 1>,
                              (const void*)prompt_merge_kernel<1>, (const void*)prompt_merge_kernel<8>}) {
            hipFuncAttributes fa;
            hipError_t e = hipFuncGetAttributes(&fa, f);
            if (e != hipSuccess) return (int)e;
            e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            if (e != hipSuccess) return (int)e;
            if (fa.sharedSizeBytes != 0) ok = -1;
        }
        ready.store(ok, std::memory_order_release);
    }
    if (ready.load(std::memory_order_acquire) < 0) return BGTQ_EUNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;

    uint8_t* ws = (uint8_t*)workspace;
    StageArgs g;
    g.plans = plans;
    g.kp = (const uint8_t*)k_packed; g.kp_sb = kp_sb; g.kp_sh = kp_sh;
    g.kn = (const uint16_t*)k_norms; g.kn_sb = kn_sb; g.kn_sh = kn_sh; g.kn_st = (int)kn_st;
    g.vp = (const uint8_t*)v_packed; g.vp_sb = vp_sb; g.vp_sh = vp_sh;
    g.vn = (const uint16_t*)v_norms; g.vn_sb = vn_sb; g.vn_sh = vn_sh;
    g.n_kv = n_kv; g.pairs = B * n_kv; g.T = T; g.n_tiles = (T + MT - 1) / MT;
    g.k_layout = k_layout; g.v_layout = v_layout; g.k_row_width = k_row_width; g.v_stride = (int)vp_st;
    const int raw = raw_bytes(k_row_width, (int)vp_st, (int)kn_st, g.kt, g.knr, g.vnr, g.vt);
    // two work-groups fit a compute unit; tiles in equal shares over what that makes
    g.per_wg = (int)std::max<int64_t>(1, ((int64_t)g.n_tiles * B * n_kv + 511) / 512);
    g.bf16 = x_dtype == BGTQ_X_BF16; g.rotate_q = rotate_q != 0;
    g.rot = ws;
    g.tiles = ws + (size_t)n_kv * HEAD_PARTS * PART;
    PromptArgs a;
    a.rot = g.rot; a.tiles = g.tiles;
    a.q = (const uint16_t*)q; a.q_sb = q_sb; a.q_sh = q_sh; a.q_ss = q_ss;
    a.n_kv = n_kv; a.gqa = gqa; a.S = S; a.T = T; a.n_tiles = g.n_tiles; a.q_pos_offset = q_pos_offset; a.causal = is_causal != 0;
    a.n_splits = ns; a.rows = rows; a.n_qb = n_qb; a.scale = scale; a.rotate_q = rotate_q != 0; a.unrotate = unrotate != 0;
    a.part_o = (float*)(g.tiles + (size_t)B * n_kv * g.n_tiles * TILE);
    a.part_ml = a.part_o + (size_t)B * n_kv * n_qb * ns * (rows / 32) * 64 * 64;
    a.out = (uint16_t*)out; a.o_sb = o_sb; a.o_sh = o_sh; a.o_ss = o_ss;
    const int wgs_per = (g.n_tiles + g.per_wg - 1) / g.per_wg;
    hipLaunchKernelGGL(prompt_stage_kernel, dim3((unsigned)(n_kv * ROT_WGS + wgs_per * B * n_kv)), dim3(DQ_THR), (size_t)RAW_OFF + raw + DQ_TILE_BYTES, st, g);
    const dim3 grid((unsigned)n_kv, (unsigned)B, (unsigned)(n_qb * ns));
    auto attn = g.bf16 ? (rows == 256 ? prompt_attn_kernel<true, 8, 1> : teams == 2 ? prompt_attn_kernel<true, 4, 2> : prompt_attn_kernel<true, 4, 1>)
                       : (rows == 256 ? prompt_attn_kernel<false, 8, 1> : teams == 2 ? prompt_attn_kernel<false, 4, 2> : prompt_attn_kernel<false, 4, 1>);
    hipLaunchKernelGGL(attn, grid, dim3(2 * rows * teams), prompt_lds(rows / 32, teams), st, a);
    if (ns > 1) {
        const int groups = n_qb * (rows / 32);
        if ((int64_t)B * n_kv * groups > 256)
            hipLaunchKernelGGL(prompt_merge_kernel<1>, dim3((unsigned)n_kv, (unsigned)B, (unsigned)((groups + 3) / 4)), dim3(64 * merge_waves(1)), merge_lds(1), st, a);
        else
            hipLaunchKernelGGL(prompt_merge_kernel<8>, dim3((unsigned)n_kv, (unsigned)B, (unsigned)groups), dim3(64 * merge_waves(8)), merge_lds(8), st, a);
    }
    return bgtq_launch_status();
}

}  // extern "C"
