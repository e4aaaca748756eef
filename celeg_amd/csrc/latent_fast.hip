// Attention over a latent cache on the matrix cores (bfloat16).
//
// A cached row holds `rank` compressed values and `rot` rotated key values, D = rank + rot.  A
// score is q_lat . row over D; the weighted sum runs over the first `rank` values of the same
// rows.  A workgroup of four wavefronts brings 64 cached rows at a time into LDS, as they lie
// (sK [key][D]): they are the operand of the scores, and, read transposed (ds_read_b64_tr_b16, four keys of a
// dimension a lane), the operand of the weighted sum.  Scores are computed transposed (S^T = K Q^T) with the
// keys of a block dealt to the accumulator registers so that a lane's eight registers of two score
// tiles are eight neighbouring keys of one query: they are the operand of O^T = V^T P^T as they
// stand, no exchange between lanes.  Softmax state (running maximum in the base-2 domain, sum) and
// the output accumulators are 32-bit.  With EXACT a 32-bit weight enters the product with the values
// as two bfloat16 numbers (its rounding, and what that left), else as one.
//
// Form 0, portions of prompts: a workgroup owns 64 rows of one sequence and one head, a wavefront
// 16 of the rows; keys 0..position of its last row.  Form 1, single tokens: a workgroup owns one
// row, 16 heads and one share of the row's keys; a wavefront makes the scores of 16 of a block's 64 keys, they meet
// in LDS, every wavefront turns all of them into weights and sums a quarter of the dimensions.  The shares'
// partial results meet in a second kernel, which also adds the sink.
//
// KS steps of 32 dimensions and DT tiles of 16 values are the smallest of three sizes that hold a row (zeros
// beyond it), so that no loop has a condition and operands are read from LDS steps ahead of the products that use
// them.  (With the row's own sizes as conditions every read was waited for by itself: a block of 64 keys took 7.6 us in
// a workgroup alone on its compute unit, now 2.5.)  The next block's rows are asked for ahead of a block's products and
// laid into a second buffer behind them: one barrier a block.  What bounds a block now: its matrix
// instructions (1,600 cycles a wavefront), softmax and addresses (about 2,000) and LDS (68 KB a wavefront) each take 0.7 to
// 0.9 us and overlap in part.
// Measured in a recorded chain, 16 heads, rank 256 with 32 rotated, weights as two numbers, a window of 1,024, the same bits
// (before: conditions as above, rows copied transposed within LDS, four barriers a block, one wavefront of four at
// work in form 1): 2,048 rows of a prompt 152 -> 72 us, 77 rows behind 1,100 keys 127 -> 46, four single tokens with the
// join 14.3 -> 8.8; rank 512 with 64 rotated, no window, 1,024 rows 277 -> 96.  Sizes between the three gain less but gain (every
// key; 2,048 rows, 77 behind 1,100 keys, four single tokens at 400): rank 16 with 8 rotated 61.5 -> 61.9, 36.3 -> 31.9, 8.5 -> 7.8, 128 with 32
// 138 -> 65, 77 -> 32, 10.7 -> 8.2, 128 with 64 171 -> 96, 97 -> 48, 12.4 -> 9.1, 256 with 64, which runs as 576 with 512, 691 -> 309,
// 204 -> 94, 20.7 -> 11.1.
//
// With a window the blocks begin at the first key that any column of the workgroup sees, and keys a column
// no longer sees are masked; pages wholly before the window may be another request's by then and are not read.
#include "common.h"

typedef __bf16 lat_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 lat_bf16x4 __attribute__((ext_vector_type(4)));
typedef short lat_s16x4 __attribute__((ext_vector_type(4)));
typedef short lat_s16x8 __attribute__((ext_vector_type(8)));
typedef float lat_f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int lat_u32x4 __attribute__((ext_vector_type(4)));

#define LATF_KEYS 64
#define LATF_SROW (LATF_KEYS + 4)
#define LOG2E 1.4426950408889634f

__device__ __forceinline__ float quad_max(float v) {      // over the four lanes that share a column
    return max_half32(max_row16(v));
}
__device__ __forceinline__ float quad_sum(float v) {
    return sum_half32(sum_row16(v));
}

// Four keys of one dimension: the 16 lanes of a quad together read 4 keys x 16 dimensions, lane i at key i / 4,
// dimensions 4 (i % 4) .., and lane i gets dimension i of the four.
__device__ __forceinline__ lat_s16x4 read_turned(const __bf16* at) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lat_s16x4*)at);
}

template <int KS, int DT>
struct LatentLds {
    static constexpr int KROW = KS * 32 + 8;              // values between rows: 16 lanes at one chunk fall on all banks
    static constexpr int ROWS = LATF_KEYS * KROW;         // values of a buffer
    static constexpr size_t bytes = static_cast<size_t>(2) * ROWS * 2;
};

template <int FORM, int KS, int DT, bool EXACT>
__global__ __launch_bounds__(256, (KS <= 9 ? 2 : 1)) void latent_attention_mfma_kernel(
    const __bf16* __restrict__ q, int ldq, const __bf16* __restrict__ pool, const int* __restrict__ table, int table_stride,
    const int* __restrict__ cu_seqlens, const int* __restrict__ seq_slot, const int* __restrict__ seq_start, int n_seqs,
    const int* __restrict__ token_slot, const int* __restrict__ positions, const float* __restrict__ sink,
    __bf16* __restrict__ out, int ldo, float* __restrict__ ws_o, float* __restrict__ ws_ml, int n_splits,
    int blocks_per_split, int heads, int rank, int rot, int page_tokens, int n_layers, int layer, float scale_log2e,
    int window) {
    extern __shared__ __attribute__((aligned(16))) unsigned char latf_lds[];
    __shared__ int s_page[2][LATF_KEYS];
    __shared__ __attribute__((aligned(16))) float s_scores[FORM == 1 ? 16 * LATF_SROW : 4];      // [column][key]
    constexpr int KROW = LatentLds<KS, DT>::KROW, CHUNKS = KS * 4;    // 16-byte pieces of a padded row
    constexpr int DEEP = KS <= 9 ? 2 : 3;  // operands from LDS: DEEP - 1 steps ahead
    constexpr bool AHEAD = KS <= 9;        // (the largest size has no registers to hold the next rows beside its sums)
    constexpr int OT = FORM == 1 ? DT / 4 : DT;                       // tiles of 16 values that a wavefront sums
    const int D = rank + rot;
    __bf16* const sK = reinterpret_cast<__bf16*>(latf_lds);           // [2][64][KROW]
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 15, qd = lane >> 4;
    const int dt0 = FORM == 1 ? wave * OT : 0;
    constexpr int TILE = 64;               // rows of a workgroup (form 0)

    // ---- which columns this workgroup owns
    int slot, first_block, end_block;      // key blocks [first_block, end_block)
    int wg_limit, wg_first;                // the last and the first key any column of the workgroup sees
    int col_row, col_head, col_limit;      // this lane's column: row of q / out, head, last key seen (-1: none)
    bool wave_computes;
    if (FORM == 0) {
        int tile = blockIdx.x, s = 0, len = 0, row0 = 0;
        for (; s < n_seqs; ++s) {
            row0 = cu_seqlens[s];
            len = cu_seqlens[s + 1] - row0;
            const int tiles = len > 1 ? (len + TILE - 1) / TILE : 0;     // single tokens go to the other form
            if (tile < tiles) break;
            tile -= tiles;
        }
        if (s >= n_seqs) return;
        slot = seq_slot[s];
        const int start = seq_start[s];
        col_head = blockIdx.y;
        const int r = tile * TILE + wave * 16 + c;         // row within the sequence
        col_row = row0 + min(r, len - 1);
        col_limit = r < len ? start + r : -1;
        const int last = min(len, tile * TILE + TILE) - 1;
        wg_first = window > 0 ? max(0, start + tile * TILE - window + 1) : 0;
        first_block = wg_first / LATF_KEYS;
        wg_limit = start + last;
        end_block = wg_limit / LATF_KEYS + 1;
        wave_computes = tile * TILE + wave * 16 < len;
    } else {
        const int t = blockIdx.x;
        slot = token_slot[t];
        const int pos = positions[t];
        col_head = blockIdx.y * 16 + c;
        col_row = t;
        col_limit = col_head < heads ? pos : -1;
        wg_limit = pos;
        wg_first = window > 0 ? max(0, pos - window + 1) : 0;
        first_block = wg_first / LATF_KEYS + blockIdx.z * blocks_per_split;
        end_block = min(pos / LATF_KEYS + 1, first_block + blocks_per_split);
        wave_computes = true;
    }
    const int* pages = table + static_cast<size_t>(slot) * table_stride;
    // (in pieces of 8 values, so that 32 bits hold pages of up to 64 GiB; the host has checked that they do)
    const unsigned row_pieces = static_cast<unsigned>(D) / 8, page_stride = static_cast<unsigned>(n_layers) * page_tokens * row_pieces;
    const __bf16* layer_base = pool + static_cast<size_t>(layer) * page_tokens * D;
    const int page_shift = 31 - __clz(page_tokens);     // page_tokens is a power of two

    // ---- a block's rows on their way to LDS: the rows' pages, then the pieces (zeros beyond D and beyond the last key
    // any column sees: pages there may not be the request's); this thread's pieces are tid + 256 j of the block's 64 x CHUNKS
    const auto page_of = [&](int blk) {
        const int pos = blk * LATF_KEYS + (tid & (LATF_KEYS - 1));
        const int page = pages[min(max(pos, wg_first), wg_limit) >> page_shift];      // (no branch round a load)
        return blk < end_block && pos <= wg_limit && pos >= wg_first ? page : -1;
    };
    lat_u32x4 staged[KS];
    unsigned there;                        // bit j: piece j is a row's, not zeros
    const auto ask = [&](int blk, const int* block_pages) {
        there = 0u;
        int page[KS];
#pragma unroll
        for (int j = 0; j < KS; ++j) page[j] = block_pages[(tid + 256 * j) / CHUNKS];
#pragma unroll
        for (int j = 0; j < KS; ++j) {
            const int i = tid + 256 * j, key = i / CHUNKS, ch = i - key * CHUNKS;
            there |= (page[j] >= 0 && ch * 8 < D ? 1u : 0u) << j;
            // (no branch round a load: a piece that is not there asks for one of page 0 or for its row's last)
            const unsigned in_page = static_cast<unsigned>((blk * LATF_KEYS + key) & (page_tokens - 1)) * row_pieces + min(static_cast<unsigned>(ch), row_pieces - 1);
            staged[j] = reinterpret_cast<const lat_u32x4*>(
                layer_base)[static_cast<unsigned long long>(static_cast<unsigned>(max(page[j], 0))) * page_stride + in_page];
        }
    };
    // key 32 h + 8 a + 4 b + r of a block lies at row 32 h + 16 b + 4 a + r: the 16 keys of a tile of scores in 16 rows
    const auto lay = [&](__bf16* to) {
#pragma unroll
        for (int j = 0; j < KS; ++j) {
            const int i = tid + 256 * j, key = i / CHUNKS, ch = i - key * CHUNKS;
            const int row = (key & 35) | ((key & 4) << 2) | ((key & 24) >> 1);
            *reinterpret_cast<lat_u32x4*>(to + row * KROW + ch * 8) = there >> j & 1 ? staged[j] : lat_u32x4{0u, 0u, 0u, 0u};
        }
    };
    const int page0 = page_of(first_block), page1 = page_of(first_block + 1);

    // a column tile's last key (blocks beyond it hold nothing for its columns) and the first key that some column does not see
    int tile_limit = col_limit, tile_min_limit = col_limit < 0 ? 0x7fffffff : col_limit;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
        tile_limit = max(tile_limit, __shfl_xor(tile_limit, off, 64));
        tile_min_limit = min(tile_min_limit, __shfl_xor(tile_min_limit, off, 64));
    }

    // ---- the queries of this lane's column, as the operand of the scores
    lat_bf16x8 qreg[KS];
    const __bf16* qrow = q + static_cast<size_t>(col_row) * ldq + static_cast<size_t>(min(col_head, heads - 1)) * D;
#pragma unroll
    for (int st = 0; st < KS; ++st) {
        lat_u32x4 v = {0u, 0u, 0u, 0u};
        const int d = st * 32 + qd * 8;
        if (d < D && col_limit >= 0) v = *reinterpret_cast<const lat_u32x4*>(qrow + d);
        qreg[st] = __builtin_bit_cast(lat_bf16x8, v);
    }
    lat_f32x4 oacc[OT];
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int dt = 0; dt < OT; ++dt) oacc[dt] = lat_f32x4{0.f, 0.f, 0.f, 0.f};

    if (tid < LATF_KEYS) {
        s_page[0][tid] = page0;
        s_page[1][tid] = page1;
    }
    __syncthreads();
    ask(first_block, s_page[0]);
    lay(sK);
    __syncthreads();
    for (int blk = first_block; blk < end_block; ++blk) {
        const int kb = blk * LATF_KEYS, at = (blk - first_block) & 1;
        const __bf16* const rows = sK + at * LatentLds<KS, DT>::ROWS;
        // ---- what the next block needs (its pages are there; those of the block behind it are asked for first)
        const int page2 = page_of(blk + 2);
        if (AHEAD && blk + 1 < end_block) ask(blk + 1, s_page[at ^ 1]);
        const bool live = wave_computes && kb <= tile_limit && (window <= 0 || kb + LATF_KEYS - 1 > tile_min_limit - window);
        if (live) {
            // ---- scores, transposed: register r of lane quad qd, tile kt, is key 32 (kt / 2) + 8 qd + 4 (kt % 2) + r
            // (tile kt is rows 16 kt .. of the buffer)
            lat_f32x4 sacc[4];
            if constexpr (FORM == 1) {
                const __bf16* const kp = rows + (16 * wave + c) * KROW + qd * 8;
                lat_bf16x8 kf[KS];
#pragma unroll
                for (int st = 0; st < KS; ++st) kf[st] = *reinterpret_cast<const lat_bf16x8*>(kp + st * 32);
                lat_f32x4 sum{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int st = 0; st < KS; ++st) sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[st], qreg[st], sum, 0, 0, 0);
                *reinterpret_cast<lat_f32x4*>(s_scores + c * LATF_SROW + 32 * (wave >> 1) + 8 * qd + 4 * (wave & 1)) = sum;
                __syncthreads();                          // (form 1: all wavefronts are live alike)
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
                    sacc[kt] = *reinterpret_cast<const lat_f32x4*>(s_scores + c * LATF_SROW + 32 * (kt >> 1) + 8 * qd + 4 * (kt & 1));
            } else {
                // a step's operands of all four tiles come two steps ahead of its products (left alone, the compiler waits
                // for each read ahead of the instruction that uses it)
                const __bf16* const kp = rows + c * KROW + qd * 8;
                lat_bf16x8 kf[DEEP][4];
                const auto read = [&](int st) {
#pragma unroll
                    for (int kt = 0; kt < 4; ++kt) kf[st % DEEP][kt] = *reinterpret_cast<const lat_bf16x8*>(kp + 16 * kt * KROW + st * 32);
                };
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) sacc[kt] = lat_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int st = 0; st < DEEP - 1; ++st) read(st);
#pragma unroll
                for (int st = 0; st < KS; ++st) {
                    if (st + DEEP - 1 < KS) read(st + DEEP - 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int kt = 0; kt < 4; ++kt) sacc[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[st % DEEP][kt], qreg[st], sacc[kt], 0, 0, 0);
                }
            }
            if (kb + LATF_KEYS - 1 > tile_min_limit || (window > 0 && kb <= tile_limit - window)) {
                const int col_first = window > 0 ? col_limit - window + 1 : 0;
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int key = kb + 32 * (kt >> 1) + 8 * qd + 4 * (kt & 1) + r;
                        if (key > col_limit || key < col_first) sacc[kt][r] = -INFINITY;
                    }
            }
            float mx = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                for (int r = 0; r < 4; ++r) mx = fmaxf(mx, sacc[kt][r]);
            mx = quad_max(mx) * scale_log2e;          // the scale is positive
            const float m_new = fmaxf(m, mx);
            const float alpha = __builtin_amdgcn_exp2f(m - (m_new == -INFINITY ? 0.f : m_new));
            l *= alpha;
            m = m_new;
#pragma unroll
            for (int dt = 0; dt < OT; ++dt) oacc[dt] *= alpha;
            const float m_use = m_new == -INFINITY ? 0.f : m_new;
            float psum = 0.f;
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float p = __builtin_amdgcn_exp2f(fmaf(sacc[kt][r], scale_log2e, -m_use));
                    sacc[kt][r] = p;
                    psum += p;
                }
            l += psum;
            lat_bf16x8 pb[2], rest[2];
#pragma unroll
            for (int kp = 0; kp < 2; ++kp)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float p = sacc[2 * kp + e / 4][e % 4];
                    pb[kp][e] = static_cast<__bf16>(p);
                    if (EXACT) rest[kp][e] = static_cast<__bf16>(p - static_cast<float>(pb[kp][e]));
                }
            // ---- O^T += V^T P^T, likewise: the operands of two tiles of values two steps ahead
            const __bf16* const vp = rows + (4 * qd + (c >> 2)) * KROW + dt0 * 16 + 4 * (c & 3);
            lat_s16x4 vf[DEEP][2][4];
            const auto read = [&](int g) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int part = 0; part < 4; ++part)           // 16 rows each: keys 0..3 and 4..7 of eight, then the next 32
                        vf[g % DEEP][i][part] = read_turned(vp + 16 * part * KROW + (2 * g + i) * 16);
            };
#pragma unroll
            for (int g = 0; g < DEEP - 1 && g < OT / 2; ++g) read(g);
#pragma unroll
            for (int g = 0; g < OT / 2; ++g) {
                if (g + DEEP - 1 < OT / 2) read(g + DEEP - 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int kp = 0; kp < 2; ++kp)
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        const int dt = 2 * g + i;
                        const lat_bf16x8 v = __builtin_bit_cast(lat_bf16x8, __builtin_shufflevector(vf[g % DEEP][i][2 * kp], vf[g % DEEP][i][2 * kp + 1], 0, 1, 2, 3, 4, 5, 6, 7));
                        oacc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, pb[kp], oacc[dt], 0, 0, 0);
                        if (EXACT) oacc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, rest[kp], oacc[dt], 0, 0, 0);
                    }
            }
        }
        if (blk + 1 < end_block) {
            if (!AHEAD) ask(blk + 1, s_page[at ^ 1]);
            lay(sK + (at ^ 1) * LatentLds<KS, DT>::ROWS);
            if (tid < LATF_KEYS) s_page[at][tid] = page2;
            __syncthreads();
        }
    }
    if (!wave_computes || col_limit < 0) return;
    float l_all = quad_sum(l);
    if (FORM == 0) {
        float corr = 1.f;
        if (sink) {
            const float sk = sink[col_head] * LOG2E;
            const float m_all = fmaxf(m, sk);
            corr = exp2f(m - m_all);
            l_all = l_all * corr + exp2f(sk - m_all);
        }
        const float f = corr / l_all;
        __bf16* orow = out + static_cast<size_t>(col_row) * ldo + static_cast<size_t>(col_head) * rank + qd * 4;
#pragma unroll
        for (int dt = 0; dt < OT; ++dt)
            if (dt * 16 < rank)
                *reinterpret_cast<lat_bf16x4*>(orow + dt * 16) =
                    lat_bf16x4{static_cast<__bf16>(oacc[dt][0] * f), static_cast<__bf16>(oacc[dt][1] * f),
                               static_cast<__bf16>(oacc[dt][2] * f), static_cast<__bf16>(oacc[dt][3] * f)};
    } else {
        const size_t part = (static_cast<size_t>(col_row) * heads + col_head) * n_splits + blockIdx.z;
        float* o = ws_o + part * rank + qd * 4;
#pragma unroll
        for (int dt = 0; dt < OT; ++dt)
            if ((dt0 + dt) * 16 < rank) *reinterpret_cast<lat_f32x4*>(o + (dt0 + dt) * 16) = oacc[dt];
        if (wave == 0 && qd == 0) {
            ws_ml[part * 2] = m;
            ws_ml[part * 2 + 1] = l_all;
        }
    }
}

// The shares of a single token's keys meet: out = sum_i o_i 2^(m_i - M) / (sum_i l_i 2^(m_i - M) + 2^(sink - M)).
// A thread owns an output dimension.  Every wavefront works out the shares' factors for itself, lane i
// that of share i, and takes them from its lanes; the outputs of the first JOIN_CHUNK shares are asked
// for before anything is waited for, so that 17 shares of a context are two trips to memory (4 rows of 16 heads: 5.3 -> 4.8 us).
#define LATF_MAX_SPLITS 64
#define JOIN_CHUNK 16
__global__ __launch_bounds__(256) void latent_attention_join_kernel(const float* __restrict__ ws_o, const float* __restrict__ ws_ml,
                                                                    int n_splits, const float* __restrict__ sink,
                                                                    __bf16* __restrict__ out, int ldo, int heads, int rank) {
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & (CELEG_WAVE - 1);
    const size_t part0 = (static_cast<size_t>(t) * heads + h) * n_splits;
    const int share = min(lane, n_splits - 1);
    const float m_raw = ws_ml[(part0 + share) * 2], l_raw = ws_ml[(part0 + share) * 2 + 1];
    const float sk = sink ? sink[h] * LOG2E : -INFINITY;
    float o[JOIN_CHUNK];
    const auto fetch = [&](int i0, int d) {
#pragma unroll
        for (int j = 0; j < JOIN_CHUNK; ++j) o[j] = ws_o[(part0 + min(i0 + j, n_splits - 1)) * rank + min(d, rank - 1)];
    };
    fetch(0, threadIdx.x);
    const float mi = lane < n_splits ? m_raw : -INFINITY;
    const float M = fmaxf(wave_max(mi), sk);
    const float f = mi == -INFINITY ? 0.f : exp2f(mi - M);
    const float L = wave_sum(lane < n_splits ? l_raw * f : 0.f) + (sink ? exp2f(sk - M) : 0.f);
    const float inv_total = 1.0f / L;
    for (int d0 = 0; d0 < rank; d0 += 256) {          // the same for every thread
        const int d = d0 + static_cast<int>(threadIdx.x);
        float acc = 0.f;
        for (int i0 = 0; i0 < n_splits; i0 += JOIN_CHUNK) {
            if (d0 > 0 || i0 > 0) fetch(i0, d);       // the first are here already
#pragma unroll
            for (int j = 0; j < JOIN_CHUNK; ++j)
                if (i0 + j < n_splits)
                    acc = fmaf(o[j], __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), i0 + j)), acc);
        }
        if (d < rank) out[static_cast<size_t>(t) * ldo + static_cast<size_t>(h) * rank + d] = static_cast<__bf16>(acc * inv_total);
    }
}

template <int FORM, int KS, int DT, bool EXACT>
static int latent_mfma_launch(dim3 grid, hipStream_t stream, const void* q, int ldq, const void* pool,
                              const int* table, int table_stride, const int* cu_seqlens, const int* seq_slot,
                              const int* seq_start, int n_seqs, const int* token_slot, const int* positions,
                              const float* sink, void* out, int ldo, float* ws_o, float* ws_ml, int n_splits,
                              int blocks_per_split, int heads, int rank, int rot, int page_tokens, int n_layers, int layer,
                              float scale_log2e, int window) {
    auto kernel = latent_attention_mfma_kernel<FORM, KS, DT, EXACT>;
    constexpr size_t lds = LatentLds<KS, DT>::bytes;
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 static_cast<int>(lds));
        if (e != hipSuccess) return static_cast<int>(e);
    }
    hipLaunchKernelGGL(kernel, grid, dim3(256), lds, stream, static_cast<const __bf16*>(q), ldq,
                       static_cast<const __bf16*>(pool), table, table_stride, cu_seqlens, seq_slot, seq_start, n_seqs,
                       token_slot, positions, sink, static_cast<__bf16*>(out), ldo, ws_o, ws_ml, n_splits, blocks_per_split,
                       heads, rank, rot, page_tokens, n_layers, layer, scale_log2e, window);
    return CELEG_LAUNCH_RESULT();
}

// rank a multiple of 16 up to 512, rank + rot a multiple of 8 up to 576
// rows of a workgroup's tile in form 0
extern "C" int celeg_latent_attention_tile_rows(int rank, int rot) {
    (void)rank;
    (void)rot;
    return 64;        // one tile of 16 columns a wavefront (two were measured slower: half the workgroups, and no more overlap)
}

extern "C" int celeg_latent_attention_fast_ok(int rank, int rot, int n_layers, int page_tokens) {
    return rank > 0 && rank % 16 == 0 && rank <= 512 && rot >= 0 && (rank + rot) % 8 == 0 && rank + rot <= 576 && n_layers > 0 &&
           page_tokens > 0 && (page_tokens & (page_tokens - 1)) == 0 &&
           static_cast<unsigned long long>(n_layers) * page_tokens * ((rank + rot) / 8) < (1ull << 32);
}

// form 0: rows of the sequences of more than one token (max_tiles: a bound on their tiles of 64 rows);
// form 1: rows [0, n_single), each one token of its request, keys in n_splits shares of blocks_per_split
// blocks of 64 (of the keys in the row's window); exact: weights as two bfloat16 numbers; ws_o [n_single, heads, n_splits, rank] and ws_ml [n_single, heads, n_splits, 2] 32-bit.
extern "C" int celeg_latent_attention_fast(int form, const void* q, int ldq, const void* pool, const int* table,
                                           int table_stride, const int* cu_seqlens, const int* seq_slot,
                                           const int* seq_start, int n_seqs, int max_tiles, const int* token_slot,
                                           const int* positions, int n_single, const float* sink, void* out, int ldo,
                                           float* ws_o, float* ws_ml, int n_splits, int blocks_per_split, int heads,
                                           int rank, int rot, int page_tokens, int n_layers, int layer, float scale,
                                           int window, int exact, hipStream_t stream) {
    if (!celeg_latent_attention_fast_ok(rank, rot, n_layers, page_tokens) || (form == 1 && n_splits > LATF_MAX_SPLITS))
        return static_cast<int>(hipErrorInvalidValue);
    const int D = rank + rot, KS = (D + 31) / 32, DT = rank / 16;
    const float scale_log2e = scale * LOG2E;
    if (form == 0 ? max_tiles <= 0 : n_single <= 0) return 0;
    const dim3 grid = form == 0 ? dim3(max_tiles, heads) : dim3(n_single, (heads + 15) / 16, n_splits);
#define LATF_GO(FORM, KSM, DTM, EXACT)                                                                                      \
    latent_mfma_launch<FORM, KSM, DTM, EXACT>(grid, stream, q, ldq, pool, table, table_stride, cu_seqlens, seq_slot, \
                                                 seq_start, n_seqs, token_slot, positions, sink, out, ldo, ws_o, ws_ml,      \
                                                 n_splits, blocks_per_split, heads, rank, rot, page_tokens, n_layers, layer, \
                                                 scale_log2e, window)
#define LATF_SIZES(FORM)                                                                        \
    (KS <= 5 && DT <= 8    ? (exact ? LATF_GO(FORM, 5, 8, true) : LATF_GO(FORM, 5, 8, false))   \
     : KS <= 9 && DT <= 16 ? (exact ? LATF_GO(FORM, 9, 16, true) : LATF_GO(FORM, 9, 16, false)) \
                           : (exact ? LATF_GO(FORM, 18, 32, true) : LATF_GO(FORM, 18, 32, false)))
    if (form == 0) return LATF_SIZES(0);
    const int rc = LATF_SIZES(1);
    if (rc) return rc;
    hipLaunchKernelGGL(latent_attention_join_kernel, dim3(n_single, heads), dim3(256), 0, stream, ws_o, ws_ml, n_splits, sink,
                       static_cast<__bf16*>(out), ldo, heads, rank);
    return CELEG_LAUNCH_RESULT();
#undef LATF_SIZES
#undef LATF_GO
}
