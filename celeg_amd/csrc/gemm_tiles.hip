// bfloat16 products for many rows on gfx950 (portions of prompts: hundreds to thousands of
// rows), with what surrounds them fused in, under the same contract as the products for
// few rows:
//   out[M,N] = epilogue(scale[m] * (A[M,K] W[N,K]^T) + bias)
// A is bfloat16 with its rows one after the other; behind an RMSNorm it is the bfloat16
// copy of the residual stream, W has the norm's weight folded in and
// scale[m] = rsqrt(mean(x_m^2) + eps) comes from the partial sums of squares that the
// producer of the stream left.  Epilogues: store | add into the 32-bit residual stream,
// refresh its bfloat16 copy and leave partial sums of squares | SwiGLU of a gate and an
// up stream.
//
// The weights lie as they are ([rows, K]) or, for the residual epilogue, packed in blocks of 32 values of k ([K/32, rows, 32],
// the copy that the products of few rows read): a load then asks for 1 KB in a row where it otherwise asks for 128 bytes of
// eight rows.  With weights from memory (2,048 rows: 75 MB cross the fabric behind the L2s) w2 of 1,024 x 4,608 takes 32.1 us
// packed and 35.0 as they are, out_proj of 1,024 x 1,024 12.1 and 12.5; celeg_gemm_tiles_packed says where it is worth it.
//
// Layout.  A workgroup owns a tile of BM rows x BN weight rows (for SwiGLU: BN/2 gate rows
// and the BN/2 up rows of the same columns) over the whole of K.  Blocks of 64 values of k
// of both operands travel from memory straight into LDS (16 bytes a lane,
// global_load_lds), STAGES blocks deep, so that loads of later blocks are in flight while
// the matrix instructions work on the current one; the compiler's barrier would wait for
// every load, so the loop waits for the oldest block by count and uses the bare barrier.
// A row of a block is 128 bytes = 8 chunks of 16; chunk c of row r lies at chunk
// c ^ (r & 7) of its row, which spreads the rows that neighbouring lanes read at the same
// chunk over the banks (measured: as fast as reading 1 KB in a row; rows padded to 144 bytes
// or a swap of neighbouring rows on top were 1.6 times slower).
// (A row of packed weights is 64 bytes a half of the block, its chunk c at c ^ ((r / 2) & 3): read by lane % 16 as the row and
// lane / 16 as the chunk, both lie over all banks, 4 cycles a KB; at c ^ ((r / 4) & 3) 8 cycles.)
// The loads place the chunks: a load instruction writes 1 KB = 8 rows, lane l at row l / 8,
// chunk l % 8, so lane l asks memory for the chunk that belongs there.
// WGM x WGN wavefronts share the tile; a wavefront keeps (BN/WGN/16) x (BM/WGM/16) tiles of
// 16x16 sums (v_mfma_f32_16x16x32_bf16 with the weights as the first operand: a lane then
// holds 4 neighbouring columns of one row, which it finishes and writes as one piece).
//
// Reference semantics of the fused parts: RMSNorm src/backend/cpu/kernels/elementwise.cpp:56-76,
// SwiGLU elementwise.cpp:101-119, projections y = x W^T src/model/weight_plan.cpp:82-130;
// the reference fuses the residual addition into its products with beta = 1
// (src/backend/cuda/model/prefill_batched/non_attention.cpp:175-201).
#include "common.h"
#include "tile_params.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

enum { T_STORE = 0, T_RESIDUAL = 2, T_SWIGLU = 3, T_QKV = 5 };   // (0, 2, 3: the numbers of the few-rows products)


#define GPTR(p) ((const __attribute__((address_space(1))) void*)(p))
#define LPTR(p) ((__attribute__((address_space(3))) void*)(p))

__device__ __forceinline__ float round_bf16(float x) { return to_float(from_float<bf16>(x)); }

// o = g / (1 + e^-g) * u with the hardware's exponential (an ulp, in 32-bit: the exact one cost the SwiGLU product
// of 2,048 rows 3 us) and a correctly rounded reciprocal.  One Newton step behind v_rcp_f32 rounds correctly wherever the
// reciprocal is a normal number (tried: every 24-bit divisor), for a third of the instructions of the exact division, which
// stays for the gates whose 1 + e^-g is 2^126 or more (below -87.3; v_rcp_f32 makes 0 of their reciprocals).  w1 with w3,
// exact division | this | v_rcp_f32 alone: 2,048 rows 42.9 | 40.5 | 39.7 us, 1,000 rows 25.5 | 24.3 | 23.9, 600 rows 19.5 | 19.2 | 18.9.
template <int N>
__device__ __forceinline__ void tile_swiglu(const float (&g)[N], const float (&u)[N], float (&o)[N]) {
    float x[N], largest = 1.0f;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        x[i] = 1.0f + __expf(-g[i]);
        largest = fmaxf(largest, x[i]);
        const float r = __builtin_amdgcn_rcpf(x[i]);
        o[i] = g[i] * fmaf(fmaf(-x[i], r, 1.0f), r, r) * u[i];
    }
    if (largest >= 0x1p126f)
#pragma unroll
        for (int i = 0; i < N; ++i) o[i] = g[i] * __frcp_rn(x[i]) * u[i];
}

// A store of 16 bytes a lane that does not stay in the die's L2 until the kernel's end.  Where a product's workgroups all
// end together, what they wrote leaves the L2s only then, with nothing beside it: written through, w1 with w3 at 2,048 rows (19
// MB) takes 39.3 us instead of 40.9, at 1,000 rows 26.9 instead of 27.8.  (The residual epilogue, 32-bit and bfloat16
// values of 12 MB at 2,048 rows, gains 0.2 to 0.6 us there and loses as much at 300 rows and 3 us of 58 at 4,000: it stores plainly.)
// `s_nop`: the data's registers may not be written right behind the instruction.
__device__ __forceinline__ void store_through(bf16x8_t* const to, const bf16x8_t& v) {
    asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 2" ::"v"(to), "v"(v) : "memory");
}

template <int N>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int EPI> struct TileStreams { static constexpr int n = EPI == T_SWIGLU ? 2 : 1; };

// The 1/rms of a lane's rows (first, first + 16, ..) from the partial sums of squares that
// the producer of the stream left; 1 without a norm.  The four lanes that share a row (q = 0..3)
// take four partial sums each, as one load where the rows are aligned, and add up over the
// lanes: a few loads a lane, all in flight at once.  (One lane reading all of a row's sums,
// eight at a time, cost a product of 2,048 rows 12 us: 64 loads a lane in two trips, queued
// behind the first blocks of the operands.)
template <int FM>
__device__ __forceinline__ void tile_row_scales(const TileParams& p, const int first, const int q, float (&scale)[FM]) {
#pragma unroll
    for (int tm = 0; tm < FM; ++tm) scale[tm] = 1.f;
    if (!p.stats) return;
    const int nb = p.n_stat_blocks;
    const bool aligned = (p.stats_ld & 3) == 0 && (reinterpret_cast<uintptr_t>(p.stats) & 15) == 0;
    float ssq[FM];
#pragma unroll
    for (int tm = 0; tm < FM; ++tm) ssq[tm] = 0.f;
    for (int c0 = 0; c0 < nb; c0 += 16) {         // (once, up to 16 partial sums a row)
        const int b = c0 + 4 * q;
        floatx4_t part[FM];
#pragma unroll
        for (int tm = 0; tm < FM; ++tm) {
            const float* const srow = p.stats + static_cast<size_t>(min(first + tm * 16, p.M - 1)) * p.stats_ld;
            if (aligned && b + 4 <= nb) {
                part[tm] = *reinterpret_cast<const floatx4_t*>(srow + b);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) part[tm][i] = b + i < nb ? srow[b + i] : 0.f;
            }
        }
#pragma unroll
        for (int tm = 0; tm < FM; ++tm) ssq[tm] += (part[tm][0] + part[tm][1]) + (part[tm][2] + part[tm][3]);
    }
#pragma unroll
    for (int tm = 0; tm < FM; ++tm) {
        float t = ssq[tm];
        t = sum_half32(sum_row16(t));
        scale[tm] = 1.0f / sqrtf(t / static_cast<float>(p.K) + p.eps);
    }
}

// What becomes of a wavefront's sums (shared by the kernels below).  The wavefront (wm, wn) of
// the tile holds rows m0 + wm*WTM .. of `pieces` (<= FNS) column pieces of 16 from column col0 of
// every stream:  acc[s*FNS + j][tm][i] is row .. + tm*16 + lane%16, column col0 + j*16 + 4*(lane/16) + i.
// ROWS_VIA_LDS (store and SwiGLU): a lane's pieces of 4 columns go to the wavefront's corner of
// LDS first and leave in whole rows of the wavefront's tile, 16 bytes a lane; straight from the
// registers a store instruction would touch 16 rows with 32 bytes each.
template <int BM, int WGM, int WGN, int FNS, int EPI, bool ROWS_VIA_LDS>
__device__ __forceinline__ void tile_epilogue(
    const TileParams& p, floatx4_t (&acc)[TileStreams<EPI>::n * FNS][BM / WGM / 16], const float (&scale)[BM / WGM / 16],
    const int m0, const int col0, const int pieces, const int tile_n, const int wm, const int wn, const int lane,
    char* const lds) {
    constexpr int NW = WGM * WGN;
    constexpr int NS = TileStreams<EPI>::n;
    constexpr int WTM = BM / WGM;
    constexpr int FM = WTM / 16;
    const int M = p.M, N = p.N;
    const int r16 = lane & 15, q = lane >> 4;
    // the residual stream's old values: all asked for at once where the registers hold them
    // beside the sums, else a row of pieces at a time
    constexpr bool RES = EPI == T_RESIDUAL;
    constexpr bool OLD_AT_ONCE = FM * FNS <= 32;
    floatx4_t old_[RES && OLD_AT_ONCE ? FM : 1][RES ? FNS : 1];
    auto fetch_old = [&](int tm, floatx4_t (&to)[RES ? FNS : 1]) {
#pragma unroll
        for (int j = 0; j < (RES ? FNS : 1); ++j) {
            const int m = min(m0 + wm * WTM + tm * 16 + r16, M - 1);
            const int n = min(col0 + j * 16 + 4 * q, N - 4);
            to[j] = *reinterpret_cast<const floatx4_t*>(static_cast<const float*>(p.out) + static_cast<size_t>(m) * p.ldo + n);
        }
    };
    if (RES && OLD_AT_ONCE) {
#pragma unroll
        for (int tm = 0; tm < FM; ++tm) fetch_old(tm, old_[RES && OLD_AT_ONCE ? tm : 0]);
    }
    constexpr int PITCH = FNS * 32 + 16;          // bytes between a wavefront's rows in LDS
    constexpr bool VIA_LDS = ROWS_VIA_LDS && !RES;
    char* const corner = lds + static_cast<size_t>(wm * WGN + wn) * WTM * PITCH;
    if (VIA_LDS) __syncthreads();                 // the stages are no longer read
    float sq[FM];
#pragma unroll
    for (int tm = 0; tm < FM; ++tm) sq[tm] = 0.f;
#pragma unroll
    for (int tm = 0; tm < FM; ++tm) {
        const int m = m0 + wm * WTM + tm * 16 + r16;
        if (RES && !OLD_AT_ONCE) fetch_old(tm, old_[0]);
#pragma unroll
        for (int j = 0; j < FNS; ++j) {
            const int n = col0 + j * 16 + 4 * q;
            if (j >= pieces || m >= M || n >= N) continue;       // N % 4 == 0: a lane's four columns are inside together
            float v[NS][4];
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    v[s][i] = acc[s * FNS + j][tm][i] * scale[tm] +
                              (p.bias ? p.bias[static_cast<size_t>(s) * p.stream_rows + n + i] : 0.f);
            if (EPI == T_RESIDUAL) {
                float* const h = static_cast<float*>(p.out) + static_cast<size_t>(m) * p.ldo + n;
                floatx4_t old = old_[RES && OLD_AT_ONCE ? tm : 0][RES ? j : 0];
                // the product enters the sum rounded to bfloat16, as where it is a tensor of its own
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    old[i] += round_bf16(v[0][i]);
                    sq[tm] += old[i] * old[i];
                }
                *reinterpret_cast<floatx4_t*>(h) = old;
                if (p.out_bf16)     // (the conversion rounds to nearest even, as from_float<bf16>)
                    *reinterpret_cast<bf16x4_t*>(p.out_bf16 + static_cast<size_t>(m) * p.ld_bf16 + n) =
                        bf16x4_t{static_cast<__bf16>(old[0]), static_cast<__bf16>(old[1]),
                                 static_cast<__bf16>(old[2]), static_cast<__bf16>(old[3])};
            } else {
                float o[4];
                if constexpr (EPI == T_SWIGLU) {
                    float g[4], u[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        g[i] = round_bf16(v[0][i]);
                        u[i] = round_bf16(v[NS - 1][i]);
                    }
                    tile_swiglu(g, u, o);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] = v[0][i];
                }
                const bf16x4_t piece = bf16x4_t{static_cast<__bf16>(o[0]), static_cast<__bf16>(o[1]),
                                                static_cast<__bf16>(o[2]), static_cast<__bf16>(o[3])};
                if (VIA_LDS) *reinterpret_cast<bf16x4_t*>(corner + (tm * 16 + r16) * PITCH + (j * 16 + 4 * q) * 2) = piece;
                else *reinterpret_cast<bf16x4_t*>(static_cast<bf16*>(p.out) + static_cast<size_t>(m) * p.ldo + n) = piece;
            }
        }
    }
    if (VIA_LDS) {
        // (the wavefront reads what its own lanes wrote: LDS keeps a wavefront's accesses in order)
        const int cpr = pieces * 2;               // chunks of 8 columns a row
        const bool wide_stores = (p.ldo % 8) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0;
        for (int idx = lane; idx < WTM * cpr; idx += 64) {
            const int row = idx / cpr, ch = idx % cpr;
            const int m = m0 + wm * WTM + row, n = col0 + ch * 8;
            if (m >= M || n >= N) continue;
            const char* const from = corner + row * PITCH + ch * 16;
            bf16* const to = static_cast<bf16*>(p.out) + static_cast<size_t>(m) * p.ldo + n;
            if (wide_stores && n + 8 <= N) {
                *reinterpret_cast<bf16x8_t*>(to) = *reinterpret_cast<const bf16x8_t*>(from);
            } else {
                *reinterpret_cast<bf16x4_t*>(to) = *reinterpret_cast<const bf16x4_t*>(from);
                if (n + 8 <= N) *reinterpret_cast<bf16x4_t*>(to + 4) = *reinterpret_cast<const bf16x4_t*>(from + 8);
            }
        }
    }

    if (EPI == T_RESIDUAL && p.stats_out) {
        // a row's squares: over the lane's columns (above), the four lanes that share the
        // row, then the wavefronts that share it, always in the same order
        float* const red = reinterpret_cast<float*>(lds);
        __syncthreads();                          // the stages are no longer read
#pragma unroll
        for (int tm = 0; tm < FM; ++tm) {
            float s = sq[tm];
            s = sum_half32(sum_row16(s));
            if (q == 0) red[wn * BM + wm * WTM + tm * 16 + r16] = s;
        }
        __syncthreads();
        for (int r = threadIdx.x; r < BM; r += NW * 64) {
            float s = 0.f;
#pragma unroll
            for (int w = 0; w < WGN; ++w) s += red[w * BM + r];
            if (m0 + r < M) p.stats_out[static_cast<size_t>(m0 + r) * p.stats_ld_out + tile_n] = s;
        }
    }
}

// ---- the q/k/v epilogue (heads of 64 columns: a wavefront holds 16 or 32 rows of one head)
#define QKV_HD 64
// What it needs from memory, asked for before the product: the positions of the lane's rows
// and the head's norm weight at the lane's columns; and, lanes 0 .. rows-1 of the wavefront, the
// position and the slot of one row each (whose page is looked up once they have arrived).
template <int FM>
struct QkvEarly {
    int pos[FM];
    floatx4_t weight[4];
    int row_pos, row_slot, row_page;
};

template <int BM, int WGM, int WGN>
__device__ __forceinline__ void qkv_early_rows(const TileParams& p, QkvEarly<BM / WGM / 16>& e, const int m0, const int col0,
                                               const int wm, const int lane) {
    constexpr int WTM = BM / WGM, FM = WTM / 16;
    const int r16 = lane & 15, q = lane >> 4;
    const int head = min(col0, p.N - QKV_HD) / QKV_HD;
    const float* const weight = head < p.q_heads ? p.q_weight : (head < p.q_heads + p.kv_heads ? p.k_weight : nullptr);
#pragma unroll
    for (int tm = 0; tm < FM; ++tm) e.pos[tm] = p.positions[min(m0 + wm * WTM + tm * 16 + r16, p.M - 1)];
#pragma unroll
    for (int j = 0; j < 4; ++j)
        e.weight[j] = weight ? *reinterpret_cast<const floatx4_t*>(weight + j * 16 + 4 * q) : floatx4_t{1.f, 1.f, 1.f, 1.f};
    const int row = min(m0 + wm * WTM + min(lane, WTM - 1), p.M - 1);
    e.row_pos = p.positions[row];
    e.row_slot = p.token_slot[row];
    e.row_page = 0;
}

// (behind the first blocks' loads: the page of the lane's row)
template <int BM, int WGM, int WGN>
__device__ __forceinline__ void qkv_early_pages(const TileParams& p, QkvEarly<BM / WGM / 16>& e, const int col0) {
    const int head = min(col0, p.N - QKV_HD) / QKV_HD;
    if (head >= p.q_heads)
        e.row_page = p.table[static_cast<size_t>(e.row_slot) * p.table_stride + e.row_pos / p.page_tokens];
}

// acc[j][tm][i]: row .. + tm*16 + lane%16, column col0 + j*16 + 4*(lane/16) + i of the head at col0.
// The sums are rounded to bfloat16 first, as where the product is a tensor of its own; norm,
// rotation (split halves: pair (c, c + 32)) as qk_norm_rope_store makes them.  The head's rows
// go to the wavefront's corner of LDS and leave from there: query rows to `out`, key rows to
// their places in the pages, values by groups of four tokens that lie side by side in a page.
template <int BM, int WGM, int WGN>
__device__ __forceinline__ void qkv_epilogue(const TileParams& p, floatx4_t (&acc)[4][BM / WGM / 16],
                                             const float (&scale)[BM / WGM / 16], const QkvEarly<BM / WGM / 16>& e,
                                             const int m0, const int col0, const int wm, const int wn, const int lane,
                                             char* const lds) {
    constexpr int WTM = BM / WGM, FM = WTM / 16;
    constexpr int PITCH = QKV_HD * 2 + 16;            // bytes between a wavefront's rows in LDS
    constexpr int CORNER = WTM * PITCH + WTM * 16;    // the rows, then (position, slot, page, -) of every row
    const int M = p.M;
    const int r16 = lane & 15, q = lane >> 4;
    char* const corner = lds + static_cast<size_t>(wm * WGN + wn) * CORNER;
    int* const rowinfo = reinterpret_cast<int*>(corner + WTM * PITCH);
    const int head = min(col0, p.N - QKV_HD) / QKV_HD;
    const bool is_q = head < p.q_heads, is_k = !is_q && head < p.q_heads + p.kv_heads;
    const int kv_head = is_q ? 0 : (is_k ? head - p.q_heads : head - p.q_heads - p.kv_heads);
    const bool normed = is_q ? p.q_weight != nullptr : (is_k && p.k_weight != nullptr);
    const bool rotate = p.cos_sin && (is_q || is_k);
    // (cos, sin) of the lane's 2 x 4 column pairs for each of its rows: asked for only now (the
    // registers they take would cost the product a wavefront a SIMD), ahead of the barrier
    floatx4_t cs[FM][4];
    if (rotate) {
#pragma unroll
        for (int tm = 0; tm < FM; ++tm) {
            const float* const c = p.cos_sin + static_cast<size_t>(e.pos[tm]) * QKV_HD;     // 32 pairs of two
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                cs[tm][2 * j] = *reinterpret_cast<const floatx4_t*>(c + (j * 16 + 4 * q) * 2);
                cs[tm][2 * j + 1] = *reinterpret_cast<const floatx4_t*>(c + (j * 16 + 4 * q) * 2 + 4);
            }
        }
    }
    __syncthreads();                                  // the stages are no longer read
    if (col0 >= p.N) return;                          // (a tile that hangs over the last head)
#pragma unroll
    for (int tm = 0; tm < FM; ++tm) {
        float x[4][4];
        float ssq = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[j][i] = round_bf16(acc[j][tm][i] * scale[tm] + (p.bias ? p.bias[col0 + j * 16 + 4 * q + i] : 0.f));
                ssq += x[j][i] * x[j][i];
            }
        if (normed) {
            ssq = sum_half32(sum_row16(ssq));
            const float inv = 1.0f / sqrtf(ssq / static_cast<float>(QKV_HD) + p.qk_eps);
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) x[j][i] = x[j][i] * inv * e.weight[j][i];
        }
        if (rotate) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    // (cos, sin) of pair j*16 + 4q + i: four pairs are two loads of four floats
                    const float c = i < 2 ? cs[tm][2 * j][2 * i] : cs[tm][2 * j + 1][2 * (i - 2)];
                    const float s = i < 2 ? cs[tm][2 * j][2 * i + 1] : cs[tm][2 * j + 1][2 * (i - 2) + 1];
                    const float a = x[j][i], b = x[j + 2][i];
                    x[j][i] = a * c - b * s;
                    x[j + 2][i] = b * c + a * s;
                }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *reinterpret_cast<bf16x4_t*>(corner + (tm * 16 + r16) * PITCH + (j * 16 + 4 * q) * 2) =
                bf16x4_t{static_cast<__bf16>(x[j][0]), static_cast<__bf16>(x[j][1]), static_cast<__bf16>(x[j][2]),
                         static_cast<__bf16>(x[j][3])};
    }
    if (lane < WTM) {
        rowinfo[4 * lane] = e.row_pos;
        rowinfo[4 * lane + 1] = e.row_slot;
        rowinfo[4 * lane + 2] = e.row_page;
    }
    // (the wavefront reads what its own lanes wrote: LDS keeps a wavefront's accesses in order)
    const int page_mask = p.page_tokens - 1;
    const int row_base = m0 + wm * WTM;
    if (is_q || is_k) {
        for (int idx = lane; idx < WTM * 8; idx += 64) {
            const int row = idx >> 3, ch = idx & 7;
            if (row_base + row >= M) continue;
            const bf16x8_t piece = *reinterpret_cast<const bf16x8_t*>(corner + row * PITCH + ch * 16);
            bf16* to;
            if (is_q) {
                to = static_cast<bf16*>(p.out) + static_cast<size_t>(row_base + row) * p.ldo + col0 + ch * 8;
            } else {
                const int pos = rowinfo[4 * row], page = rowinfo[4 * row + 2];
                to = p.k_pool + (((static_cast<size_t>(page) * p.n_layers + p.layer) * p.kv_heads + kv_head) * p.page_tokens +
                                 (pos & page_mask)) * QKV_HD + ch * 8;
            }
            *reinterpret_cast<bf16x8_t*>(to) = piece;
        }
        return;
    }
    // values: [dimension][token] inside a page
    for (int u = lane; u < (WTM / 4) * QKV_HD; u += 64) {
        const int g = u % (WTM / 4), d = u / (WTM / 4);
        const int r0 = 4 * g;
        const int pos0 = rowinfo[4 * r0], slot0 = rowinfo[4 * r0 + 1];
        bool together = row_base + r0 + 3 < M && (pos0 & 3) == 0;
        unsigned short val[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            together = together && rowinfo[4 * (r0 + k)] == pos0 + k && rowinfo[4 * (r0 + k) + 1] == slot0;
            val[k] = *reinterpret_cast<const unsigned short*>(corner + (r0 + k) * PITCH + d * 2);
        }
        if (together) {
            bf16* const to = p.v_pool + ((static_cast<size_t>(rowinfo[4 * r0 + 2]) * p.n_layers + p.layer) * p.kv_heads + kv_head) *
                                            p.page_tokens * QKV_HD + static_cast<size_t>(d) * p.page_tokens + (pos0 & page_mask);
            *reinterpret_cast<uint2*>(to) = uint2{static_cast<unsigned>(val[0]) | (static_cast<unsigned>(val[1]) << 16),
                                                  static_cast<unsigned>(val[2]) | (static_cast<unsigned>(val[3]) << 16)};
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (row_base + r0 + k >= M) continue;
                const int pos = rowinfo[4 * (r0 + k)], page = rowinfo[4 * (r0 + k) + 2];
                unsigned short* const to = reinterpret_cast<unsigned short*>(
                    p.v_pool + ((static_cast<size_t>(page) * p.n_layers + p.layer) * p.kv_heads + kv_head) * p.page_tokens * QKV_HD +
                    static_cast<size_t>(d) * p.page_tokens + (pos & page_mask));
                *to = val[k];
            }
        }
    }
}

// A tile whose K is cut over several workgroups: each leaves its sums in memory and counts itself in; the last one to arrive
// adds them all up, in the order of the slices, and goes on (true), the others are done.  Nobody waits for anybody.
// The sums are written and read past the dies' caches (accesses of device scope), and they have arrived where a wavefront's
// count of accesses in flight is down to none: no cache is written back or invalidated in between.
// [tile][slice][wavefront][piece][lane] of four sums.
template <int NW, int FN, int FM>
__device__ __forceinline__ bool tile_join(const TileParams& p, floatx4_t (&acc)[FN][FM], const int tile, const int slice,
                                          const int wave, const int lane, char* const lds) {
    typedef unsigned long long u64;
    constexpr int PIECES = FN * FM;
    const int slices = p.k_slices;
    const auto part = [&](int s, int piece) {
        return reinterpret_cast<u64*>(p.parts) + (((static_cast<size_t>(tile) * slices + s) * NW + wave) * PIECES + piece) * 128 + 2 * lane;
    };
    floatx4_t own[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        own[i] = acc[i / FM][i % FM];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float pair[2] = {own[i][2 * h], own[i][2 * h + 1]};
            __hip_atomic_store(part(slice, i) + h, __builtin_bit_cast(u64, pair), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                              // (the stages are no longer read)
    if (threadIdx.x == 0)
        *reinterpret_cast<int*>(lds) = __hip_atomic_fetch_add(p.arrived + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const bool last = *reinterpret_cast<int*>(lds) == slices - 1;
    __syncthreads();
    if (!last) return false;
    if (threadIdx.x == 0) __hip_atomic_store(p.arrived + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);     // (for the next launch)
#pragma unroll
    for (int i = 0; i < PIECES; ++i) acc[i / FM][i % FM] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < slices; ++s) {
        u64 v[PIECES][2];
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) v[i][h] = __hip_atomic_load(part(s, i) + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i < PIECES; ++i) acc[i / FM][i % FM] += s == slice ? own[i] : __builtin_bit_cast(floatx4_t, v[i]);
    }
    return true;
}

// PACKED: the weights are.  SPLIT: p.k_slices workgroups a tile share its K.
template <int BM, int BN, int WGM, int WGN, int STAGES, int EPI, bool PACKED, bool SPLIT>
__global__ __launch_bounds__(WGM * WGN * 64)
void gemm_tiles_kernel(const TileParams p, const int tiles_m, const int tiles_n, const int dies_m) {
    constexpr int NW = WGM * WGN;
    constexpr int NS = TileStreams<EPI>::n;
    constexpr int WTM = BM / WGM, WTN = BN / WGN;
    constexpr int FM = WTM / 16, FN = WTN / 16;
    constexpr int STAGE_BYTES = (BM + BN) * 128;
    constexpr int GROUPS = (BM + BN) / 8;          // loads of 1 KB a block of k
    constexpr int GPW = (GROUPS + NW - 1) / NW;    // of which a wavefront issues this many (where they do
                                                   // not divide, the last ones ask for the last group again)
    static_assert(FN % NS == 0 && WTM % 16 == 0 && WTN % 16 == 0, "tile shape");
    static_assert(GPW * STAGES < 64, "more loads in flight than the counter holds");
    static_assert(!PACKED || (BM / 8 % NW == 0 && EPI == T_RESIDUAL), "a wavefront's load i is of A or of packed weights");
    extern __shared__ __attribute__((aligned(1024))) char lds[];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int wm = wave / WGN, wn = wave % WGN;
    const int M = p.M, N = p.N, K = p.K;

    // Workgroups go to the 8 dies in turn, and every die has an L2 of its own: die x gets the
    // tiles of a rectangle of the tile grid (dies_m x dies_n rectangles), walked down its rows
    // first, so that the tiles that run together on a die share rows of A and of W and each
    // operand crosses the fabric behind the L2s few times.
    const int dies_n = 8 / dies_m;
    const int die = blockIdx.x & 7, local = blockIdx.x >> 3;
    const int di = die / dies_n, dj = die % dies_n;
    const int r0 = di * tiles_m / dies_m, rows = (di + 1) * tiles_m / dies_m - r0;
    const int c0 = dj * tiles_n / dies_n, cols = (dj + 1) * tiles_n / dies_n - c0;
    const int slices = SPLIT ? p.k_slices : 1;
    if (local >= rows * cols * slices) return;
    const int slice = SPLIT ? local % slices : 0, place = SPLIT ? local / slices : local;
    const int tile_n = c0 + place / rows;
    const int tile_m = r0 + place % rows, m0 = tile_m * BM;
    const int n0 = tile_n * (BN / NS);

    // ---- what this lane asks memory for: group g = wave + i * NW, rows 8g .. 8g+7 of the stage
    const int first_kb = SPLIT ? slice * (K >> 6) / slices : 0;
    const size_t w_next = PACKED ? static_cast<size_t>(p.w_block) * 4 : 128;      // bytes from a block of weights to the next
    const char* src[GPW];
#pragma unroll
    for (int i = 0; i < GPW; ++i) {
        const int g = min(wave + i * NW, GROUPS - 1);
        const int row = 8 * g + (lane >> 3);               // the row whose chunk lands at this lane's place
        const int chunk = (lane & 7) ^ (row & 7);
        if (g < BM / 8) {
            const int m = min(m0 + row, M - 1);
            src[i] = reinterpret_cast<const char*>(p.a + static_cast<size_t>(m) * p.lda) + chunk * 16;
        } else if (PACKED) {
            // 16 rows of half a block of k: the first half's groups, then the second's
            const int half = (g - BM / 8) / (BN / 16), b = (g - BM / 8) % (BN / 16) * 16 + (lane >> 2);
            const int s = b / (BN / NS), n = min(n0 + b % (BN / NS), N - 1);
            src[i] = reinterpret_cast<const char*>(p.w + half * p.w_block + (static_cast<size_t>(s) * p.stream_rows + n) * 32) +
                     ((lane & 3) ^ ((b >> 1) & 3)) * 16;
        } else {
            const int b = row - BM;
            const int s = b / (BN / NS), j = b % (BN / NS);
            const int n = min(n0 + j, N - 1);
            src[i] = reinterpret_cast<const char*>(p.w + (static_cast<size_t>(s) * p.stream_rows + n) * p.ldw) + chunk * 16;
        }
        if (SPLIT) src[i] += static_cast<size_t>(first_kb) * (g < BM / 8 ? 128 : w_next);
    }
    auto issue = [&](int stage, int kb) {
        char* const base = lds + stage * STAGE_BYTES;
#pragma unroll
        for (int i = 0; i < GPW; ++i)
            __builtin_amdgcn_global_load_lds(GPTR(src[i] + static_cast<size_t>(kb) * (i < BM / 8 / NW ? 128 : w_next)),
                                             LPTR(base + min(wave + i * NW, GROUPS - 1) * 1024), 16, 0, 0);
    };

    // ---- where this lane's operands lie inside a 16-row piece of a stage (k-step 0 and 1)
    const int r16 = lane & 15, q = lane >> 4;
    int lane_off[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
        lane_off[ks] = r16 * 128 + (((ks * 4 + q) ^ (r16 & 7)) * 16);
    const int packed_off = r16 * 64 + ((q ^ ((r16 >> 1) & 3)) * 16);

    floatx4_t acc[FN][FM];
#pragma unroll
    for (int tn = 0; tn < FN; ++tn)
#pragma unroll
        for (int tm = 0; tm < FM; ++tm) acc[tn][tm] = floatx4_t{0.f, 0.f, 0.f, 0.f};

    // ---- the rows' 1/rms, asked for ahead of the first blocks
    float scale[FM];
    tile_row_scales<FM>(p, m0 + wm * WTM + r16, q, scale);
    QkvEarly<EPI == T_QKV ? FM : 1> qkv_early;
    if constexpr (EPI == T_QKV) qkv_early_rows<BM, WGM, WGN>(p, qkv_early, m0, n0 + wn * WTN, wm, lane);

    const int nkb = (SPLIT ? (slice + 1) * (K >> 6) / slices : K >> 6) - first_kb;      // K % 64 == 0 (checked by the host)
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
        if (s < nkb) issue(s, s);
    if constexpr (EPI == T_QKV) qkv_early_pages<BM, WGM, WGN>(p, qkv_early, n0 + wn * WTN);

    // Operands of a k-step (32 values of k) travel from LDS to registers one step ahead of
    // the matrix instructions that use them: a wavefront asks for step 1 of a block, then
    // multiplies step 0; at the barrier in the middle everybody holds the whole block in
    // registers, so its stage is refilled there, and step 0 of the next block is asked for
    // before step 1 is multiplied.
    bf16x8_t af[2][FM], wf[2][FN];
    auto fetch = [&](int stage, int ks, bf16x8_t (&a)[FM], bf16x8_t (&w)[FN]) {
        const char* const sa = lds + stage * STAGE_BYTES + (wm * WTM) * 128 + lane_off[ks];
        const char* const sw = lds + stage * STAGE_BYTES + BM * 128 + (PACKED ? ks * BN * 64 + packed_off : lane_off[ks]);
#pragma unroll
        for (int tm = 0; tm < FM; ++tm) a[tm] = *reinterpret_cast<const bf16x8_t*>(sa + tm * 2048);
#pragma unroll
        for (int tn = 0; tn < FN; ++tn) {
            const int brow = (tn / (FN / NS)) * (BN / NS) + wn * (WTN / NS) + (tn % (FN / NS)) * 16;
            w[tn] = *reinterpret_cast<const bf16x8_t*>(sw + brow * (PACKED ? 64 : 128));
        }
    };
    auto multiply = [&](const bf16x8_t (&a)[FM], const bf16x8_t (&w)[FN]) {
#pragma unroll
        for (int tn = 0; tn < FN; ++tn)
#pragma unroll
            for (int tm = 0; tm < FM; ++tm)
                acc[tn][tm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[tn], a[tm], acc[tn][tm], 0, 0, 0);
    };
    // block 0 has arrived when at most the later blocks' loads are out
    if (STAGES - 1 < nkb) wait_loads<GPW * (STAGES - 1)>(); else wait_loads<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fetch(0, 0, af[0], wf[0]);
    int stage = 0;
    for (int kb = 0; kb < nkb; ++kb) {
        fetch(stage, 1, af[1], wf[1]);
        multiply(af[0], wf[0]);
        int next = stage + 1;
        if (next == STAGES) next = 0;
        if (kb + 1 < nkb) {
            if (kb + STAGES - 1 < nkb) wait_loads<GPW * (STAGES - 2)>(); else wait_loads<0>();
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (kb + STAGES < nkb) issue(stage, kb + STAGES);
            fetch(next, 0, af[0], wf[0]);
        }
        multiply(af[1], wf[1]);
        stage = next;
    }

    if constexpr (SPLIT) {
        if (!tile_join<NW>(p, acc, tile_m * tiles_n + tile_n, slice, wave, lane, lds)) return;
    }
    if constexpr (EPI == T_QKV) {
        static_assert(EPI != T_QKV || (WTN == QKV_HD && FN == 4), "a wavefront holds one head of 64 columns");
        qkv_epilogue<BM, WGM, WGN>(p, acc, scale, qkv_early, m0, n0 + wn * WTN, wm, wn, lane, lds);
    } else {
        tile_epilogue<BM, WGM, WGN, FN / NS, EPI, false>(p, acc, scale, m0, n0 + wn * (WTN / NS), FN / NS, tile_n, wm, wn, lane, lds);
    }
}

// A read of 16 bytes a lane from LDS at `address` + index * STRIDE, and the waits that go with
// such reads, written as instructions: the compiler does not see the read, so every use of
// `to` has to come behind a wait that names it (the wait takes the registers in and out, which
// keeps the uses behind it), with no branch and no indexing by a variable in between (either
// would let the compiler copy the registers before the data is there).  `left`: how many later
// reads may still be out.
template <int STRIDE>
__device__ __forceinline__ void lds_read(bf16x8_t& to, const unsigned address, const int index) {
    switch (index) {
#define CELEG_LDS_READ_CASE(I) \
    case I: asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(to) : "v"(address), "n"(I * STRIDE)); break;
        CELEG_LDS_READ_CASE(0) CELEG_LDS_READ_CASE(1) CELEG_LDS_READ_CASE(2) CELEG_LDS_READ_CASE(3)
        CELEG_LDS_READ_CASE(4) CELEG_LDS_READ_CASE(5) CELEG_LDS_READ_CASE(6) CELEG_LDS_READ_CASE(7)
        CELEG_LDS_READ_CASE(8) CELEG_LDS_READ_CASE(9) CELEG_LDS_READ_CASE(10) CELEG_LDS_READ_CASE(11)
#undef CELEG_LDS_READ_CASE
        default: __builtin_trap();
    }
}
__device__ __forceinline__ void lds_wait(const int left, bf16x8_t& x) {
    switch (left) {
        case 0: asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(x)); break;
        case 1: asm volatile("s_waitcnt lgkmcnt(1)" : "+v"(x)); break;
        case 2: asm volatile("s_waitcnt lgkmcnt(2)" : "+v"(x)); break;
        default: asm volatile("s_waitcnt lgkmcnt(3)" : "+v"(x)); break;
    }
}
template <int FM>
__device__ __forceinline__ void lds_wait_rows(const int left, bf16x8_t& x, bf16x8_t (&rows)[FM]) {
    lds_wait(left, x);
#pragma unroll
    for (int tm = 0; tm < FM; ++tm) asm volatile("" : "+v"(rows[tm]));     // (behind the wait above: volatile statements keep their order)
}

// The reads from LDS of a block of the wide kernel, in the order of issue: the rows' operands of step 0,
// weights 0 and 1; then with piece t = step * FN + j weights t + 2 and, for the first FM pieces of a step,
// one of the rows' operands of the next step.  LDS answers in this order.
template <int FM, int FN, int KS>
struct WideReads {
    static constexpr int PIECES = KS * FN;
    static_assert(FM <= FN, "the rows' operands of a step are asked for with the pieces of the step before");
    static constexpr bool row_with(int t) { return t / FN + 1 < KS && t % FN < FM; }
    // reads that are asked for ahead of piece t
    static constexpr int ahead_of(int t) {
        int n = FM + 2;
        for (int p = 0; p < t; ++p) n += (p + 2 < PIECES ? 1 : 0) + (row_with(p) ? 1 : 0);
        return n;
    }
    static constexpr int weights(int t) { return t < 2 ? FM + t : ahead_of(t - 2); }           // the place of weights t
    static constexpr int last_row(int t) {         // the place of the last of the rows' operands of piece t's step
        const int with = (t / FN - 1) * FN + FM - 1;
        return t < FN ? FM - 1 : ahead_of(with) + (with + 2 < PIECES ? 1 : 0);
    }
    // how many reads may still be out where piece t starts: those behind its weights and its step's rows, whichever
    // is later (the rows where FM > FN - 2)
    static constexpr int may_be_out(int t) {
        const int needed = weights(t) > last_row(t) ? weights(t) : last_row(t);
        return ahead_of(t) - 1 - needed;
    }
    // the reads replayed: where piece t starts, its weights and all rows' operands of its step are there
    static constexpr bool sound() {
        int weight_at[PIECES] = {}, row_at[KS][FM] = {}, asked = 0;
        for (int r = 0; r < FM; ++r) row_at[0][r] = asked++;
        weight_at[0] = asked++;
        weight_at[1] = asked++;
        for (int t = 0; t < PIECES; ++t) {
            const int there = asked - may_be_out(t);
            if (may_be_out(t) < 0 || may_be_out(t) > 3 || weight_at[t] >= there) return false;      // (lds_wait counts to 3)
            for (int r = 0; r < FM; ++r)
                if (row_at[t / FN][r] >= there) return false;
            if (t + 2 < PIECES) weight_at[t + 2] = asked++;
            if (row_with(t)) row_at[t / FN + 1][t % FN] = asked++;
        }
        return true;
    }
};

// SwiGLU of a wide tile whose wavefronts each hold columns of one stream only: gate and up
// (rounded to bfloat16, as where they are tensors of their own) meet in LDS, [stream][row], and
// leave as whole rows, 16 bytes a lane.
template <int BM, int BN, int WGM, int WGN>
__device__ __forceinline__ void wide_swiglu_epilogue(
    const TileParams& p, floatx4_t (&acc)[BN / 16 / WGN][BM / WGM / 16], const float (&scale)[BM / WGM / 16],
    const int m0, const int n0, const int wm, const int wn, const int lane, char* const lds) {
    constexpr int NW = WGM * WGN, WTM = BM / WGM, FM = WTM / 16, FN = BN / 16 / WGN;
    constexpr int PS = BN / 32;                   // column pieces of a stream
    constexpr int OC = BN / 2, PITCH = OC * 2 + 16;
    const int M = p.M, N = p.N;
    const int r16 = lane & 15, q = lane >> 4;
    const int s = (wn * FN) / PS, j0 = (wn * FN) % PS;
    __syncthreads();                              // the stages are no longer read
    char* const mine = lds + static_cast<size_t>(s) * BM * PITCH;
    floatx4_t bias[FN];                           // of the lane's columns
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int n = n0 + (j0 + j) * 16 + 4 * q;
        bias[j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
        if (p.bias && n < N) bias[j] = *reinterpret_cast<const floatx4_t*>(p.bias + static_cast<size_t>(s) * p.stream_rows + n);
    }
#pragma unroll
    for (int tm = 0; tm < FM; ++tm)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const floatx4_t v = acc[j][tm] * scale[tm] + bias[j];
            *reinterpret_cast<bf16x4_t*>(mine + (wm * WTM + tm * 16 + r16) * PITCH + ((j0 + j) * 16 + 4 * q) * 2) =
                bf16x4_t{static_cast<__bf16>(v[0]), static_cast<__bf16>(v[1]), static_cast<__bf16>(v[2]), static_cast<__bf16>(v[3])};
        }
    __syncthreads();
    constexpr int CPR = OC / 8;                   // chunks of 8 columns a row
    const bool wide_stores = (p.ldo % 8) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0;
    for (int idx = threadIdx.x; idx < BM * CPR; idx += NW * 64) {
        const int row = idx / CPR, ch = idx % CPR;
        const int m = m0 + row, n = n0 + ch * 8;
        if (m >= M || n >= N) continue;
        const bf16x8_t g = *reinterpret_cast<const bf16x8_t*>(lds + row * PITCH + ch * 16);
        const bf16x8_t u = *reinterpret_cast<const bf16x8_t*>(lds + static_cast<size_t>(BM) * PITCH + row * PITCH + ch * 16);
        float gate[8], up[8], y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            gate[i] = static_cast<float>(g[i]);
            up[i] = static_cast<float>(u[i]);
        }
        tile_swiglu(gate, up, y);
        bf16x8_t o;
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = static_cast<__bf16>(y[i]);
        bf16* const to = static_cast<bf16*>(p.out) + static_cast<size_t>(m) * p.ldo + n;
        if (wide_stores && n + 8 <= N) {
            store_through(reinterpret_cast<bf16x8_t*>(to), o);
        } else {
            *reinterpret_cast<bf16x4_t*>(to) = bf16x4_t{o[0], o[1], o[2], o[3]};
            if (n + 8 <= N) *reinterpret_cast<bf16x4_t*>(to + 4) = bf16x4_t{o[4], o[5], o[6], o[7]};
        }
    }
}

// The same product with wide tiles (256 rows x up to 288 weight rows a workgroup), for the
// products whose operands would otherwise cross from the L2 caches to the compute units many
// times over.  A wavefront's tile is too large to hold a block's operands in registers beside
// its sums, so the weights' operands stream from LDS a piece (16 weight rows) at a time, two
// pieces ahead of the matrix instructions that use them, and the rows' operands of the next
// step of 32 values of k come in between; the order is pinned (sched_barrier) and the reads and
// their waits are written as instructions, because left alone the compiler reads two pieces
// into the same registers, waits for them, multiplies, and reads again.  Blocks are KB = 32 or 64 values of k (rows of 64 or 128 bytes in LDS, a load
// instruction fills 16 or 8 rows), STAGES of them, with one barrier a block: behind it
// everybody's loads of this block have landed and nobody reads the block before any more,
// whose stage the loads of block + STAGES - 1 then fill.  Chunk c (16 bytes) of row r lies at
// chunk c ^ ((r / 4) % 4) (rows of 64 bytes) or c ^ (r % 8) (128), so that the 16 rows that
// lanes read at one chunk fall on all banks.  Rows of 64 bytes ask memory for half a cache
// line at a time, and the vector cache fetches the whole line for each half (measured: the
// loads alone then take a third longer).
// The tile's BN / 16 column pieces (gate pieces, then up pieces) are dealt evenly to the WGN
// wavefronts of a row of wavefronts, each within one stream.
template <int BM, int BN, int WGM, int WGN, int STAGES, int KB, int EPI>
__global__ __launch_bounds__(WGM * WGN * 64)
void gemm_tiles_wide_kernel(const TileParams p, const int tiles_m, const int tiles_n, const int dies_m) {
    constexpr int NW = WGM * WGN;
    constexpr int NS = TileStreams<EPI>::n;
    constexpr int WTM = BM / WGM;
    constexpr int FM = WTM / 16;
    constexpr int FN = BN / 16 / WGN;              // column pieces of a wavefront
    constexpr int PS = BN / 16 / NS;               // column pieces of a stream in the tile
    constexpr int KS = KB / 32;                    // steps of 32 values of k a block
    constexpr int ROW_BYTES = KB * 2, CPR = ROW_BYTES / 16, RPL = 1024 / ROW_BYTES;   // chunks a row, rows a load
    constexpr int STAGE_BYTES = (BM + BN) * ROW_BYTES;
    constexpr int GROUPS = (BM + BN) / RPL;        // loads of 1 KB a block of k
    constexpr int GPW = (GROUPS + NW - 1) / NW;
    static_assert(BN % (16 * WGN) == 0 && BN % (16 * NS) == 0 && PS % FN == 0 && WTM % 16 == 0 &&
                  (BM + BN) % 16 == 0 && STAGES >= 2 && FN >= 2 && FN <= 12 && FM <= 12 && (KB == 32 || KB == 64), "tile shape");
    static_assert(GPW * STAGES < 64, "more loads in flight than the counter holds");
    using Reads = WideReads<FM, FN, KS>;
    static_assert(Reads::sound(), "an operand is used ahead of its read");
    extern __shared__ __attribute__((aligned(1024))) char lds[];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int wm = wave / WGN, wn = wave % WGN;
    const int M = p.M, N = p.N, K = p.K;

    // (the dies' rectangles: as in gemm_tiles_kernel)
    const int dies_n = 8 / dies_m;
    const int die = blockIdx.x & 7, local = blockIdx.x >> 3;
    const int di = die / dies_n, dj = die % dies_n;
    const int r0 = di * tiles_m / dies_m, rows = (di + 1) * tiles_m / dies_m - r0;
    const int c0 = dj * tiles_n / dies_n, cols = (dj + 1) * tiles_n / dies_n - c0;
    if (local >= rows * cols) return;
    const int tile_n = c0 + local / rows;
    const int m0 = (r0 + local % rows) * BM;
    const int n0 = tile_n * (BN / NS);

    // ---- what this lane asks memory for: group g, rows RPL*g .. of the stage
    const char* src[GPW];
#pragma unroll
    for (int i = 0; i < GPW; ++i) {
        const int g = min(wave + i * NW, GROUPS - 1);
        const int row = RPL * g + lane / CPR;
        const int chunk = (lane % CPR) ^ (KB == 32 ? (row >> 2) & 3 : row & 7);
        if (row < BM) {
            const int m = min(m0 + row, M - 1);
            src[i] = reinterpret_cast<const char*>(p.a + static_cast<size_t>(m) * p.lda) + chunk * 16;
        } else {
            const int b = row - BM;
            const int s = b / (BN / NS), j = b % (BN / NS);
            const int n = min(n0 + j, N - 1);
            src[i] = reinterpret_cast<const char*>(p.w + (static_cast<size_t>(s) * p.stream_rows + n) * p.ldw) + chunk * 16;
        }
    }
    auto issue = [&](int stage, int kb) {
        char* const base = lds + stage * STAGE_BYTES;
#pragma unroll
        for (int i = 0; i < GPW; ++i)
            __builtin_amdgcn_global_load_lds(GPTR(src[i] + static_cast<size_t>(kb) * ROW_BYTES),
                                             LPTR(base + min(wave + i * NW, GROUPS - 1) * 1024), 16, 0, 0);
    };

    const int r16 = lane & 15, q = lane >> 4;
    int lane_off[KS];                             // per step of 32 values of k
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
        lane_off[ks] = r16 * ROW_BYTES + (((ks * 4 + q) ^ (KB == 32 ? (r16 >> 2) & 3 : r16 & 7)) * 16);

    floatx4_t acc[FN][FM];
#pragma unroll
    for (int tn = 0; tn < FN; ++tn)
#pragma unroll
        for (int tm = 0; tm < FM; ++tm) acc[tn][tm] = floatx4_t{0.f, 0.f, 0.f, 0.f};

    float scale[FM];                              // (asked for ahead of the first blocks)
    tile_row_scales<FM>(p, m0 + wm * WTM + r16, q, scale);

    const int nkb = K / KB;                       // K % 64 == 0 (checked by the host)
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
        if (s < nkb) issue(s, s);

    const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<uintptr_t>(LPTR(lds)));
    int stage = 0;
    for (int kb = 0; kb < nkb; ++kb) {
        // this wavefront's loads of block kb have landed when at most the later blocks' are out
        if (kb + STAGES - 2 < nkb) wait_loads<GPW * (STAGES - 2)>(); else wait_loads<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        int refill = stage - 1;
        if (refill < 0) refill = STAGES - 1;
        if (kb + STAGES - 1 < nkb) issue(refill, kb + STAGES - 1);
        __builtin_amdgcn_sched_barrier(0);
        // LDS addresses of this lane's operands per step of 32 values of k; pieces are 16 rows apart
        unsigned at_a[KS], at_w[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            at_a[ks] = lds_base + stage * STAGE_BYTES + (wm * WTM) * ROW_BYTES + lane_off[ks];
            at_w[ks] = lds_base + stage * STAGE_BYTES + (BM + wn * FN * 16) * ROW_BYTES + lane_off[ks];
        }
        // The reads and the waits for them are written out (the compiler, left to count, waits for
        // every read in flight before each second piece).  Piece t = ks * FN + j of the block: step
        // ks, column piece j; its reads go behind its first matrix instruction (WideReads: their order).
        bf16x8_t a[2][FM], w[3];
#pragma unroll
        for (int tm = 0; tm < FM; ++tm) lds_read<16 * ROW_BYTES>(a[0][tm], at_a[0], tm);
        lds_read<16 * ROW_BYTES>(w[0], at_w[0], 0);
        lds_read<16 * ROW_BYTES>(w[1], at_w[1 / FN < KS ? 1 / FN : 0], 1 % FN);
#pragma unroll
        for (int t = 0; t < KS * FN; ++t) {
            const int ks = t / FN, j = t % FN;
            if (j == 0) lds_wait_rows(Reads::may_be_out(t), w[t % 3], a[ks & 1]);
            else lds_wait(Reads::may_be_out(t), w[t % 3]);
            acc[j][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t % 3], a[ks & 1][0], acc[j][0], 0, 0, 0);
            if (t + 2 < KS * FN) lds_read<16 * ROW_BYTES>(w[(t + 2) % 3], at_w[(t + 2) / FN < KS ? (t + 2) / FN : 0], (t + 2) % FN);
            if (Reads::row_with(t)) lds_read<16 * ROW_BYTES>(a[(ks + 1) & 1][j < FM ? j : 0], at_a[ks + 1 < KS ? ks + 1 : 0], j);
#pragma unroll
            for (int tm = 1; tm < FM; ++tm)
                acc[j][tm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t % 3], a[ks & 1][tm], acc[j][tm], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (++stage == STAGES) stage = 0;
    }
    if constexpr (EPI == T_SWIGLU) {
        wide_swiglu_epilogue<BM, BN, WGM, WGN>(p, acc, scale, m0, n0, wm, wn, lane, lds);
    } else {
        // (rows leave through LDS where the stages have room for the whole tile's output)
        constexpr bool ROWS_FIT = NW * WTM * (FN * 32 + 16) <= STAGES * STAGE_BYTES;
        tile_epilogue<BM, WGM, WGN, FN, EPI, ROWS_FIT>(p, acc, scale, m0, n0 + wn * FN * 16, FN, tile_n, wm, wn, lane, lds);
    }
}

// ---- the shape of the work for given sizes
struct TileShape {
    int id;         // index into the table below
    int bm, bn;     // bn counts weight rows of all streams
    int slices;     // workgroups a tile, which share its K
};

// For tests and tuning: a shape that overrides the choice below (-1: none).
static int g_force_shape = -1, g_force_dies_m = 0;
extern "C" void celeg_gemm_tiles_force(int shape) { g_force_shape = shape; }
extern "C" void celeg_gemm_tiles_force_dies(int dies_m) { g_force_dies_m = dies_m; }

// id, rows, weight rows, wavefronts along rows and along weight rows, stages, values of k a block of
// the wide kernel (0: the kernel with tiles up to 128x192)
#define TILE_SHAPES(X) \
    X(0, 32, 64, 2, 2, 8, 0)  \
    X(1, 64, 64, 4, 2, 4, 0)  \
    X(2, 128, 64, 4, 2, 4, 0) \
    X(3, 64, 128, 2, 4, 4, 0) \
    X(4, 64, 192, 4, 2, 4, 0) \
    X(5, 64, 128, 2, 2, 3, 0) \
    X(6, 128, 128, 4, 2, 4, 0) \
    X(7, 128, 192, 4, 2, 3, 0) \
    X(8, 128, 128, 4, 2, 2, 0) \
    X(9, 256, 192, 4, 2, 2, 64) \
    X(10, 256, 288, 4, 2, 2, 64) \
    X(11, 256, 256, 4, 2, 2, 64)

#define TILE_ROWS(ID, BM, BN, WGM, WGN, STAGES, KB) BM,
#define TILE_COLUMNS(ID, BM, BN, WGM, WGN, STAGES, KB) BN,
static const int k_shape_bm[] = {TILE_SHAPES(TILE_ROWS)};
static const int k_shape_bn[] = {TILE_SHAPES(TILE_COLUMNS)};
#undef TILE_ROWS
#undef TILE_COLUMNS
static constexpr int N_TILE_SHAPES = sizeof(k_shape_bm) / sizeof(k_shape_bm[0]);
extern "C" int celeg_gemm_tiles_shapes() { return N_TILE_SHAPES; }      // (how many there are to force)

// How the dies share the grid of tiles: every row of tiles of A is read by 8 / m dies, every column of
// tiles of W by m of them; the split with the fewest bytes read of those that leave no die more tiles than it
// has compute units, or of all if none does.
#define DIE_UNITS 32
struct Dies {
    int m, per_die;      // dies along the rows; the most tiles a die gets
};
static Dies dies_of(int tiles_m, int tiles_n, int M, int weight_rows) {
    Dies best{1, 0};
    double best_cost = -1.;
    for (int dm = 1; dm <= 8; dm *= 2) {
        const int dn = 8 / dm;
        if (dm > tiles_m || dn > tiles_n) continue;       // a die without a tile
        const int per_die = ((tiles_m + dm - 1) / dm) * ((tiles_n + dn - 1) / dn);
        const double cost = static_cast<double>(dn) * M + static_cast<double>(dm) * weight_rows;
        const bool over = per_die > DIE_UNITS, best_over = best.per_die > DIE_UNITS;
        if (best_cost < 0. || (over == best_over ? cost < best_cost : best_over)) {
            best_cost = cost;
            best = Dies{dm, per_die};
        }
    }
    if (best_cost < 0.) best.per_die = tiles_m * ((tiles_n + 7) / 8);
    return best;
}

// Whether K is cut over workgroups of which the last to arrive adds the sums (packed weights, residual): where the product's
// own tiles leave most compute units idle and K is long, so that each slice keeps 16 blocks of k, and no die gets more
// workgroups than it has compute units.  Measured with weights from memory, us (cut | whole, both packed):
//   rows                     65 to 70       130           200           300           450           600
//   1,024 x 4,608            11.1 | 17.8   12.1 | 17.8   14.0 | 17.9   16.5 | 17.9   17.3 | 18.2   21.4 | 21.8
//   2,048 x 8,192            18.1 | 28.6   24.6 | 28.8   24.7 | 28.9   29.0 | 36.5   (35.4 | 35.9)
// (2,048 x 2,048 and less: the same or slower; tiles that fill the compute units, cut: 2 to 20 % slower; a second round of
// workgroups on one die, 772 x 5,120 at 700 rows: 31.5 us against 26.3.)
// The number of slices, and with it the order of a sum, goes by the rows of the step: other tiles all give the same bits.
static TileShape tile_split(int M, int N, int K) {
    const auto fits = [&](int id, int slices) {
        return dies_of((M + k_shape_bm[id] - 1) / k_shape_bm[id], (N + k_shape_bn[id] - 1) / k_shape_bn[id], M, N).per_die * slices <= DIE_UNITS;
    };
    const auto shape = [&](int id, int slices) { return TileShape{id, k_shape_bm[id], k_shape_bn[id], slices}; };
    if (K < 4096) return shape(0, 1);
    if (fits(0, 4)) return shape(0, 4);
    if (fits(0, 3)) return shape(0, 3);
    if (fits(1, 4)) return shape(1, 4);
    if (fits(1, 2)) return shape(1, 2);
    if (fits(3, 3)) return shape(3, 3);
    return shape(0, 1);
}
// For tests and tuning: so many slices instead of the rule's (0: the rule; 1: none).
static int g_force_slices = 0;
extern "C" void celeg_gemm_tiles_force_slices(int slices) { g_force_slices = slices; }

static TileShape tile_shape(int M, int N, int K, int streams, bool may_split = false) {
    if (may_split && g_force_slices != 1 && g_force_shape < 0) {
        const TileShape cut = tile_split(M, N, K);
        if (cut.slices > 1) return cut;
    }
    int id = 0;
    if (g_force_shape >= 0 && g_force_shape < N_TILE_SHAPES) id = g_force_shape;
    else {
        // The smallest tile of which no die gets more than one for each of its compute units: the workgroups then
        // run side by side, each for as long as its own chain of blocks of k takes, and a smaller tile's
        // chain is shorter (less to pull from L2 and from LDS a block, room for more blocks in flight).  Measured
        // with weights from memory, us (chosen | the tiles of the rule before, which wanted few and large ones):
        //   rows   w2 (1,024 x 4,608)  out_proj (1,024 x 1,024)  in_proj (3,072 x 1,024)  w1 with w3 (9,216 x 1,024)
        //    100      17.7 | 25.6          7.1 |  9.2               6.9 |  8.7                11.1 | 12.3
        //    300      17.8 | 26.1          7.3 |  9.4               7.9 |  8.9                13.9 | 16.8
        //    600      21.1 | 26.3          8.5 |  9.6               9.8 |  9.8                19.1 | 21.2
        //  1,000      24.9 | 27.3          8.9 | 10.1              15.1 | 15.4                28.4 | 37.4
        //  2,048      37.4 | 37.4         12.3 | 12.3              19.3 | 19.3                41.4 | 41.4
        // Where two shapes fit, both at 300 to 4,096 rows of 20 products in turn:
        //   128x64 before 64x128 from 2,048 values of k on: 1 to 7 % faster in all of 56 (at 1,024 the same within 2 %)
        //   64x192 before 128x128: 0 to 11 % faster in all of 51
        //   64x128 on 4 wavefronts, two a compute unit, before 128x128 on 8, one: 2 to 6 % faster, up to 10 Mi weights;
        //   with more than the dies' L2s hold beside the rows (2,048 x 8,192, 4,096 x 4,096) 10 to 25 % slower
        //   128x128, two a compute unit, before 256x192: w1 with w3 at 800 rows 23.2 us against 27.5
        const auto fits = [&](int bm, int bn) {
            return dies_of((M + bm - 1) / bm, (N * streams + bn - 1) / bn, M, N * streams).per_die <= DIE_UNITS;
        };
        const long long weights = static_cast<long long>(N) * streams * K;
        if (fits(32, 64)) id = 0;
        else if (fits(64, 64)) id = 1;
        else if (K >= 2048 && fits(128, 64)) id = 2;
        else if (fits(64, 128)) id = 3;
        else if (fits(64, 192)) id = 4;
        else if (fits(128, 128)) id = weights <= (10 << 20) ? 5 : 6;
        else {
            // Beyond that the tile whose rounds cover the product in the least time.  A round (on the die with the most
            // tiles) takes, in us, SwiGLU at 1,024 | 2,048 values of k: 128x192 17.5 | 29.5, 128x128, two a compute unit,
            // 20.5 | 38.5, 256x192 26 | 45, 256x256 30.8 | 56, 256x288 34 | 60.  Of these five, at 512 to 4,096 rows of
            // 6,144 x 2,048, 9,216 x 1,024, 12,288 x 1,536 and 16,384 x 2,048, the sums choose the fastest or one within 3 %
            // in all of 36.  16,384 x 2,048: 2,048 rows 111.9 us in two rounds of 256x256 (128x128 150, 256x288 119.3), 1,200
            // rows 87.0 in two of 256x192 (100), 4,096 rows 228 (322, 245); 9,216 x 1,024 at 1,500 rows 31.5 in one of 256x256
            // (39.4 in two of 128x128).  The costs hold for the other epilogues too, though 256x256 into the stream has 40 registers
            // too few behind its loop (164 bytes of scratch a lane) and pays for it once a tile.  Into the stream, us,
            // 256x256 | 256x288 | 128x128 | 256x192: 1,024 columns, 1,024 values of k, 10,400 rows 58.8 | 61.8 | 64.0 | 66.4, 16,000 rows
            // 74.1 | 74.4 | 77.0 | 86.9; 4,608 values of k 136 | 142 | 161 | 194 and 158 | 162 | 180 | 223; 2,048 columns, 5,300 rows,
            // 2,048 values of k 84.8 | 85.3 | 91.5 | 109 and 8,192 211 | 218 | 243 | 318; 8,000 rows 99.8 | 99.5 | 108 | 126 and 244 | 252 |
            // 288 | 337.  Where another tile is faster (8,192 rows of 1,024: 52.4 | 53.1 | 39.0 | 40.9) the sums choose that.
            struct Cost { int id, on_a_unit; long long fixed, per_k; };      // tenths of us a round and 1,024 values of k
            static constexpr Cost costs[] = {{7, 1, 55, 120}, {8, 2, 25, 180}, {9, 1, 70, 190}, {11, 1, 85, 230}, {10, 1, 110, 240}};
            long long best = -1;
            for (const Cost& c : costs) {
                const int bm = k_shape_bm[c.id], bn = k_shape_bn[c.id];
                const int per_die = dies_of((M + bm - 1) / bm, (N * streams + bn - 1) / bn, M, N * streams).per_die;
                const long long rounds = (per_die + DIE_UNITS * c.on_a_unit - 1) / (DIE_UNITS * c.on_a_unit);
                const long long cost = rounds * (1024 * c.fixed + c.per_k * K);
                if (best < 0 || cost < best) {
                    best = cost;
                    id = c.id;
                }
            }
        }
    }
    return TileShape{id, k_shape_bm[id], k_shape_bn[id], 1};
}

#define TILE_SPLITS(ID) ((ID) == 0 || (ID) == 1 || (ID) == 3)      // the shapes that tile_split names
#define TILE_SPLIT_MOST_BYTES (256 * 64 * 128 * 4)                 // of sums: 256 workgroups of the largest of them

template <int BM, int BN, int WGM, int WGN, int STAGES, int KB, int EPI, bool PACKED, bool SPLIT>
static int launch_tiles(const TileParams& p, hipStream_t stream) {
    constexpr int NS = TileStreams<EPI>::n;
    constexpr size_t stages_lds = static_cast<size_t>(STAGES) * (BM + BN) * (KB == 32 ? 64 : 128);
    // (the wide kernel's SwiGLU lays the tile's gate and up values out in LDS)
    constexpr size_t swiglu_lds = KB != 0 && EPI == T_SWIGLU ? static_cast<size_t>(2) * BM * (BN + 16) : 0;
    constexpr size_t lds = stages_lds > swiglu_lds ? stages_lds : swiglu_lds;
    void (*kernel)(const TileParams, const int, const int, const int);
    if constexpr (KB != 0) kernel = &gemm_tiles_wide_kernel<BM, BN, WGM, WGN, STAGES, KB, EPI>;
    else kernel = &gemm_tiles_kernel<BM, BN, WGM, WGN, STAGES, EPI, PACKED, SPLIT>;
    static_assert(lds <= 160 * 1024, "more LDS than a compute unit has");
    static bool raised = false;              // once per instantiation: more LDS than the default limit
    if (lds > 48 * 1024 && !raised) {
        hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        if (err != hipSuccess) return static_cast<int>(err);
        raised = true;
    }
    const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N * NS + BN - 1) / BN;
    int dies_m = dies_of(tiles_m, tiles_n, p.M, p.N * NS).m;
    if (g_force_dies_m > 0) dies_m = g_force_dies_m;
    const int dies_n = 8 / dies_m;
    const int per_die = ((tiles_m + dies_m - 1) / dies_m) * ((tiles_n + dies_n - 1) / dies_n);
    dim3 grid(per_die * 8 * (SPLIT ? p.k_slices : 1)), block(WGM * WGN * 64);
    hipLaunchKernelGGL(kernel, grid, block, lds, stream, p, tiles_m, tiles_n, dies_m);
    return CELEG_LAUNCH_RESULT();
}

// (for tests: which of the shapes a product of weights as they are takes)
extern "C" int celeg_gemm_tiles_chosen(int M, int N, int K, int epi) { return tile_shape(M, N, K, epi == T_SWIGLU ? 2 : 1).id; }

template <int EPI>
static int launch_epilogue(const TileParams& p, hipStream_t stream) {
    const TileShape s = tile_shape(p.M, p.N, p.K, TileStreams<EPI>::n);
#define TILE_CASE(ID, BM, BN, WGM, WGN, STAGES, KB) \
    if (s.id == ID) return launch_tiles<BM, BN, WGM, WGN, STAGES, KB, EPI, false, false>(p, stream);
    TILE_SHAPES(TILE_CASE)
#undef TILE_CASE
    return static_cast<int>(hipErrorInvalidValue);
}

// The residual epilogue with packed weights, K cut where there is room for the sums.
template <int EPI>
static int launch_packed(const TileParams& params, hipStream_t stream) {
    TileParams p = params;
    TileShape s = tile_shape(p.M, p.N, p.K, 1, p.parts && p.arrived);
    if (g_force_slices > 1 && p.parts && p.arrived && TILE_SPLITS(s.id) && g_force_slices <= p.K / 64) s.slices = g_force_slices;
    p.k_slices = s.slices;
    const long long tiles = static_cast<long long>((p.M + s.bm - 1) / s.bm) * ((p.N + s.bn - 1) / s.bn);
    if (s.slices > 1 && (tiles > 256 || tiles * s.slices * s.bm * s.bn * 4 > TILE_SPLIT_MOST_BYTES)) return static_cast<int>(hipErrorInvalidValue);
#define TILE_CASE(ID, BM, BN, WGM, WGN, STAGES, KB)                                                                     \
    if constexpr (KB == 0) {                                                                                            \
        if constexpr (TILE_SPLITS(ID)) {                                                                                \
            if (s.id == ID && s.slices > 1) return launch_tiles<BM, BN, WGM, WGN, STAGES, KB, EPI, true, true>(p, stream); \
        }                                                                                                               \
        if (s.id == ID) return launch_tiles<BM, BN, WGM, WGN, STAGES, KB, EPI, true, false>(p, stream);          \
    }
    TILE_SHAPES(TILE_CASE)
#undef TILE_CASE
    return static_cast<int>(hipErrorInvalidValue);      // (the wide tiles read weights as they are)
}

// Whether the residual epilogue is better given packed weights for these sizes, and room for a cut K's sums (bytes, and zeros
// ahead of them that the launch leaves as zeros, 256 numbers).  Us, packed | as they are, with weights from memory:
//   1,024 x 4,608    1,000 rows 22.6 | 23.8, 1,300 31.1 | 29.7, 1,500 31.5 | 32.8, 1,700 31.6 | 30.2, 2,048 33.0 | 35.4, 4,096 58.6 | 63.5
//   1,024 x 1,024    600 8.4 | 8.4, 1,500 11.6 | 12.0, 2,048 12.2 | 12.5, 8,192 33.9 | 34.6
//   2,048 x 2,048    512 13.4 | 13.9, 700 18.0 | 17.7, 1,024 19.7 | 20.0, 1,500 29.6 | 30.9, 2,048 33.2 | 34.1, 4,096 47.8 | 50.3
//   2,048 x 8,192    512 38.4 | 39.5, 600 49.8 | 48.7, 1,024 53.2 | 52.3, 1,500 71.3 | 75.1, 2,048 77.3 | 82.2
// (128x64, the tile of 1,024 x 4,608 from 1,025 rows on and of 2,048 x 8,192 at 513 to 1,024: only where it is on nearly all
// compute units and K below 8,192; 64x192 and 128x192, which none of these takes, and the wide tiles: not.)
extern "C" int celeg_gemm_tiles_packed(int M, int N, int K) {
    if (tile_split(M, N, K).slices > 1) return 1;
    const TileShape s = tile_shape(M, N, K, 1);
    if (s.id == 2) return K < 8192 && static_cast<long long>((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn) >= 240;
    return s.id == 0 || s.id == 1 || s.id == 3 || s.id == 5 || s.id == 6 || s.id == 8;
}
extern "C" size_t celeg_gemm_tiles_split_bytes() { return TILE_SPLIT_MOST_BYTES; }

// Number of partial sums of squares a row gets from the "residual" epilogue for these
// sizes (one per tile column): the caller sizes stats_out [>= M, >= blocks].  packed: with packed weights and room
// for a cut K's sums.
extern "C" int celeg_gemm_tiles_blocks(int M, int N, int K, int packed) {
    const TileShape s = tile_shape(M, N, K, 1, packed != 0);
    return (N + s.bn - 1) / s.bn;
}

extern "C" int celeg_gemm_tiles_params_size() { return static_cast<int>(sizeof(TileParams)); }

// K % 64 == 0, N % 4 == 0, lda, ldw % 8 == 0, outputs with rows aligned to their vector
// stores (ldo % 4 == 0).  Any M >= 1.
extern "C" int celeg_gemm_tiles(const TileParams* params, int epi, hipStream_t stream) {
    const TileParams& p = *params;
    if (p.M <= 0 || p.N <= 0) return 0;
    if (p.K <= 0 || (p.K % 64) || (p.N % 4) || (p.lda % 8) || (p.ldw % 8) || (p.ldo % 4) ||
        p.lda < p.K || (p.w_block ? p.ldw != 32 || p.w_block % 8 || p.w_block < 32LL * p.N || epi != T_RESIDUAL : p.ldw < p.K) || p.ldo < p.N)
        return static_cast<int>(hipErrorInvalidValue);
    if (p.stats && p.n_stat_blocks < 1) return static_cast<int>(hipErrorInvalidValue);
    if (reinterpret_cast<uintptr_t>(p.bias) & 15) return static_cast<int>(hipErrorInvalidValue);
    if (p.out_bf16 && ((p.ld_bf16 % 4) || p.ld_bf16 < p.N)) return static_cast<int>(hipErrorInvalidValue);
    if (epi == T_SWIGLU && p.stream_rows < p.N) return static_cast<int>(hipErrorInvalidValue);
    switch (epi) {
        case T_STORE: return launch_epilogue<T_STORE>(p, stream);
        case T_RESIDUAL: return p.w_block ? launch_packed<T_RESIDUAL>(p, stream) : launch_epilogue<T_RESIDUAL>(p, stream);
        case T_SWIGLU: return launch_epilogue<T_SWIGLU>(p, stream);
        case T_QKV: {
            const auto misaligned = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) != 0; };
            const long long heads = static_cast<long long>(p.q_heads) + 2LL * p.kv_heads;
            if (p.q_heads <= 0 || p.kv_heads <= 0 || p.N != heads * QKV_HD || p.ldo % 8 || misaligned(p.out) ||
                !p.positions || !p.token_slot || !p.table || p.table_stride <= 0 || !p.k_pool || !p.v_pool ||
                misaligned(p.k_pool) || misaligned(p.v_pool) || p.page_tokens < 4 || (p.page_tokens & (p.page_tokens - 1)) ||
                p.n_layers <= 0 || p.layer < 0 || p.layer >= p.n_layers || misaligned(p.q_weight) || misaligned(p.k_weight) ||
                misaligned(p.cos_sin))
                return static_cast<int>(hipErrorInvalidValue);
            // (a wavefront holds 16 or 32 rows of one head of 64 columns; the smallest tile of which no die gets
            // more than one for each of its compute units, as above.  In a model, 2,048 columns by
            // 1,024: 301 rows 12.4 us, 600 rows 14.4, 2,048 rows 21.3; with the last of these for all 22.4, 22.6 and 23.0)
            const auto fits = [&](int bm, int bn) { return dies_of((p.M + bm - 1) / bm, (p.N + bn - 1) / bn, p.M, p.N).per_die <= DIE_UNITS; };
            if (fits(64, 64)) return launch_tiles<64, 64, 4, 1, 4, 0, T_QKV, false, false>(p, stream);
            if (fits(64, 128)) return launch_tiles<64, 128, 4, 2, 4, 0, T_QKV, false, false>(p, stream);
            if (fits(128, 128)) return launch_tiles<128, 128, 4, 2, 4, 0, T_QKV, false, false>(p, stream);
            return launch_tiles<128, 128, 4, 2, 2, 0, T_QKV, false, false>(p, stream);
        }
        default: return static_cast<int>(hipErrorInvalidValue);
    }
}
