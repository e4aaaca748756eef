// The gated delta rule over long portions of prompts, 64 tokens at a time, on the 64-bit matrix instructions.
//
// The recurrence (delta_rule.hip) is a chain from token to token: 0.15 us each, whatever the chip has idle beside it.  Over
// a chunk of C = 64 tokens with the state S before it, with
// A_i = a_1 .. a_i and R_ij = a_(j+1) .. a_i (products of decays, never quotients):
//     (I + L) U = b (V - A K S),   L_ij = b_i R_ij k_i.k_j  (j < i)
//     O_i = A_i q_i S + sum_(j <= i) R_ij q_i.k_j u_j,      S <- A_C S + sum_j R_Cj k_j u_j^T
// so what hangs on S is three products a chunk.  Three kernels:
//  * delta_chunk_prepare, a workgroup a (chunk, head), all at once: L, then W and U' with (I + L) W = b A K and
//    (I + L) U' = b V by blocks of 16 rows, P_ij = R_ij q_i.k_j, A_i and R_Cj;
//  * delta_chunk_scan, a workgroup per (request, head, 16 columns of S), the chain: U = U' - W S, then the state;
//    four wavefronts share a chunk's rows and meet twice, the next two chunks' operands on their way meanwhile;
//  * delta_chunk_out, a workgroup a (chunk, head, 16 columns), all at once: O = A q S + P U.
//
// U' - W S and A q S + P U are differences of large numbers where keys are alike, so in 32-bit this form is 1.2 to 3.5 times
// as far from the exact result as the chain of tokens.  All sums are therefore 64-bit, and so is what is kept between the
// kernels of U and P; W and the states before the chunks are rounded to 32-bit.  A result is then the exact one
// rounded once, nearly.  Against 64 bits, of the result (token by token in 32-bit | these sums in 32-bit | as they are): ordinary keys
// 0.8e-7 | 1.3e-7 | 0.25e-7, alike and no decay 2.0e-7 | 3.4e-7 | 0.43e-7, of four dimensions 0.9e-7 | 3.1e-7 | 0.29e-7.
// 16 heads of 64 x 64: 1,500 tokens 269 us token by token, 117 as these three (37 + 60 + 19; all 32-bit they were 72), three
// requests of 2,048 in all 207 and 126.  (Operands two chunks ahead and four chains of sums in the scan: 127 -> 117.)
//
// Keys of 64 only: at 128 a chunk's keys, triangle and right sides do not fit LDS.
//
// v_mfma_f64_16x16x4_f64: lane l gives row l % 16 of the first operand and column l % 16 of the second at value l / 16 of k,
// and holds rows l / 16 + 4 e of column l % 16 of the sums.  The first operand's rows are dealt to the lanes so that these
// are rows 4 (l / 16) + e of the tile (dc_row), which lie side by side.  Both operands take k in the order in which a lane's
// four neighbours bring it: value e of quarter l / 16 of a piece of 16 is k = 4 (l / 16) + e in step e.
#include "common.h"

namespace {

typedef float dc_f4 __attribute__((ext_vector_type(4)));
typedef double dc_d2 __attribute__((ext_vector_type(2)));
typedef double dc_d4 __attribute__((ext_vector_type(4)));
#define DC_ROWS 64                 // tokens of a chunk, and numbers of a key
#define DC_PITCH 68                // 32-bit numbers between rows in LDS
#define DC_PITCH64 66              // 64-bit ones
#define DC_PREPARE_THREADS 512

// A (chunk, head) in the workspace, offsets in floats.  32-bit: W [token][d], K [d][token], the state before the chunk
// [column][d]; 64-bit: P [token][token], A [token], R_C [token], U [column][token].
constexpr size_t DC_W = 0, DC_KT = 4096, DC_P = 8192, DC_A = DC_P + 2 * 4096, DC_RC = DC_A + 2 * 64, DC_U = DC_RC + 2 * 64;
__host__ __device__ constexpr size_t dc_state(int V) { return DC_U + static_cast<size_t>(2) * DC_ROWS * V; }
__host__ __device__ constexpr size_t dc_floats(int V) { return dc_state(V) + static_cast<size_t>(DC_ROWS) * V; }

__device__ __forceinline__ int dc_row(int r16) { return 4 * (r16 & 3) + (r16 >> 2); }
__device__ __forceinline__ dc_d4 dc_wide(const dc_f4 x) { return dc_d4{x[0], x[1], x[2], x[3]}; }
// four numbers of LDS or memory, in 64-bit (rows of 64-bit numbers start at multiples of 16 bytes)
__device__ __forceinline__ dc_d4 dc_load(const float* p) { return dc_wide(*reinterpret_cast<const dc_f4*>(p)); }
__device__ __forceinline__ dc_d4 dc_load(const double* p) {
    const dc_d2 lo = reinterpret_cast<const dc_d2*>(p)[0], hi = reinterpret_cast<const dc_d2*>(p)[1];
    return dc_d4{lo[0], lo[1], hi[0], hi[1]};
}
__device__ __forceinline__ void dc_store(double* p, const dc_d4 x) {
    reinterpret_cast<dc_d2*>(p)[0] = dc_d2{x[0], x[1]};
    reinterpret_cast<dc_d2*>(p)[1] = dc_d2{x[2], x[3]};
}
// sum += a piece of 16 values of k of both operands
__device__ __forceinline__ dc_d4 dc_piece(const dc_d4 a, const dc_d4 b, dc_d4 sum) {
#pragma unroll
    for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_mfma_f64_16x16x4f64(a[e], b[e], sum, 0, 0, 0);
    return sum;
}

// sum += four pieces, in four chains of sums (one chain of 16 instructions that wait for each other: 0.1 us a chunk more)
__device__ __forceinline__ dc_d4 dc_pieces(const dc_f4 (&a)[4], const double* b, const dc_d4 sum) {
    dc_d4 part[4] = {sum, {0., 0., 0., 0.}, {0., 0., 0., 0.}, {0., 0., 0., 0.}}, left[4], right[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        left[p] = dc_wide(a[p]);
        right[p] = dc_load(b + 16 * p);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int p = 0; p < 4; ++p) part[p] = __builtin_amdgcn_mfma_f64_16x16x4f64(left[p][e], right[p][e], part[p], 0, 0, 0);
    return (part[0] + part[1]) + (part[2] + part[3]);
}

// chunk number `chunk` of the step: its request, that one's first row, and the chunk's first row and rows; requests of
// fewer than `least` rows have none
__device__ __forceinline__ bool dc_find(const int* __restrict__ cu_seqlens, int n_seqs, int least, int chunk, int& row0, int& rows) {
    for (int s = 0; s < n_seqs; ++s) {
        const int first = cu_seqlens[s], n = cu_seqlens[s + 1] - first;
        if (n < least) continue;
        const int chunks = (n + DC_ROWS - 1) / DC_ROWS;
        if (chunk < chunks) {
            row0 = first + chunk * DC_ROWS;
            rows = min(DC_ROWS, n - chunk * DC_ROWS);
            return true;
        }
        chunk -= chunks;
    }
    return false;
}

__global__ __launch_bounds__(DC_PREPARE_THREADS) void delta_chunk_prepare_kernel(
    const float* __restrict__ qk, const float* __restrict__ v, const float* __restrict__ beta_decay, const int* __restrict__ cu_seqlens,
    float* __restrict__ ws, const int n_seqs, const int least, const int G, const int H, const int V) {
    constexpr int D = DC_ROWS, C = DC_ROWS, P = DC_PITCH, PD = DC_PITCH64, THREADS = DC_PREPARE_THREADS, WAVES = THREADS / CELEG_WAVE;
    extern __shared__ __attribute__((aligned(16))) float dc_lds[];
    float* const ks = dc_lds;                                        // K [token][d]
    double* const ls = reinterpret_cast<double*>(ks + C * P);        // L [token][token]
    double* const xs = ls + C * PD;                                  // W and U', [column][token]
    __shared__ double a_s[C], b_s[C], tile_before[C], tile_behind[C], all_before[C];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / CELEG_WAVE), lane = tid % CELEG_WAVE;
    const int r16 = lane & 15, q = lane >> 4;
    const int h = blockIdx.y, g = h / (H / G);
    int row0, rows;
    if (!dc_find(cu_seqlens, n_seqs, least, blockIdx.x, row0, rows)) return;
    const size_t ldqk = static_cast<size_t>(2) * G * D;
    const float* const q_rows = qk + row0 * ldqk + static_cast<size_t>(g) * D;
    const float* const k_rows = q_rows + static_cast<size_t>(G) * D;
    float* const mine = ws + (static_cast<size_t>(blockIdx.x) * H + h) * dc_floats(V);
    double* const p_out = reinterpret_cast<double*>(mine + DC_P);
    // the tiles on and under the diagonal, 10 of q.k and then 10 of k.k, dealt to the wavefronts in turn; the queries' rows of
    // the first ones are asked for now
    const auto tile_row = [](int tile) { return tile < 1 ? 0 : tile < 3 ? 1 : tile < 6 ? 2 : 3; };
    dc_f4 q4[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int p = 0; p < 4; ++p)
            q4[i][p] = *reinterpret_cast<const dc_f4*>(q_rows + min(16 * tile_row(min(wave + WAVES * i, 9)) + dc_row(r16), rows - 1) * ldqk + 16 * p + 4 * q);
    // tokens behind the portion's last: no key, nothing written, no decay
    if (tid < C) {
        const float* const bd = beta_decay + static_cast<size_t>(row0 + min(tid, rows - 1)) * 2 * H + h;
        b_s[tid] = tid < rows ? bd[0] : 0.f;
        a_s[tid] = tid < rows ? bd[H] : 1.f;
    }
#pragma unroll
    for (int i = 0; i < C * D / 4 / THREADS; ++i) {
        const int at = tid + THREADS * i, row = at >> 4, d = 4 * (at & 15);
        dc_f4 x = *reinterpret_cast<const dc_f4*>(k_rows + min(row, rows - 1) * ldqk + d);
        if (row >= rows) x = dc_f4{0.f, 0.f, 0.f, 0.f};
        *reinterpret_cast<dc_f4*>(ks + row * P + d) = x;
    }
    __syncthreads();
    // products of decays: over the token's tile of 16 up to it and from behind it on, and over the chunk
    if (wave == 0) {
        double before = a_s[lane], behind = r16 == 15 ? 1. : a_s[lane + 1 < C ? lane + 1 : lane];
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) {
            const double b = __shfl_up(before, off, 16), e = __shfl_down(behind, off, 16);
            if (r16 >= off) before *= b;
            if (r16 + off < 16) behind *= e;
        }
        tile_before[lane] = before;
        tile_behind[lane] = behind;
        double all = before, rest = behind;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const double whole = __shfl(before, 16 * t + 15, CELEG_WAVE);
            if (t < q) all *= whole;
            if (t > q) rest *= whole;
        }
        all_before[lane] = all;
        reinterpret_cast<double*>(mine + DC_A)[lane] = all;
        reinterpret_cast<double*>(mine + DC_RC)[lane] = rest;
    }
    __syncthreads();
    // the right sides b A K and b V, and the keys turned over
    for (int at = tid; at < C * D / 4; at += THREADS) {
        const int row = at & 63, d = 4 * (at >> 6);
        const double f = b_s[row] * all_before[row];
        const dc_f4 x = *reinterpret_cast<const dc_f4*>(ks + row * P + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            xs[(d + e) * PD + row] = f * x[e];
            mine[DC_KT + static_cast<size_t>(d + e) * C + row] = x[e];
        }
    }
    for (int at = tid; at < C * V / 4; at += THREADS) {
        const int row = at / (V / 4), j = 4 * (at - row * (V / 4));
        const dc_f4 x = *reinterpret_cast<const dc_f4*>(v + static_cast<size_t>(row0 + min(row, rows - 1)) * H * V + static_cast<size_t>(h) * V + j);
#pragma unroll
        for (int e = 0; e < 4; ++e) xs[(D + j + e) * PD + row] = b_s[row] * x[e];
    }
    // the tiles of q.k (P) and of k.k (L)
    const auto decays = [&](int ti, int tj) {
        dc_d4 decay;
        if (ti == tj) {
            double r = 1.;
#pragma unroll
            for (int m = 1; m < 16; ++m) r *= m > r16 && m <= 4 * q ? a_s[16 * ti + m] : 1.;
            decay[0] = r;
#pragma unroll
            for (int e = 1; e < 4; ++e) decay[e] = 4 * q + e > r16 ? decay[e - 1] * a_s[16 * ti + 4 * q + e] : 1.;
        } else {
            double r = tile_behind[16 * tj + r16];
            for (int t = tj + 1; t < ti; ++t) r *= tile_before[16 * t + 15];
#pragma unroll
            for (int e = 0; e < 4; ++e) decay[e] = tile_before[16 * ti + 4 * q + e] * r;
        }
        return decay;
    };
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int job = wave + WAVES * i;
        if (job >= 20) break;
        const bool of_q = job < 10;
        const int tile = of_q ? job : job - 10, ti = tile_row(tile), tj = tile - ti * (ti + 1) / 2;
        dc_d4 sum = {0., 0., 0., 0.};
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            dc_f4 left = *reinterpret_cast<const dc_f4*>(ks + (16 * ti + dc_row(r16)) * P + 16 * p + 4 * q);
            if (i < 2 && of_q) left = q4[i < 2 ? i : 0][p];
            sum = dc_piece(dc_wide(left), dc_load(ks + (16 * tj + r16) * P + 16 * p + 4 * q), sum);
        }
        const dc_d4 decay = decays(ti, tj);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = 16 * ti + 4 * q + e, j = 16 * tj + r16;
            if (of_q) p_out[row * C + j] = row >= j ? decay[e] * sum[e] : 0.;
            else ls[row * PD + j] = row > j ? b_s[row] * (decay[e] * sum[e]) : 0.;
        }
    }
    __syncthreads();
    // (I + L) X = right sides, 16 rows at a time: a thread a column inside the block, the rows behind it on the matrix cores
    const int columns = D + V;
    for (int t = 0; t < 4; ++t) {
        if (tid < columns) {
            double x[16];
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const dc_d4 x4 = dc_load(xs + tid * PD + 16 * t + 4 * p);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[4 * p + e] = x4[e];
            }
#pragma unroll
            for (int i = 1; i < 16; ++i)
#pragma unroll
                for (int p = 0; 4 * p < i; ++p) {
                    const dc_d4 l4 = dc_load(ls + (16 * t + i) * PD + 16 * t + 4 * p);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (4 * p + e < i) x[i] = fma(-l4[e], x[4 * p + e], x[i]);
                }
#pragma unroll
            for (int p = 0; p < 4; ++p) dc_store(xs + tid * PD + 16 * t + 4 * p, dc_d4{x[4 * p], x[4 * p + 1], x[4 * p + 2], x[4 * p + 3]});
        }
        __syncthreads();
        const int n_tiles = columns / 16;
        for (int job = wave; job < (3 - t) * n_tiles; job += WAVES) {
            const int below = t + 1 + job / n_tiles, col = 16 * (job % n_tiles) + r16;
            double* const to = xs + col * PD + 16 * below + 4 * q;
            dc_store(to, dc_piece(-dc_load(ls + (16 * below + dc_row(r16)) * PD + 16 * t + 4 * q), dc_load(xs + col * PD + 16 * t + 4 * q), dc_load(to)));
        }
        __syncthreads();
    }
    for (int at = tid; at < C * D / 4; at += THREADS) {
        const int row = at >> 4, d = 4 * (at & 15);
        dc_f4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = static_cast<float>(xs[(d + e) * PD + row]);
        *reinterpret_cast<dc_f4*>(mine + DC_W + row * D + d) = w;
    }
    double* const u_out = reinterpret_cast<double*>(mine + DC_U);
    for (int at = tid; at < V * C / 2; at += THREADS) {
        const int col = at >> 5, row = 2 * (at & 31);
        *reinterpret_cast<dc_d2*>(u_out + static_cast<size_t>(col) * C + row) = *reinterpret_cast<const dc_d2*>(xs + (D + col) * PD + row);
    }
}

__global__ __launch_bounds__(256) void delta_chunk_scan_kernel(float* __restrict__ state, const size_t state_stride,
                                                               const int* __restrict__ cu_seqlens, const int* __restrict__ seq_slot,
                                                               float* __restrict__ ws, const int least, const int H, const int V) {
    constexpr int D = DC_ROWS, C = DC_ROWS, PD = DC_PITCH64;
    __shared__ __attribute__((aligned(16))) double s_s[16 * PD], u_s[16 * PD];       // [column][d] and [column][token]
    const int s = blockIdx.x, h = blockIdx.y, n0 = blockIdx.z * 16;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / CELEG_WAVE), lane = threadIdx.x % CELEG_WAVE, r16 = lane & 15, q = lane >> 4;
    const int n = cu_seqlens[s + 1] - cu_seqlens[s];
    if (n < least) return;
    int chunk = 0;
    for (int other = 0; other < s; ++other) {
        const int rows = cu_seqlens[other + 1] - cu_seqlens[other];
        if (rows >= least) chunk += (rows + C - 1) / C;
    }
    const int chunks = (n + C - 1) / C;
    const size_t stride = static_cast<size_t>(H) * dc_floats(V);
    float* at = ws + (static_cast<size_t>(chunk) * H + h) * dc_floats(V);
    float* const mine = state + static_cast<size_t>(seq_slot[s]) * state_stride + static_cast<size_t>(h) * D * V + n0 + r16;
    const size_t tile = static_cast<size_t>(16 * wave + dc_row(r16)) * 64 + 4 * q, column = static_cast<size_t>(n0 + r16) * 64 + 16 * wave + 4 * q;
    const int lds_own = r16 * PD + 16 * wave + 4 * q, lds_all = r16 * PD + 4 * q;
    dc_d4 state4;
#pragma unroll
    for (int e = 0; e < 4; ++e) state4[e] = mine[static_cast<size_t>(16 * wave + 4 * q + e) * V];
    struct Operands {
        dc_f4 w[4], k[4];
        dc_d4 u, rest;
        double decay;
    } ahead[2];
    auto fetch = [&](const float* from, Operands& to) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            to.w[p] = *reinterpret_cast<const dc_f4*>(from + DC_W + tile + 16 * p);
            to.k[p] = *reinterpret_cast<const dc_f4*>(from + DC_KT + tile + 16 * p);
        }
        to.u = dc_load(reinterpret_cast<const double*>(from + DC_U) + column);
        to.rest = dc_load(reinterpret_cast<const double*>(from + DC_RC) + 16 * wave + 4 * q);
        to.decay = reinterpret_cast<const double*>(from + DC_A)[C - 1];
    };
    // (everybody's writes to LDS are there, while loads from memory stay on their way)
    auto meet = [] {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // (operands come from memory two chunks ahead)
    fetch(at, ahead[0]);
    if (chunks > 1) fetch(at + stride, ahead[1]);
    for (int c0 = 0; c0 < chunks; c0 += 2) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            if (c0 + half >= chunks) break;
            const Operands now = ahead[half];
            if (c0 + half + 2 < chunks) fetch(at + 2 * stride, ahead[half]);
            dc_store(s_s + lds_own, state4);
            // (the state before the chunk, for delta_chunk_out)
            *reinterpret_cast<dc_f4*>(at + dc_state(V) + column) =
                dc_f4{static_cast<float>(state4[0]), static_cast<float>(state4[1]), static_cast<float>(state4[2]), static_cast<float>(state4[3])};
            meet();
            const dc_d4 u = -dc_pieces(now.w, s_s + lds_all, -now.u);
            dc_store(u_s + lds_own, now.rest * u);
            dc_store(reinterpret_cast<double*>(at + DC_U) + column, u);
            meet();
            state4 = dc_pieces(now.k, u_s + lds_all, state4 * now.decay);
            at += stride;
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) mine[static_cast<size_t>(16 * wave + 4 * q + e) * V] = static_cast<float>(state4[e]);
}

__global__ __launch_bounds__(256) void delta_chunk_out_kernel(const float* __restrict__ qk, const int* __restrict__ cu_seqlens,
                                                              const float* __restrict__ ws, float* __restrict__ out, const int n_seqs,
                                                              const int least, const int G, const int H, const int V) {
    constexpr int D = DC_ROWS, C = DC_ROWS;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / CELEG_WAVE), lane = threadIdx.x % CELEG_WAVE, r16 = lane & 15, q = lane >> 4;
    const int h = blockIdx.y, g = h / (H / G);
    int row0, rows;
    if (!dc_find(cu_seqlens, n_seqs, least, blockIdx.x, row0, rows) || 16 * wave >= rows) return;
    const float* const mine = ws + (static_cast<size_t>(blockIdx.x) * H + h) * dc_floats(V);
    const int row16 = 16 * wave + dc_row(r16), n0 = 16 * blockIdx.z;
    const float* const q_row = qk + static_cast<size_t>(row0 + min(row16, rows - 1)) * 2 * G * D + static_cast<size_t>(g) * D + 4 * q;
    const double* const p_row = reinterpret_cast<const double*>(mine + DC_P) + static_cast<size_t>(row16) * C + 4 * q;
    const double* const u = reinterpret_cast<const double*>(mine + DC_U) + static_cast<size_t>(n0 + r16) * C + 4 * q;
    const float* const s = mine + dc_state(V) + static_cast<size_t>(n0 + r16) * C + 4 * q;
    dc_f4 q4[4], s4[4];
    dc_d4 p4[4], u4[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        q4[p] = *reinterpret_cast<const dc_f4*>(q_row + 16 * p);
        s4[p] = *reinterpret_cast<const dc_f4*>(s + 16 * p);
        p4[p] = dc_load(p_row + 16 * min(p, wave));
        u4[p] = dc_load(u + 16 * min(p, wave));
    }
    const dc_d4 before = dc_load(reinterpret_cast<const double*>(mine + DC_A) + 16 * wave + 4 * q);
    dc_d4 sum = {0., 0., 0., 0.};
#pragma unroll
    for (int p = 0; p < 4; ++p) sum = dc_piece(dc_wide(q4[p]), dc_wide(s4[p]), sum);
    sum *= before;
#pragma unroll
    for (int p = 0; p < 3; ++p)
        if (p < wave) sum = dc_piece(p4[p], u4[p], sum);
    // (the tile on the diagonal, whose operands are the last piece's whatever the wavefront; the zeros above the diagonal
    // must not meet a later token's infinities or NaN)
    bool odd = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) odd = odd || !(fabs(u4[3][e]) < static_cast<double>(INFINITY));
    if (__ballot(odd) == 0ull) {
        sum = dc_piece(p4[3], u4[3], sum);
    } else {
        const double* const p_tile = reinterpret_cast<const double*>(mine + DC_P) + static_cast<size_t>(16 * wave) * C + 16 * wave;
        const double* const u_tile = u - 4 * q + 16 * wave;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            for (int j = 0; j <= 4 * q + e; ++j) sum[e] = fma(p_tile[(4 * q + e) * C + j], u_tile[j], sum[e]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int row = 16 * wave + 4 * q + e;
        if (row < rows) out[static_cast<size_t>(row0 + row) * H * V + static_cast<size_t>(h) * V + n0 + r16] = static_cast<float>(sum[e]);
    }
}

}  // namespace

// Sizes that the chunked form takes.
extern "C" int celeg_delta_chunks_ok(int G, int H, int D, int V) {
    return D == DC_ROWS && V >= 16 && V <= 128 && V % 16 == 0 && G > 0 && H % G == 0;
}
// floats of workspace for `chunks` chunks
extern "C" long long celeg_delta_chunks_floats(int chunks, int H, int V) { return static_cast<long long>(chunks) * H * dc_floats(V); }

// The requests of the step with `least` rows or more (the others are not touched); max_chunks: at least the sum over
// them of ceil(rows / 64).
extern "C" int celeg_delta_chunks(const float* qk, const float* v, const float* beta_decay, float* state, size_t state_stride,
                                  const int* cu_seqlens, const int* seq_slot, float* out, float* ws, int n_seqs, int max_chunks, int least,
                                  int G, int H, int D, int V, hipStream_t stream) {
    if (n_seqs <= 0 || max_chunks <= 0) return 0;
    if (!celeg_delta_chunks_ok(G, H, D, V) || least < 1) return static_cast<int>(hipErrorInvalidValue);
    // (V = 64: 119 KB, 128: 153 KB; asked for with every call, since the limit is the current device's)
    const size_t lds = DC_ROWS * DC_PITCH * sizeof(float) + static_cast<size_t>(2 * DC_ROWS + V) * DC_PITCH64 * sizeof(double);
    const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(&delta_chunk_prepare_kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (err != hipSuccess) return static_cast<int>(err);
    hipLaunchKernelGGL(delta_chunk_prepare_kernel, dim3(max_chunks, H), dim3(DC_PREPARE_THREADS), lds, stream, qk, v, beta_decay, cu_seqlens, ws,
                       n_seqs, least, G, H, V);
    hipLaunchKernelGGL(delta_chunk_scan_kernel, dim3(n_seqs, H, V / 16), dim3(256), 0, stream, state, state_stride, cu_seqlens, seq_slot, ws,
                       least, H, V);
    hipLaunchKernelGGL(delta_chunk_out_kernel, dim3(max_chunks, H, V / 16), dim3(256), 0, stream, qk, cu_seqlens, ws, out, n_seqs, least, G, H, V);
    return CELEG_LAUNCH_RESULT();
}
