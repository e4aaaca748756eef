// The gated delta rule over long portions of prompts, 64 tokens at a time, on the matrix cores in 32-bit.
//
// The recurrence (delta_rule.hip) is a chain from token to token: 0.15 us each, whatever the chip has idle beside it (a
// portion of 1,500 tokens: 223 us).  Over a chunk of C = 64 tokens with the state S before it, with
// A_i = a_1 .. a_i and R_ij = a_(j+1) .. a_i (products of decays, never quotients):
//     (I + L) U = b (V - A K S),   L_ij = b_i R_ij k_i.k_j  (j < i)
//     O_i = A_i q_i S + sum_(j <= i) R_ij q_i.k_j u_j,      S <- A_C S + sum_j R_Cj k_j u_j^T
// so what hangs on S is three products a chunk.  Three kernels:
//  * delta_chunk_prepare, a workgroup a (chunk, head), all at once: L, then W and U' with (I + L) W = b A K and
//    (I + L) U' = b V by blocks of 16 rows, P_ij = R_ij q_i.k_j, R_Cj k_j and A;
//  * delta_chunk_scan, a workgroup per (request, head, 16 columns of S), the chain: U = U' - W S, then the state;
//    four wavefronts share a chunk's rows and meet twice, the next chunk's operands on their way meanwhile;
//  * delta_chunk_out, a workgroup a (chunk, head, 16 columns), all at once: O = A q S + P U.
// 1,500 tokens, 16 heads of 64 x 64: 266 us token by token (in a chain of such calls), 72 as these three (24 + 36 + 12);
// three requests of 2,048 tokens in all 207 and 84.
//
// v_mfma_f32_16x16x4_f32: lane l gives row l % 16 of the first operand and column l % 16 of the second at one of 4 values
// of k, and holds rows 4 (l / 16) + e of column l % 16 of the sums.  Both operands take k in the order in which 16 bytes a
// lane bring it: value e of quarter l / 16 of a piece of 16 is k = 4 (l / 16) + e in step e.
#include "common.h"

namespace {

typedef float dc_f4 __attribute__((ext_vector_type(4)));
#define DC_ROWS 64                 // tokens of a chunk, and numbers of a key
#define DC_PITCH 68                // floats between rows in LDS

// floats of a (chunk, head) in the workspace: W [token][d], R_Cj k_j [d][token], P [token][token], A [token], then
// U [column][token] and the state before the chunk [column][d]
constexpr size_t DC_W = 0, DC_KT = 4096, DC_P = 8192, DC_A = 12288, DC_U = 12352;
__host__ __device__ constexpr size_t dc_floats(int V) { return DC_U + static_cast<size_t>(2) * DC_ROWS * V; }

// the sums of four pieces, added up as a tree (one chain over all 64 values of k rounds about half as much again)
__device__ __forceinline__ dc_f4 dc_total(const dc_f4 (&x)[4]) { return (x[0] + x[1]) + (x[2] + x[3]); }
// sum += a piece of 16 values of k of both operands
__device__ __forceinline__ dc_f4 dc_piece(const dc_f4 a, const dc_f4 b, dc_f4 sum) {
#pragma unroll
    for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], sum, 0, 0, 0);
    return sum;
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

__global__ __launch_bounds__(256) void delta_chunk_prepare_kernel(const float* __restrict__ qk, const float* __restrict__ v,
                                                                  const float* __restrict__ beta_decay, const int* __restrict__ cu_seqlens,
                                                                  float* __restrict__ ws, const int n_seqs, const int least, const int G,
                                                                  const int H, const int V) {
    constexpr int D = DC_ROWS, C = DC_ROWS, P = DC_PITCH;
    extern __shared__ __attribute__((aligned(16))) float dc_lds[];
    float* const ks = dc_lds;                  // K [token][d]
    float* const ls = ks + C * P;              // L [token][token]
    float* const xs = ls + C * P;              // W and U', [column][token]
    __shared__ float a_s[C], b_s[C], tile_before[C], tile_behind[C], all_before[C], all_behind[C];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / CELEG_WAVE), lane = tid % CELEG_WAVE;
    const int r16 = lane & 15, q = lane >> 4;
    const int h = blockIdx.y, g = h / (H / G);
    int row0, rows;
    if (!dc_find(cu_seqlens, n_seqs, least, blockIdx.x, row0, rows)) return;
    const size_t ldqk = static_cast<size_t>(2) * G * D;
    const float* const q_rows = qk + row0 * ldqk + static_cast<size_t>(g) * D;
    const float* const k_rows = q_rows + static_cast<size_t>(G) * D;
    float* const mine = ws + (static_cast<size_t>(blockIdx.x) * H + h) * dc_floats(V);
    // this wavefront's tiles on and under the diagonal (of 10, up to 3 of k.k and 3 of q.k); the queries' rows are asked for now
    const auto tile_row = [](int tile) { return tile < 1 ? 0 : tile < 3 ? 1 : tile < 6 ? 2 : 3; };
    const int q_tile0 = (wave + 2) & 3;
    dc_f4 q4[3][4];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int p = 0; p < 4; ++p)
            q4[i][p] = *reinterpret_cast<const dc_f4*>(q_rows + min(16 * tile_row(min(q_tile0 + 4 * i, 9)) + r16, rows - 1) * ldqk + 16 * p + 4 * q);
    // tokens behind the portion's last: no key, nothing written, no decay
    if (tid < C) {
        const float* const bd = beta_decay + static_cast<size_t>(row0 + min(tid, rows - 1)) * 2 * H + h;
        b_s[tid] = tid < rows ? bd[0] : 0.f;
        a_s[tid] = tid < rows ? bd[H] : 1.f;
    }
#pragma unroll
    for (int i = 0; i < C * D / 4 / 256; ++i) {
        const int at = tid + 256 * i, row = at >> 4, d = 4 * (at & 15);
        dc_f4 x = *reinterpret_cast<const dc_f4*>(k_rows + min(row, rows - 1) * ldqk + d);
        if (row >= rows) x = dc_f4{0.f, 0.f, 0.f, 0.f};
        *reinterpret_cast<dc_f4*>(ks + row * P + d) = x;
    }
    __syncthreads();
    // products of decays: over the token's tile of 16 up to it and from behind it on, and over the chunk
    if (wave == 0) {
        float before = a_s[lane], behind = r16 == 15 ? 1.f : a_s[lane + 1 < C ? lane + 1 : lane];
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) {
            const float b = __shfl_up(before, off, 16), e = __shfl_down(behind, off, 16);
            if (r16 >= off) before *= b;
            if (r16 + off < 16) behind *= e;
        }
        tile_before[lane] = before;
        tile_behind[lane] = behind;
        float all = before, rest = behind;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float whole = __shfl(before, 16 * t + 15, CELEG_WAVE);
            if (t < q) all *= whole;
            if (t > q) rest *= whole;
        }
        all_before[lane] = all;
        all_behind[lane] = rest;
        mine[DC_A + lane] = all;
    }
    __syncthreads();
    // the right sides b A K and b V
    for (int at = tid; at < C * D / 4; at += 256) {
        const int row = at & 63, d = 4 * (at >> 6);
        const float f = b_s[row] * all_before[row];
        const dc_f4 x = *reinterpret_cast<const dc_f4*>(ks + row * P + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) xs[(d + e) * P + row] = f * x[e];
    }
    for (int at = tid; at < C * V / 4; at += 256) {
        const int row = at / (V / 4), j = 4 * (at - row * (V / 4));
        const dc_f4 x = *reinterpret_cast<const dc_f4*>(v + static_cast<size_t>(row0 + min(row, rows - 1)) * H * V + static_cast<size_t>(h) * V + j);
#pragma unroll
        for (int e = 0; e < 4; ++e) xs[(D + j + e) * P + row] = b_s[row] * x[e];
    }
    // the tiles of k.k (L) and of q.k (P)
    const auto decays = [&](int ti, int tj) {
        dc_f4 decay;
        if (ti == tj) {
            float r = 1.f;
#pragma unroll
            for (int m = 1; m < 16; ++m) r *= m > r16 && m <= 4 * q ? a_s[16 * ti + m] : 1.f;
            decay[0] = r;
#pragma unroll
            for (int e = 1; e < 4; ++e) decay[e] = 4 * q + e > r16 ? decay[e - 1] * a_s[16 * ti + 4 * q + e] : 1.f;
        } else {
            float r = tile_behind[16 * tj + r16];
            for (int t = tj + 1; t < ti; ++t) r *= tile_before[16 * t + 15];
#pragma unroll
            for (int e = 0; e < 4; ++e) decay[e] = tile_before[16 * ti + 4 * q + e] * r;
        }
        return decay;
    };
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int k_tile = wave + 4 * i, q_tile = q_tile0 + 4 * i;
        const dc_f4 zero = {0.f, 0.f, 0.f, 0.f};
        dc_f4 part[4];
        if (k_tile < 10) {
            const int ti = tile_row(k_tile), tj = k_tile - ti * (ti + 1) / 2;
#pragma unroll
            for (int p = 0; p < 4; ++p)
                part[p] = dc_piece(*reinterpret_cast<const dc_f4*>(ks + (16 * ti + r16) * P + 16 * p + 4 * q),
                                   *reinterpret_cast<const dc_f4*>(ks + (16 * tj + r16) * P + 16 * p + 4 * q), zero);
            const dc_f4 sum = dc_total(part), decay = decays(ti, tj);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = 16 * ti + 4 * q + e, j = 16 * tj + r16;
                ls[row * P + j] = row > j ? b_s[row] * (decay[e] * sum[e]) : 0.f;
            }
        }
        if (q_tile < 10) {
            const int ti = tile_row(q_tile), tj = q_tile - ti * (ti + 1) / 2;
#pragma unroll
            for (int p = 0; p < 4; ++p)
                part[p] = dc_piece(q4[i][p], *reinterpret_cast<const dc_f4*>(ks + (16 * tj + r16) * P + 16 * p + 4 * q), zero);
            const dc_f4 sum = dc_total(part), decay = decays(ti, tj);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = 16 * ti + 4 * q + e, j = 16 * tj + r16;
                mine[DC_P + row * C + j] = row >= j ? decay[e] * sum[e] : 0.f;
            }
        }
    }
    __syncthreads();
    // (I + L) X = right sides, 16 rows at a time: a thread a column inside the block, the rows behind it on the matrix cores
    const int columns = D + V;
    for (int t = 0; t < 4; ++t) {
        if (tid < columns) {
            float x[16];
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const dc_f4 x4 = *reinterpret_cast<const dc_f4*>(xs + tid * P + 16 * t + 4 * p);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[4 * p + e] = x4[e];
            }
#pragma unroll
            for (int i = 1; i < 16; ++i)
#pragma unroll
                for (int p = 0; 4 * p < i; ++p) {
                    const dc_f4 l4 = *reinterpret_cast<const dc_f4*>(ls + (16 * t + i) * P + 16 * t + 4 * p);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (4 * p + e < i) x[i] = fmaf(-l4[e], x[4 * p + e], x[i]);
                }
#pragma unroll
            for (int p = 0; p < 4; ++p)
                *reinterpret_cast<dc_f4*>(xs + tid * P + 16 * t + 4 * p) = dc_f4{x[4 * p], x[4 * p + 1], x[4 * p + 2], x[4 * p + 3]};
        }
        __syncthreads();
        const int n_tiles = columns / 16;
        for (int job = wave; job < (3 - t) * n_tiles; job += 4) {
            const int below = t + 1 + job / n_tiles, col = 16 * (job % n_tiles) + r16;
            const dc_f4 l4 = *reinterpret_cast<const dc_f4*>(ls + (16 * below + r16) * P + 16 * t + 4 * q);
            dc_f4* const to = reinterpret_cast<dc_f4*>(xs + col * P + 16 * below + 4 * q);
            *to = dc_piece(-l4, *reinterpret_cast<const dc_f4*>(xs + col * P + 16 * t + 4 * q), *to);
        }
        __syncthreads();
    }
    for (int at = tid; at < C * D / 4; at += 256) {
        const int row = at >> 4, d = 4 * (at & 15);
        dc_f4 w, k;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            w[e] = xs[(d + e) * P + row];
            k[e] = all_behind[d + e] * ks[(d + e) * P + row];       // (here `row` is the key's number d, and d + e the token)
        }
        *reinterpret_cast<dc_f4*>(mine + DC_W + row * D + d) = w;
        *reinterpret_cast<dc_f4*>(mine + DC_KT + row * C + d) = k;
    }
    for (int at = tid; at < V * C / 4; at += 256) {
        const int col = at >> 4, row = 4 * (at & 15);
        *reinterpret_cast<dc_f4*>(mine + DC_U + static_cast<size_t>(col) * C + row) = *reinterpret_cast<const dc_f4*>(xs + (D + col) * P + row);
    }
}

__global__ __launch_bounds__(256) void delta_chunk_scan_kernel(float* __restrict__ state, const size_t state_stride,
                                                               const int* __restrict__ cu_seqlens, const int* __restrict__ seq_slot,
                                                               float* __restrict__ ws, const int least, const int H, const int V) {
    constexpr int D = DC_ROWS, C = DC_ROWS, P = DC_PITCH;
    __shared__ __attribute__((aligned(16))) float s_s[16 * P], u_s[16 * P];       // [column][d] and [column][token]
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
    const size_t tile = static_cast<size_t>(16 * wave + r16) * 64 + 4 * q, column = static_cast<size_t>(n0 + r16) * 64 + 16 * wave + 4 * q;
    const int lds_own = r16 * P + 16 * wave + 4 * q, lds_all = r16 * P + 4 * q;
    dc_f4 state4;
#pragma unroll
    for (int e = 0; e < 4; ++e) state4[e] = mine[static_cast<size_t>(16 * wave + 4 * q + e) * V];
    dc_f4 w[4], k[4], u;
    float decay;
    auto fetch = [&](const float* from) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            w[p] = *reinterpret_cast<const dc_f4*>(from + DC_W + tile + 16 * p);
            k[p] = *reinterpret_cast<const dc_f4*>(from + DC_KT + tile + 16 * p);
        }
        u = *reinterpret_cast<const dc_f4*>(from + DC_U + column);
        decay = from[DC_A + C - 1];
    };
    // (everybody's writes to LDS are there, while loads from memory stay on their way)
    auto meet = [] {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    fetch(at);
    for (int c = 0; c < chunks; ++c, at += stride) {
        dc_f4 w_now[4], k_now[4], u_now = u;
        const float decay_now = decay;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            w_now[p] = -w[p];
            k_now[p] = k[p];
        }
        if (c + 1 < chunks) fetch(at + stride);
        *reinterpret_cast<dc_f4*>(s_s + lds_own) = state4;
        *reinterpret_cast<dc_f4*>(at + DC_U + static_cast<size_t>(V) * C + column) = state4;      // (the state before the chunk, for delta_chunk_out)
        meet();
        dc_f4 in[4], part[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            in[p] = *reinterpret_cast<const dc_f4*>(s_s + lds_all + 16 * p);
            part[p] = dc_f4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int p = 0; p < 4; ++p) part[p] = __builtin_amdgcn_mfma_f32_16x16x4f32(w_now[p][e], in[p][e], part[p], 0, 0, 0);
        u_now += dc_total(part);
        *reinterpret_cast<dc_f4*>(u_s + lds_own) = u_now;
        *reinterpret_cast<dc_f4*>(at + DC_U + column) = u_now;
        meet();
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            in[p] = *reinterpret_cast<const dc_f4*>(u_s + lds_all + 16 * p);
            part[p] = dc_f4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int p = 0; p < 4; ++p) part[p] = __builtin_amdgcn_mfma_f32_16x16x4f32(k_now[p][e], in[p][e], part[p], 0, 0, 0);
        const dc_f4 added = dc_total(part);
#pragma unroll
        for (int e = 0; e < 4; ++e) state4[e] = fmaf(state4[e], decay_now, added[e]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) mine[static_cast<size_t>(16 * wave + 4 * q + e) * V] = state4[e];
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
    const float* const q_row = qk + static_cast<size_t>(row0 + min(16 * wave + r16, rows - 1)) * 2 * G * D + static_cast<size_t>(g) * D + 4 * q;
    dc_f4 q4[4], p4[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        q4[p] = *reinterpret_cast<const dc_f4*>(q_row + 16 * p);
        p4[p] = *reinterpret_cast<const dc_f4*>(mine + DC_P + static_cast<size_t>(16 * wave + r16) * C + 16 * min(p, wave) + 4 * q);
    }
    const dc_f4 before = *reinterpret_cast<const dc_f4*>(mine + DC_A + 16 * wave + 4 * q);
    const int n0 = 16 * blockIdx.z;
    const float* const u = mine + DC_U + static_cast<size_t>(n0 + r16) * C + 4 * q;
    const float* const s = u + static_cast<size_t>(V) * C;
    dc_f4 s4[4], u4[4], part[4], near[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        s4[p] = *reinterpret_cast<const dc_f4*>(s + 16 * p);
        u4[p] = *reinterpret_cast<const dc_f4*>(u + 16 * min(p, wave));
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        part[p] = dc_piece(q4[p], s4[p], dc_f4{0.f, 0.f, 0.f, 0.f});
        near[p] = dc_f4{0.f, 0.f, 0.f, 0.f};
        if (p <= wave) near[p] = dc_piece(p4[p], u4[p], near[p]);
    }
    const dc_f4 sum = dc_total(part), inside = dc_total(near);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int row = 16 * wave + 4 * q + e;
        if (row < rows) out[static_cast<size_t>(row0 + row) * H * V + static_cast<size_t>(h) * V + n0 + r16] = fmaf(before[e], sum[e], inside[e]);
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
    const size_t lds = static_cast<size_t>(2 * DC_ROWS + DC_ROWS + V) * DC_PITCH * sizeof(float);
    static bool raised = false;        // (V = 128: 87 KB)
    if (!raised) {
        hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(&delta_chunk_prepare_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
        if (err != hipSuccess) return static_cast<int>(err);
        raised = true;
    }
    hipLaunchKernelGGL(delta_chunk_prepare_kernel, dim3(max_chunks, H), dim3(256), lds, stream, qk, v, beta_decay, cu_seqlens, ws, n_seqs, least,
                       G, H, V);
    hipLaunchKernelGGL(delta_chunk_scan_kernel, dim3(n_seqs, H, V / 16), dim3(256), 0, stream, state, state_stride, cu_seqlens, seq_slot, ws,
                       least, H, V);
    hipLaunchKernelGGL(delta_chunk_out_kernel, dim3(max_chunks, H, V / 16), dim3(256), 0, stream, qk, cu_seqlens, ws, out, n_seqs, least, G, H, V);
    return CELEG_LAUNCH_RESULT();
}
