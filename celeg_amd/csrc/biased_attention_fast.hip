// Softmax attention with a factor per query position and a distance bias per head, bfloat16, on
// the matrix cores:
//     score(i, j) = (q_i . k_j) * scale * f(i) - r1[h] * ln(1 + r2[h] * (i - j)),   weights = softmax over the visible j
// Visible: j <= i, inside the window where there is one, or among the first `keep_first` positions.  The
// denominator may hold one more term, a key without a value that the row meets before all others: of score 0
// (`sink_one`) or of a learned score per head (`sink`).  With `softcap` c a scaled score s is bent to
// c * tanh(s / c) = c - 2 c / (exp(2 s / c) + 1) before the bias.
// Keys of `D` numbers, values of `V` numbers a head (multiples of 32 up to 128: FULL), or of fewer, keys in
// multiples of 8 and values in multiples of 4, which are staged with zeros behind them (not FULL).
// Cache layout: K [pages, layers, kv_heads, page_tokens, D], V [pages, layers, kv_heads, V, page_tokens].
//
// Scores are computed transposed (keys as the first operand of a 16x16x32 instruction): a lane
// holds, of row r = lane % 16, the keys 16 kt + 4 (lane / 16) + i of each of a block's four tiles.
// Two tiles' weights are the second operand of the product with the values without any exchange
// between lanes; a 32-bit weight goes into that product as two bfloat16 numbers (its rounding and
// the rest), so the weights keep sixteen bits and more where the values have eight.  The softmax runs over blocks of 64 keys with a running
// maximum and normaliser per row in 32-bit, everything in powers of two (log2 e is folded into the
// scale, and r1 ln(x) log2 e = r1 log2(x)): the four lanes of a row agree on the maximum by two
// exchanges a block and keep a sum each, which meet once at the end.
//
// Three forms.  Portions of prompts: a workgroup per (64 rows of one request's step, query head), 16
// rows a wavefront; a key block is staged once for the four wavefronts into one of two buffers in
// turn while the block before is multiplied.  Short portions: a workgroup per
// (16 rows, query head) whose wavefronts take the key blocks in turn, each staging its own, and
// whose maxima, normalisers and sums meet in LDS at the end, in the order of the wavefronts.
// Single tokens: below.
#include "common.h"

#include <algorithm>

namespace {

typedef __bf16 bf_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf_bf16x4 __attribute__((ext_vector_type(4)));
typedef float bf_f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int bf_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int bf_u32x2 __attribute__((ext_vector_type(2)));

#define BF_WAVES 4
#define BF_KEYS 64
#define BF_LOG2E 1.44269504089f

__device__ __forceinline__ float bf_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float bf_log2(float x) { return __builtin_amdgcn_logf(x); }
__device__ __forceinline__ float bf_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float bf_query_factor(int p, float coef, int every) {
    return every > 0 ? 1.0f + coef * logf(static_cast<float>((p + 1) / every) + 1.0f) : 1.0f;
}

// what a lane carries of its row's softmax
template <int DT>
struct BfRow {
    float top = -INFINITY, sum = 0.f;        // the row's running maximum (the same in its four lanes); this lane's share of the normaliser
    bf_f32x4 acc[DT];
};

// the pieces of a key block that a thread brings from the pages: keys kb .. kb + 63 (those past
// pos_last: the last one again), values with zeros past pos_last
template <int D, int V, int THREADS, bool FULL>
struct BfFetch {
    static constexpr int KCH = BF_KEYS * (D / 8) / THREADS, VCH = V * (BF_KEYS / 8) / THREADS;
    bf_u32x4 k[KCH], v[VCH];
    __device__ __forceinline__ void load(int tid, int kb, int pos_last, const bf16* __restrict__ k_pool, const bf16* __restrict__ v_pool,
                                         const int* __restrict__ pages, int page_shift, int page_mask, int page_tokens,
                                         size_t head_index_stride, int kvh, size_t layer_index, int kd_, int vd_) {
        const int kd = FULL ? D : kd_, vd = FULL ? V : vd_;
        // (all pages, then all pieces, without conditions: a load under a condition of its own is waited for
        // before the next one is asked for; a thread's pieces of the values are of the same eight keys, which lie
        // side by side in one page.  4 requests at 1,100
        // keys, 16 heads of 64: 17.2 us; with a condition around each of the values' loads 21.7)
        static_assert(THREADS % (BF_KEYS / 8) == 0, "a thread's pieces of the values lie in one page");
        const int v_key = kb + 8 * (tid % (BF_KEYS / 8)), v_from = min(v_key, pos_last & ~7);
        const int v_page = pages[v_from >> page_shift];
        int k_page[KCH];
#pragma unroll
        for (int i = 0; i < KCH; ++i) k_page[i] = pages[min(kb + (tid + THREADS * i) / (D / 8), pos_last) >> page_shift];
#pragma unroll
        for (int i = 0; i < KCH; ++i) {
            const int c = tid + THREADS * i, part = c % (D / 8), key = min(kb + c / (D / 8), pos_last);
            const size_t head = (static_cast<size_t>(k_page[i]) * head_index_stride + layer_index) + kvh;
            // (pieces behind the head's last number bring that one's piece again and are zeroed)
            k[i] = *reinterpret_cast<const bf_u32x4*>(k_pool + (head * page_tokens + (key & page_mask)) * kd + (FULL ? 8 * part : min(8 * part, kd - 8)));
            if (!FULL && 8 * part >= kd) k[i] = bf_u32x4{0u, 0u, 0u, 0u};
        }
        const bf16* const v_src = v_pool + ((static_cast<size_t>(v_page) * head_index_stride + layer_index) + kvh) * vd * page_tokens + (v_from & page_mask);
#pragma unroll
        for (int i = 0; i < VCH; ++i) {
            const int d = (tid + THREADS * i) / (BF_KEYS / 8);
            v[i] = *reinterpret_cast<const bf_u32x4*>(v_src + static_cast<size_t>(FULL ? d : min(d, vd - 1)) * page_tokens);
            if (!FULL && d >= vd) v[i] = bf_u32x4{0u, 0u, 0u, 0u};
        }
        if (kb + BF_KEYS - 1 > pos_last) {         // zeros past pos_last
            const int live = pos_last - v_key + 1;
#pragma unroll
            for (int i = 0; i < VCH; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    v[i][j] &= (live > 2 * j ? 0x0000ffffu : 0u) | (live > 2 * j + 1 ? 0xffff0000u : 0u);
        }
    }
    __device__ __forceinline__ void stage(int tid, __bf16* ks, __bf16* vs) const {
        constexpr int KROW = D + 8, VROW = BF_KEYS + 8;
#pragma unroll
        for (int i = 0; i < KCH; ++i) {
            const int c = tid + THREADS * i;
            *reinterpret_cast<bf_u32x4*>(ks + (c / (D / 8)) * KROW + 8 * (c % (D / 8))) = k[i];
        }
#pragma unroll
        for (int i = 0; i < VCH; ++i) {
            const int c = tid + THREADS * i;
            *reinterpret_cast<bf_u32x4*>(vs + (c / (BF_KEYS / 8)) * VROW + 8 * (c % (BF_KEYS / 8))) = v[i];
        }
    }
};

// one staged block of 64 keys for the 16 rows of a wavefront
template <int D, int V>
__device__ __forceinline__ void bf_block(const __bf16* ks, const __bf16* vs, const bf_bf16x8 (&qreg)[D / 32], BfRow<V / 16>& row, int kb,
                                         int my_pos, int window, int keep_first, bool kept_only, int r, int quad, float s2, float b1, float b2,
                                         bool biased, float cap2) {
    constexpr int KROW = D + 8, VROW = BF_KEYS + 8, KS = D / 32, DT = V / 16;
    bf_f32x4 sacc[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
        sacc[kt] = bf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < KS; ++st) {
            const bf_bf16x8 kf = __builtin_bit_cast(bf_bf16x8, *reinterpret_cast<const bf_u32x4*>(ks + (16 * kt + r) * KROW + 32 * st + 8 * quad));
            sacc[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qreg[st], sacc[kt], 0, 0, 0);
        }
    }
    float top = -INFINITY;
    if (cap2 > 0.f) {
        // bent scores: s2 holds 2 log2(e) scale f / c, cap2 is c log2(e)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                sacc[kt][i] = fmaf(-2.0f * cap2, __builtin_amdgcn_rcpf(bf_exp2(sacc[kt][i] * s2) + 1.0f), cap2);
        s2 = 1.0f;
    }
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int key = kb + 16 * kt + 4 * quad + i;
            const bool seen = key <= my_pos && (kept_only ? key < keep_first : (window <= 0 || key > my_pos - window || key < keep_first));
            float x = sacc[kt][i] * s2;
            if (biased) x -= b1 * bf_log2(fmaf(b2, static_cast<float>(my_pos - key), 1.0f));
            x = seen ? x : -INFINITY;
            sacc[kt][i] = x;
            top = fmaxf(top, x);
        }
    top = max_half32(max_row16(top));
    const float new_top = fmaxf(row.top, top);
    const float base = new_top == -INFINITY ? 0.f : new_top;      // (a row that has seen no key yet: every weight 0)
    const float keep = bf_exp2(row.top - base);
    row.top = new_top;
    float sum = 0.f;
    bf_bf16x4 w[4], rest[4];         // a weight as two bfloat16 numbers: its rounding, and what the rounding left
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float p = bf_exp2(sacc[kt][i] - base);
            sum += p;
            w[kt][i] = static_cast<__bf16>(p);
            rest[kt][i] = static_cast<__bf16>(p - static_cast<float>(w[kt][i]));
        }
    row.sum = fmaf(row.sum, keep, sum);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) row.acc[dt][i] *= keep;
    // output, transposed: tile dt holds values 16 dt + 4 quad + i of row r
#pragma unroll
    for (int pair = 0; pair < 2; ++pair) {
        const bf_bf16x8 pw = __builtin_shufflevector(w[2 * pair], w[2 * pair + 1], 0, 1, 2, 3, 4, 5, 6, 7);
        const bf_bf16x8 pr = __builtin_shufflevector(rest[2 * pair], rest[2 * pair + 1], 0, 1, 2, 3, 4, 5, 6, 7);
        bf_bf16x8 vf[DT];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const __bf16* vrow = vs + (16 * dt + r) * VROW + 32 * pair + 4 * quad;
            const bf_u32x2 lo = *reinterpret_cast<const bf_u32x2*>(vrow), hi = *reinterpret_cast<const bf_u32x2*>(vrow + 16);
            vf[dt] = __builtin_bit_cast(bf_bf16x8, bf_u32x4{lo[0], lo[1], hi[0], hi[1]});
            row.acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt], pw, row.acc[dt], 0, 0, 0);
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) row.acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt], pr, row.acc[dt], 0, 0, 0);
    }
}

// a finished row: divided by its normaliser, times sigmoid(gate), stored
template <int V, bool FULL>
__device__ __forceinline__ void bf_store(const BfRow<V / 16>& row, float total, const bf16* __restrict__ gate_row, bf16* __restrict__ out_row,
                                         int quad, int vd) {
    const float inv = 1.0f / total;
#pragma unroll
    for (int dt = 0; dt < V / 16; ++dt) {
        if (!FULL && 16 * dt + 4 * quad >= vd) continue;
        float g[4] = {1.f, 1.f, 1.f, 1.f};
        if (gate_row) {
            const bf_bf16x4 g4 = __builtin_bit_cast(bf_bf16x4, *reinterpret_cast<const bf_u32x2*>(gate_row + 16 * dt + 4 * quad));
#pragma unroll
            for (int i = 0; i < 4; ++i) g[i] = bf_sigmoid(static_cast<float>(g4[i]));
        }
        const bf_bf16x4 o4 = {static_cast<__bf16>(row.acc[dt][0] * inv * g[0]), static_cast<__bf16>(row.acc[dt][1] * inv * g[1]),
                              static_cast<__bf16>(row.acc[dt][2] * inv * g[2]), static_cast<__bf16>(row.acc[dt][3] * inv * g[3])};
        *reinterpret_cast<bf_bf16x4*>(out_row + 16 * dt + 4 * quad) = o4;
    }
}

struct BfArgs {
    const bf16* q;
    const bf16* k_pool;
    const bf16* v_pool;
    const int* table;
    const int* cu_seqlens;
    const int* seq_slot;
    const int* seq_start;
    const float* r1;
    const float* r2;
    const float* sink;
    const bf16* gate;
    bf16* out;
    int ldq, ldg, ldo, table_stride, n_seqs, q_heads, kv_heads, page_tokens, n_layers, layer, every, window, keep_first, sink_one, kd, vd;
    float scale, coef, softcap;
};

// The key blocks of a tile whose lowest position is pos0: first the blocks that hold the kept first keys
// where the window has passed them (only those keys count there), then the blocks from the window's start on.
template <int KEYS>
struct BfBlocks {
    int n_kept, kb0;
    __device__ __forceinline__ BfBlocks(int pos0, int window, int keep) {
        const int key_first = window > 0 ? max(0, pos0 - window + 1) : 0;
        kb0 = key_first & ~7;
        n_kept = 0;
        if (keep > 0 && kb0 > 0) {
            if (kb0 >= keep) n_kept = (keep + KEYS - 1) / KEYS;
            else kb0 = 0;                 // the window begins among the kept keys: one run from the start
        }
    }
    __device__ __forceinline__ int count(int pos_last) const { return n_kept + (pos_last >= kb0 ? (pos_last - kb0) / KEYS + 1 : 0); }
    __device__ __forceinline__ bool kept(int i) const { return i < n_kept; }
    __device__ __forceinline__ int start(int i) const { return i < n_kept ? i * KEYS : kb0 + (i - n_kept) * KEYS; }
    // the last key a block may touch: pages between the kept keys and the window may be gone
    __device__ __forceinline__ int last(int i, int pos_last, int keep) const { return i < n_kept ? keep - 1 : pos_last; }
};

// a row's factor on the products q.k (in powers of two) and, where scores are bent, the bend in those units
__device__ __forceinline__ float bf_score_factor(const BfArgs& a, int pos, float& cap2) {
    const float s = a.scale * bf_query_factor(pos, a.coef, a.every) * BF_LOG2E;
    cap2 = a.softcap > 0.f ? a.softcap * BF_LOG2E : 0.f;
    return a.softcap > 0.f ? 2.0f * s / a.softcap : s;
}

// which tile of `rows` rows: tiles of all requests of the step, one after the other
__device__ __forceinline__ bool bf_find_tile(const BfArgs& a, int rows, int& tile, int& s, int& row0, int& n) {
    for (s = 0; s < a.n_seqs; ++s) {
        row0 = a.cu_seqlens[s];
        n = a.cu_seqlens[s + 1] - row0;
        const int tiles = (n + rows - 1) / rows;
        if (tile < tiles) return true;
        tile -= tiles;
    }
    return false;
}

template <int D, int V, bool FULL>
__global__ __launch_bounds__(BF_WAVES * CELEG_WAVE) void biased_attention_rows_kernel(const BfArgs a) {
    constexpr int KROW = D + 8, VROW = BF_KEYS + 8, KS = D / 32, DT = V / 16, BUF = BF_KEYS * KROW + V * VROW;
    const int kd = FULL ? D : a.kd, vd = FULL ? V : a.vd;
    constexpr int THREADS = BF_WAVES * CELEG_WAVE;
    extern __shared__ __attribute__((aligned(16))) unsigned char bf_lds[];
    __bf16* lds = reinterpret_cast<__bf16*>(bf_lds);
    const int wave = threadIdx.x / CELEG_WAVE, lane = threadIdx.x % CELEG_WAVE, tid = threadIdx.x;
    int tile = blockIdx.x, s, row0, n;
    if (!bf_find_tile(a, 64, tile, s, row0, n)) return;
    const int h = blockIdx.y, kvh = h / (a.q_heads / a.kv_heads);
    const int r = lane & 15, quad = lane >> 4;
    const int tile_row = tile * 64, tile_rows = min(64, n - tile_row);
    const int tile_pos0 = a.seq_start[s] + tile_row, pos_last = tile_pos0 + tile_rows - 1;
    const int first_row = tile_row + 16 * wave, rows_here = min(16, n - first_row);      // <= 0: this wavefront only stages
    const int my_row = first_row + max(0, min(r, rows_here - 1));
    const int safe_row = min(my_row, n - 1);
    const int my_pos = a.seq_start[s] + safe_row;
    const int wave_pos0 = a.seq_start[s] + first_row, wave_last = wave_pos0 + rows_here - 1;
    const int* pages = a.table + static_cast<size_t>(a.seq_slot[s]) * a.table_stride;
    float cap2;
    const float s2 = bf_score_factor(a, my_pos, cap2);
    const bool biased = a.r1 != nullptr;
    const float b1 = biased ? a.r1[h] : 0.f, b2 = biased ? a.r2[h] : 0.f;
    bf_bf16x8 qreg[KS];
    const bf16* qrow = a.q + static_cast<size_t>(row0 + safe_row) * a.ldq + static_cast<size_t>(h) * kd;
#pragma unroll
    for (int st = 0; st < KS; ++st) {
        bf_u32x4 piece = {0u, 0u, 0u, 0u};
        if (FULL || 32 * st + 8 * quad < kd) piece = *reinterpret_cast<const bf_u32x4*>(qrow + 32 * st + 8 * quad);
        qreg[st] = __builtin_bit_cast(bf_bf16x8, piece);
    }
    BfRow<DT> row;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) row.acc[dt] = bf_f32x4{0.f, 0.f, 0.f, 0.f};
    if (a.sink_one || a.sink) {
        row.top = a.sink ? a.sink[h] * BF_LOG2E : 0.f;
        row.sum = quad == 0 ? 1.f : 0.f;
    }
    const int page_shift = 31 - __builtin_clz(a.page_tokens), page_mask = a.page_tokens - 1;
    const size_t head_index_stride = static_cast<size_t>(a.n_layers) * a.kv_heads, layer_index = static_cast<size_t>(a.layer) * a.kv_heads;
    BfFetch<D, V, THREADS, FULL> pre;
    const BfBlocks<BF_KEYS> blocks(tile_pos0, a.window, a.keep_first);
    const int n_blocks = blocks.count(pos_last);
    pre.load(tid, blocks.start(0), blocks.last(0, pos_last, a.keep_first), a.k_pool, a.v_pool, pages, page_shift, page_mask, a.page_tokens,
             head_index_stride, kvh, layer_index, kd, vd);
    int turn = 0;
    for (int i = 0; i < n_blocks; ++i, turn ^= 1) {
        const int kb = blocks.start(i);
        __bf16* ks = lds + turn * BUF;
        __bf16* vs = ks + BF_KEYS * KROW;
        pre.stage(tid, ks, vs);
        __syncthreads();
        if (i + 1 < n_blocks)
            pre.load(tid, blocks.start(i + 1), blocks.last(i + 1, pos_last, a.keep_first), a.k_pool, a.v_pool, pages, page_shift, page_mask,
                     a.page_tokens, head_index_stride, kvh, layer_index, kd, vd);
        // blocks none of this wavefront's rows can see
        if (rows_here <= 0) continue;
        if (!blocks.kept(i) && (kb > wave_last || (a.window > 0 && kb >= a.keep_first && kb + BF_KEYS - 1 < wave_pos0 - a.window + 1))) continue;
        bf_block<D, V>(ks, vs, qreg, row, kb, my_pos, a.window, a.keep_first, blocks.kept(i), r, quad, s2, b1, b2, biased, cap2);
    }
    float total = row.sum;
    total = sum_half32(sum_row16(total));
    if (r >= rows_here) return;
    const size_t at = static_cast<size_t>(row0 + my_row);
    bf_store<V, FULL>(row, total, a.gate ? a.gate + at * a.ldg + static_cast<size_t>(h) * vd : nullptr, a.out + at * a.ldo + static_cast<size_t>(h) * vd,
                quad, vd);
}

// Wavefronts a SIMD that the registers leave room for. Where the staging areas of two workgroups of eight
// wavefronts fit LDS (heads of 32) they are four, so that two run on a compute unit (64 requests at 1,000 keys, 8
// heads: 24.6 us; with the five registers more that the compiler takes by itself, and one workgroup, 33.1).
constexpr int bf_tile_waves_a_simd(int d, int v, bool full) { return full && d <= 32 && v <= 32 ? 4 : 1; }
template <int D, int V, int WAVES, bool FULL>
__global__ __launch_bounds__(WAVES * CELEG_WAVE, bf_tile_waves_a_simd(D, V, FULL)) void biased_attention_tile_kernel(const BfArgs a) {
    constexpr int KROW = D + 8, VROW = BF_KEYS + 8, KS = D / 32, DT = V / 16, BUF = BF_KEYS * KROW + V * VROW;
    const int kd = FULL ? D : a.kd, vd = FULL ? V : a.vd;
    extern __shared__ __attribute__((aligned(16))) unsigned char bf_lds[];
    const int wave = threadIdx.x / CELEG_WAVE, lane = threadIdx.x % CELEG_WAVE;
    __bf16* ks = reinterpret_cast<__bf16*>(bf_lds) + static_cast<size_t>(wave) * BUF;
    __bf16* vs = ks + BF_KEYS * KROW;
    int tile = blockIdx.x, s, row0, n;
    if (!bf_find_tile(a, 16, tile, s, row0, n)) return;
    const int h = blockIdx.y, kvh = h / (a.q_heads / a.kv_heads);
    const int r = lane & 15, quad = lane >> 4;
    const int first_row = tile * 16, rows_here = min(16, n - first_row);
    const int pos0 = a.seq_start[s] + first_row, pos_last = pos0 + rows_here - 1;
    const int my_row = first_row + min(r, rows_here - 1);      // rows past the end repeat the last one (not stored)
    const int my_pos = a.seq_start[s] + my_row;
    const int* pages = a.table + static_cast<size_t>(a.seq_slot[s]) * a.table_stride;
    float cap2;
    const float s2 = bf_score_factor(a, my_pos, cap2);
    const bool biased = a.r1 != nullptr;
    const float b1 = biased ? a.r1[h] : 0.f, b2 = biased ? a.r2[h] : 0.f;
    bf_bf16x8 qreg[KS];
    const bf16* qrow = a.q + static_cast<size_t>(row0 + my_row) * a.ldq + static_cast<size_t>(h) * kd;
#pragma unroll
    for (int st = 0; st < KS; ++st) {
        bf_u32x4 piece = {0u, 0u, 0u, 0u};
        if (FULL || 32 * st + 8 * quad < kd) piece = *reinterpret_cast<const bf_u32x4*>(qrow + 32 * st + 8 * quad);
        qreg[st] = __builtin_bit_cast(bf_bf16x8, piece);
    }
    BfRow<DT> row;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) row.acc[dt] = bf_f32x4{0.f, 0.f, 0.f, 0.f};
    if ((a.sink_one || a.sink) && wave == 0) {        // (once a row: the first wavefront's share)
        row.top = a.sink ? a.sink[h] * BF_LOG2E : 0.f;
        row.sum = quad == 0 ? 1.f : 0.f;
    }
    const int page_shift = 31 - __builtin_clz(a.page_tokens), page_mask = a.page_tokens - 1;
    const size_t head_index_stride = static_cast<size_t>(a.n_layers) * a.kv_heads, layer_index = static_cast<size_t>(a.layer) * a.kv_heads;
    BfFetch<D, V, CELEG_WAVE, FULL> pre;
    const BfBlocks<BF_KEYS> blocks(pos0, a.window, a.keep_first);
    const int n_blocks = blocks.count(pos_last);
    if (wave < n_blocks)
        pre.load(lane, blocks.start(wave), blocks.last(wave, pos_last, a.keep_first), a.k_pool, a.v_pool, pages, page_shift, page_mask,
                 a.page_tokens, head_index_stride, kvh, layer_index, kd, vd);
    for (int i = wave; i < n_blocks; i += WAVES) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        pre.stage(lane, ks, vs);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (i + WAVES < n_blocks)
            pre.load(lane, blocks.start(i + WAVES), blocks.last(i + WAVES, pos_last, a.keep_first), a.k_pool, a.v_pool, pages, page_shift,
                     page_mask, a.page_tokens, head_index_stride, kvh, layer_index, kd, vd);
        bf_block<D, V>(ks, vs, qreg, row, blocks.start(i), my_pos, a.window, a.keep_first, blocks.kept(i), r, quad, s2, b1, b2, biased, cap2);
    }
    // the wavefronts' maxima, normalisers and sums meet in LDS (every wavefront's staging area is
    // free after the barrier); the first one joins them in the order of the wavefronts and stores
    constexpr int PER = DT * 4 + 2;
    __syncthreads();
    float* parts = reinterpret_cast<float*>(bf_lds);
    if (wave > 0) {
        float* mine = parts + static_cast<size_t>(wave - 1) * PER * CELEG_WAVE;
        mine[lane] = row.top;
        mine[CELEG_WAVE + lane] = row.sum;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) mine[(2 + dt * 4 + i) * CELEG_WAVE + lane] = row.acc[dt][i];
    }
    __syncthreads();
    if (wave > 0) return;
    float top = row.top;
#pragma unroll
    for (int w = 1; w < WAVES; ++w) top = fmaxf(top, parts[static_cast<size_t>(w - 1) * PER * CELEG_WAVE + lane]);
    // (the row's own key is visible, so the maximum over all wavefronts is finite)
    const float mine = bf_exp2(row.top - top);
    float total = row.sum * mine;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) row.acc[dt][i] *= mine;
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
        const float* theirs = parts + static_cast<size_t>(w - 1) * PER * CELEG_WAVE;
        const float f = bf_exp2(theirs[lane] - top);
        total = fmaf(theirs[CELEG_WAVE + lane], f, total);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) row.acc[dt][i] = fmaf(theirs[(2 + dt * 4 + i) * CELEG_WAVE + lane], f, row.acc[dt][i]);
    }
    total = sum_half32(sum_row16(total));
    if (r >= rows_here) return;
    const size_t at = static_cast<size_t>(row0 + my_row);
    bf_store<V, FULL>(row, total, a.gate ? a.gate + at * a.ldg + static_cast<size_t>(h) * vd : nullptr, a.out + at * a.ldo + static_cast<size_t>(h) * vd,
                quad, vd);
}

// ---- single tokens: a workgroup per (row, key/value head, part of the keys), the query heads that share the head as
// the rows of the matrix instruction (up to 16), eight wavefronts that take units of 32 keys in turn, over all parts.
// What bounds such a call is what one compute unit draws of the keys and values (some 50 GB/s: 1,100 keys of 64, 282 KB, 5.5
// us) and the chain position -> page -> keys -> weights -> sum.  So many keys are dealt to several workgroups, whose
// maxima, normalisers and sums a second kernel joins, and keys and values go from the pages straight into the
// registers of the matrix instruction: row 4 quad + i of score tile kt stands for key 8 quad + 4 kt + i of the
// unit, so that a lane ends up with the weights of the eight neighbouring keys that its 16 bytes of a page's values hold.
struct BfSingle {
    const int* positions;
    const int* token_slot;
    float* parts_out;         // [rows, kv_heads, parts, group, V + 2], or null with one part
    int parts;
};

#define BF_SINGLE_WAVES 8
#define BF_MAX_PARTS 8
#define BF_UNIT 32
template <int D, int V, bool FULL>
__global__ __launch_bounds__(BF_SINGLE_WAVES * CELEG_WAVE, (D <= 64 && V <= 64 ? 4 : 2)) void biased_attention_single_kernel(const BfArgs a, const BfSingle p) {
    constexpr int WAVES = BF_SINGLE_WAVES, KS = D / 32, DT = V / 16, VROW = V + 4;
    const int kd = FULL ? D : a.kd, vd = FULL ? V : a.vd;
    extern __shared__ __attribute__((aligned(16))) unsigned char bf_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / CELEG_WAVE), lane = threadIdx.x % CELEG_WAVE;
    const int t = blockIdx.x, kvh = blockIdx.y, group = a.q_heads / a.kv_heads;
    const int r = lane & 15, quad = lane >> 4;
    const int pos = p.positions[t];
    const int* const pages = a.table + static_cast<size_t>(p.token_slot[t]) * a.table_stride;
    const int h = kvh * group + min(r, group - 1);             // rows past the last head repeat it (not stored)
    const int page_shift = 31 - __builtin_clz(a.page_tokens), page_mask = a.page_tokens - 1;
    const BfBlocks<BF_UNIT> blocks(pos, a.window, a.keep_first);
    const int n_units = blocks.count(pos), stride = WAVES * p.parts, first = blockIdx.z * WAVES + wave;
    struct Unit {
        bf_u32x4 k[2][KS], v[DT];
    };
    auto page_of = [&](int u, int eighth) {
        const int i = min(u, n_units - 1);
        return pages[min(blocks.start(i) + 8 * eighth, blocks.last(i, pos, a.keep_first)) >> page_shift];
    };
    auto head_of = [&](int page) { return (static_cast<size_t>(page) * a.n_layers + a.layer) * a.kv_heads + kvh; };
    auto fetch = [&](int u, int k_page, int v_page, Unit& unit) __attribute__((always_inline)) {
        const int ub = blocks.start(u), last = blocks.last(u, pos, a.keep_first);
        const bf16* const k_head = a.k_pool + head_of(k_page) * a.page_tokens * kd;
        const bf16* const v_head = a.v_pool + head_of(v_page) * a.page_tokens * vd;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            const int key = min(ub + 8 * (r >> 2) + 4 * kt + (r & 3), last);
#pragma unroll
            for (int st = 0; st < KS; ++st) {
                const int d = 32 * st + 8 * quad;
                unit.k[kt][st] = *reinterpret_cast<const bf_u32x4*>(k_head + static_cast<size_t>(key & page_mask) * kd + (FULL ? d : min(d, kd - 8)));
            }
        }
        const int v_from = min(ub + 8 * quad, last & ~7);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const int d = 16 * dt + r;
            unit.v[dt] = *reinterpret_cast<const bf_u32x4*>(v_head + static_cast<size_t>(FULL ? d : min(d, vd - 1)) * a.page_tokens + (v_from & page_mask));
        }
    };
    Unit units[2];
    const int k_page0 = page_of(first, r >> 2), v_page0 = page_of(first, quad);
    int k_page = page_of(first + stride, r >> 2), v_page = page_of(first + stride, quad);
    float cap2;
    float s2 = bf_score_factor(a, pos, cap2);
    const bool biased = a.r1 != nullptr;
    const float b1 = biased ? a.r1[h] : 0.f, b2 = biased ? a.r2[h] : 0.f;
    bf_bf16x8 qreg[KS];
    const bf16* const qrow = a.q + static_cast<size_t>(t) * a.ldq + static_cast<size_t>(h) * kd;
#pragma unroll
    for (int st = 0; st < KS; ++st) {
        bf_u32x4 piece = {0u, 0u, 0u, 0u};
        if (FULL || 32 * st + 8 * quad < kd) piece = *reinterpret_cast<const bf_u32x4*>(qrow + 32 * st + 8 * quad);
        qreg[st] = __builtin_bit_cast(bf_bf16x8, piece);
    }
    BfRow<DT> row;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) row.acc[dt] = bf_f32x4{0.f, 0.f, 0.f, 0.f};
    if ((a.sink_one || a.sink) && first == 0) {       // (once a row: the first wavefront's share)
        row.top = a.sink ? a.sink[h] * BF_LOG2E : 0.f;
        row.sum = quad == 0 ? 1.f : 0.f;
    }
    auto take = [&](int u, Unit& unit) __attribute__((always_inline)) {
        const int ub = blocks.start(u), last = blocks.last(u, pos, a.keep_first);
        const bool kept_only = blocks.kept(u);
        if (!FULL) {                                  // pieces behind the head's last number are zeros
#pragma unroll
            for (int st = 0; st < KS; ++st)
                if (32 * st + 8 * quad >= kd) unit.k[0][st] = unit.k[1][st] = bf_u32x4{0u, 0u, 0u, 0u};
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                if (16 * dt + r >= vd) unit.v[dt] = bf_u32x4{0u, 0u, 0u, 0u};
        }
        if (ub + BF_UNIT - 1 > last) {                // what lies behind the last key may be anything
            const int live = last - (ub + 8 * quad) + 1;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    unit.v[dt][j] &= (live > 2 * j ? 0x0000ffffu : 0u) | (live > 2 * j + 1 ? 0xffff0000u : 0u);
        }
        float x[8], top = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            bf_f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < KS; ++st)
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf_bf16x8, unit.k[kt][st]), qreg[st], s, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = ub + 8 * quad + 4 * kt + i;
                const bool seen = key <= pos && (kept_only ? key < a.keep_first : (a.window <= 0 || key > pos - a.window || key < a.keep_first));
                float y = s[i] * s2;
                if (cap2 > 0.f) y = fmaf(-2.0f * cap2, __builtin_amdgcn_rcpf(bf_exp2(y) + 1.0f), cap2);      // (s2 holds 2 log2(e) scale f / c)
                if (biased) y -= b1 * bf_log2(fmaf(b2, static_cast<float>(pos - key), 1.0f));
                x[4 * kt + i] = seen ? y : -INFINITY;
                top = fmaxf(top, x[4 * kt + i]);
            }
        }
        top = max_half32(max_row16(top));
        const float new_top = fmaxf(row.top, top), base = new_top == -INFINITY ? 0.f : new_top;
        const float keep = bf_exp2(row.top - base);
        row.top = new_top;
        float sum = 0.f;
        bf_bf16x8 w, rest;                            // a weight as two bfloat16 numbers: its rounding, and what the rounding left
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float y = bf_exp2(x[e] - base);
            sum += y;
            w[e] = static_cast<__bf16>(y);
            rest[e] = static_cast<__bf16>(y - static_cast<float>(w[e]));
        }
        row.sum = fmaf(row.sum, keep, sum);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            row.acc[dt] *= keep;
            row.acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf_bf16x8, unit.v[dt]), w, row.acc[dt], 0, 0, 0);
            row.acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf_bf16x8, unit.v[dt]), rest, row.acc[dt], 0, 0, 0);
        }
    };
    if (first < n_units) fetch(first, k_page0, v_page0, units[0]);
    if (first + stride < n_units) fetch(first + stride, k_page, v_page, units[1]);
    for (int u = first; u < n_units; u += 2 * stride) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int mine = u + e * stride;
            if (mine >= n_units) break;
            const bool more = mine + 2 * stride < n_units;
            if (more) {
                k_page = page_of(mine + 2 * stride, r >> 2);
                v_page = page_of(mine + 2 * stride, quad);
            }
            take(mine, units[e]);
            if (more) fetch(mine + 2 * stride, k_page, v_page, units[e]);
        }
    }
    // the wavefronts' maxima, normalisers and sums meet in LDS as [wavefront][head][sums, maximum, normaliser]
    float* const meet = reinterpret_cast<float*>(bf_lds);
    const float total = sum_half32(sum_row16(row.sum));
    if (r < group) {
        float* const mine = meet + (static_cast<size_t>(wave) * group + r) * VROW;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<bf_f32x4*>(mine + 16 * dt + 4 * quad) = row.acc[dt];
        if (quad == 0) {
            mine[V] = row.top;
            mine[V + 1] = total;
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < group * V; e += WAVES * CELEG_WAVE) {
        const int head = e / V, d = e % V;
        const float* const from = meet + static_cast<size_t>(head) * VROW;
        float top = -INFINITY, sum = 0.f, norm = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) top = fmaxf(top, from[static_cast<size_t>(w) * group * VROW + V]);
        const float base = top == -INFINITY ? 0.f : top;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float* const theirs = from + static_cast<size_t>(w) * group * VROW;
            const float f = bf_exp2(theirs[V] - base);
            norm = fmaf(theirs[V + 1], f, norm);
            sum = fmaf(theirs[d], f, sum);
        }
        if (p.parts_out) {
            float* const to = p.parts_out + (((static_cast<size_t>(t) * a.kv_heads + kvh) * p.parts + blockIdx.z) * group + head) * (V + 2);
            to[d] = sum;
            if (d == 0) {
                to[V] = top;
                to[V + 1] = norm;
            }
            continue;
        }
        if (!FULL && d >= vd) continue;
        const size_t at = static_cast<size_t>(kvh * group + head) * vd + d;
        const float g = a.gate ? bf_sigmoid(to_float(a.gate[static_cast<size_t>(t) * a.ldg + at])) : 1.0f;
        a.out[static_cast<size_t>(t) * a.ldo + at] = from_float<bf16>(sum / norm * g);
    }
}

// The parts of the kernel above joined in their order, a thread a value, all parts asked for at once.
__global__ __launch_bounds__(256) void biased_attention_join_kernel(const float* __restrict__ in, const bf16* __restrict__ gate,
                                                                    bf16* __restrict__ out, const int parts, const int ldg, const int ldo,
                                                                    const int vd, const int v_pad, const int group, const int q_heads) {
    const int t = blockIdx.y, e = blockIdx.x * 256 + threadIdx.x;
    if (e >= q_heads * vd) return;
    const int head = e / vd, d = e - head * vd, kvh = head / group, row = v_pad + 2;
    const float* const mine = in + ((static_cast<size_t>(t) * q_heads + static_cast<size_t>(kvh) * group) * parts + (head - kvh * group)) * row;
    const float g = gate ? to_float(gate[static_cast<size_t>(t) * ldg + e]) : 0.f;
    float sums[BF_MAX_PARTS], tops[BF_MAX_PARTS], norms[BF_MAX_PARTS];
#pragma unroll
    for (int i = 0; i < BF_MAX_PARTS; ++i) {
        const float* const part = mine + static_cast<size_t>(min(i, parts - 1)) * group * row;
        sums[i] = part[d];
        tops[i] = part[v_pad];
        norms[i] = part[v_pad + 1];
    }
    float top = tops[0];
#pragma unroll
    for (int i = 1; i < BF_MAX_PARTS; ++i) top = fmaxf(top, tops[i]);       // (finite: the row's own key is in one of them)
    float sum = 0.f, norm = 0.f;
#pragma unroll
    for (int i = 0; i < BF_MAX_PARTS; ++i) {
        const float f = i < parts ? bf_exp2(tops[i] - top) : 0.f;
        sum = fmaf(sums[i], f, sum);
        norm = fmaf(norms[i], f, norm);
    }
    out[static_cast<size_t>(t) * ldo + e] = from_float<bf16>(sum / norm * (gate ? bf_sigmoid(g) : 1.0f));
}

template <int D, int V, bool FULL>
int bf_launch_single(int n_tokens, const BfArgs& a, const BfSingle& p, hipStream_t stream) {
    const int group = a.q_heads / a.kv_heads;
    const size_t lds = static_cast<size_t>(BF_SINGLE_WAVES) * group * (V + 4) * sizeof(float);
    auto kernel = &biased_attention_single_kernel<D, V, FULL>;
    static bool raised = false;              // (16 heads of 128: 68 KB)
    if (lds > 48 * 1024 && !raised) {
        hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
        if (err != hipSuccess) return static_cast<int>(err);
        raised = true;
    }
    hipLaunchKernelGGL(kernel, dim3(n_tokens, a.kv_heads, p.parts), dim3(BF_SINGLE_WAVES * CELEG_WAVE), lds, stream, a, p);
    if (p.parts_out)
        hipLaunchKernelGGL(biased_attention_join_kernel, dim3((a.q_heads * a.vd + 255) / 256, n_tokens), dim3(256), 0, stream, p.parts_out,
                           a.gate, a.out, p.parts, a.ldg, a.ldo, a.vd, V, group, a.q_heads);
    return CELEG_LAUNCH_RESULT();
}

constexpr int bf_block_bytes(int d, int v) { return (BF_KEYS * (d + 8) + v * (BF_KEYS + 8)) * 2; }
// single tiles: eight wavefronts share out the key blocks where their staging areas fit LDS
constexpr int bf_tile_waves(int d, int v) { return 8 * bf_block_bytes(d, v) <= 160 * 1024 ? 8 : BF_WAVES; }

template <int D, int V, bool FULL>
int bf_launch_full(int form, int max_tiles, const BfArgs& a, const BfSingle& single, hipStream_t stream) {
    if (form == 2) return bf_launch_single<D, V, FULL>(max_tiles, a, single, stream);
    if (form == 1) {
        dim3 grid(max_tiles, a.q_heads), block(BF_WAVES * CELEG_WAVE);
        hipLaunchKernelGGL((biased_attention_rows_kernel<D, V, FULL>), grid, block, 2 * bf_block_bytes(D, V), stream, a);
    } else {
        constexpr int WAVES = bf_tile_waves(D, V);
        dim3 grid(max_tiles, a.q_heads), block(WAVES * CELEG_WAVE);
        hipLaunchKernelGGL((biased_attention_tile_kernel<D, V, WAVES, FULL>), grid, block, WAVES * bf_block_bytes(D, V), stream, a);
    }
    return CELEG_LAUNCH_RESULT();
}
template <int D, int V>
int bf_launch(int form, int max_tiles, const BfArgs& a, const BfSingle& p, hipStream_t stream) {
    return a.kd == D && a.vd == V ? bf_launch_full<D, V, true>(form, max_tiles, a, p, stream) : bf_launch_full<D, V, false>(form, max_tiles, a, p, stream);
}

template <int D>
int bf_launch_v(int v_dim, int form, int max_tiles, const BfArgs& a, const BfSingle& p, hipStream_t stream) {
    switch ((v_dim + 31) / 32) {
        case 1: return bf_launch<D, 32>(form, max_tiles, a, p, stream);
        case 2: return bf_launch<D, 64>(form, max_tiles, a, p, stream);
        case 3: return bf_launch<D, 96>(form, max_tiles, a, p, stream);
        default: return bf_launch<D, 128>(form, max_tiles, a, p, stream);
    }
}

}  // namespace

// sizes of keys and values a head that the matrix-core kernels take
extern "C" int celeg_biased_attention_fast_ok(int head_dim, int v_dim) {
    return head_dim > 0 && head_dim <= 128 && head_dim % 8 == 0 && v_dim > 0 && v_dim <= 128 && v_dim % 4 == 0;
}

// How many workgroups share a key/value head's keys; keys: the most that a row may see.  With the second kernel a call
// of 4 requests over 8 heads of 64 takes 7.2 us at 300 keys and 8.2 at 1,500, without parts 6.3 and 16.7 (16-row tiles a query
// head: 7.4 and 16.9); of 10 requests 11.3 and 16.9 at 1,500, of 32 29 and 28 (42).  So, beyond 512 keys: parts of eight
// wavefronts with a unit of 32 keys each, up to eight of them, where 512 workgroups hold four at least; else none.
extern "C" int celeg_biased_attention_parts(int n_tokens, int kv_heads, int keys) {
    if (keys <= 512) return 1;
    const int useful = (keys + BF_UNIT * BF_SINGLE_WAVES - 1) / (BF_UNIT * BF_SINGLE_WAVES);
    const int parts = std::min({std::max(useful, 4), BF_MAX_PARTS, 512 / std::max(n_tokens * kv_heads, 1)});
    return parts < 4 ? 1 : parts;
}
extern "C" long long celeg_biased_attention_parts_floats(int q_heads, int v_dim, int parts) {
    return static_cast<long long>(q_heads) * ((v_dim + 31) / 32 * 32 + 2) * parts;
}

// bfloat16 on the matrix cores; form 0: tiles of 16 rows whose key blocks the wavefronts share out
// (single tokens, short portions), form 1: tiles of 64 rows that stage a key block once for four
// wavefronts (portions of prompts); max_tiles: an upper bound on the step's tiles (sum over
// requests of ceil(rows / 16 or 64)); form 2: single tokens, max_tiles rows of one token a request with their positions
// and slots, up to 16 query heads a key/value head (parts > 1: parts_out 32-bit, celeg_biased_attention_parts_floats
// of them a row); pages of a power of two of at least 8 tokens; q, gate and out
// rows start at multiples of 16, 8 and 8 bytes
extern "C" int celeg_biased_attention_fast(int form, const void* q, int ldq, const void* k_pool, const void* v_pool, const int* table,
                                           int table_stride, const int* cu_seqlens, const int* seq_slot, const int* seq_start, int n_seqs,
                                           int max_tiles, const float* r1, const float* r2, const void* gate, int ldg, void* out, int ldo,
                                           int q_heads, int kv_heads, int head_dim, int v_dim, int page_tokens, int n_layers, int layer,
                                           float scale, float coef, int every, int window, int keep_first, int sink_one,
                                           const float* sink, float softcap, const int* positions, const int* token_slot,
                                           float* parts_out, int parts, hipStream_t stream) {
    if (max_tiles <= 0 || n_seqs <= 0) return 0;
    if (form == 2 && (!positions || !token_slot || q_heads / kv_heads > 16 || parts < 1 || parts > BF_MAX_PARTS || (parts > 1 && !parts_out)))
        return static_cast<int>(hipErrorInvalidValue);
    if (!celeg_biased_attention_fast_ok(head_dim, v_dim) || q_heads % kv_heads || page_tokens < 8 || (page_tokens & (page_tokens - 1)) ||
        ldq % 8 || ldo % 4 || (gate && ldg % 4) || (r1 == nullptr) != (r2 == nullptr))
        return static_cast<int>(hipErrorInvalidValue);
    BfArgs a;
    a.q = static_cast<const bf16*>(q);
    a.k_pool = static_cast<const bf16*>(k_pool);
    a.v_pool = static_cast<const bf16*>(v_pool);
    a.table = table;
    a.cu_seqlens = cu_seqlens;
    a.seq_slot = seq_slot;
    a.seq_start = seq_start;
    a.r1 = r1;
    a.r2 = r2;
    a.gate = static_cast<const bf16*>(gate);
    a.out = static_cast<bf16*>(out);
    a.ldq = ldq;
    a.ldg = ldg;
    a.ldo = ldo;
    a.table_stride = table_stride;
    a.n_seqs = n_seqs;
    a.q_heads = q_heads;
    a.kv_heads = kv_heads;
    a.page_tokens = page_tokens;
    a.n_layers = n_layers;
    a.layer = layer;
    a.every = every;
    a.window = window;
    a.keep_first = window > 0 ? keep_first : 0;
    a.sink_one = sink_one;
    a.sink = sink;
    a.softcap = softcap;
    a.kd = head_dim;
    a.vd = v_dim;
    a.scale = scale;
    a.coef = coef;
    BfSingle single;
    single.positions = positions;
    single.token_slot = token_slot;
    single.parts = parts;
    single.parts_out = parts > 1 ? parts_out : nullptr;
    switch ((head_dim + 31) / 32) {
        case 1: return bf_launch_v<32>(v_dim, form, max_tiles, a, single, stream);
        case 2: return bf_launch_v<64>(v_dim, form, max_tiles, a, single, stream);
        case 3: return bf_launch_v<96>(v_dim, form, max_tiles, a, single, stream);
        default: return bf_launch_v<128>(v_dim, form, max_tiles, a, single, stream);
    }
}
