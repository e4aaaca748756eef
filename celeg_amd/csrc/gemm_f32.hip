// True 32-bit matrix product for the 32-bit path: Y[M,N] = X[M,K] W[N,K]^T (+ bias).
// No reduced-precision matrix mode: the matrix cores' 32-bit instruction (16x16x4).  Every output
// element is summed in the same order whatever M, the tile or the batch is, so a row's products do
// not depend on how rows were batched (nor does a norm folded into them, below; of the norm's own kernels the one for 64 and
// more rows of up to 1,024 values adds its squares in another order): k in segments of 128, a segment as a chain of 32 instructions
// (instruction i of a piece of 16 takes the values i, 4 + i, 8 + i and 12 + i), then the segments'
// sums in order.
// The reference's projections: y = x W^T, weights [out, in] row-major
// (src/model/weight_plan.cpp:82-130).
//
// A workgroup owns a tile of 16 RT rows x 16 CT columns; its wavefronts take the segments in turn and
// leave their sums in LDS, where the workgroup adds them in order.  Few rows are bound by reading W: up to 16
// columns a workgroup, up to 16 wavefronts that each ask for 8 KiB at once, so
// that even a 1024 x 1024 matrix is asked for by 512 wavefronts in one trip to memory.  Many rows are bound
// by the matrix cores: staged tiles, further down; this kernel where those are too few for the CUs.
// Measured in a chain over different matrices (before: 64 x 64 tiles of vector instructions, k in order,
// 137 us for products of up to 64 rows and few columns with K = 1,024): 2 rows, 1024 x 1024 3.3 us, 3072 x 1024
// 5.5 us, 1024 x 4608 7.2 us (before 613), 65536 x 1024 54 us (5.0 TB/s; before 247); 64 rows, 3072 x 1024
// 13.7 us; 424 rows, 1024 x 4608 64 us (before the order of its loads was pinned 74).  Error against 64 bits 2.1e-7 of the result (2-norm), before 3 times that.
#include "common.h"

typedef float f32x4_t __attribute__((ext_vector_type(4)));

#define F32_SEGMENT 128
#define F32_PIECES (F32_SEGMENT / 16)

// GROUP: pieces of 16 values of k that are asked for together.  VEC: rows of X and W lie on 16 bytes
// and K is a multiple of 4; the same sums in the same order without it.
// WAVES: wavefronts that a SIMD is to hold.
template <int RT, int CT, int GROUP, int MAX_THREADS, bool VEC, int WAVES>
__global__ __launch_bounds__(MAX_THREADS, WAVES) void gemm_f32_kernel(
    const float* __restrict__ X, int ldx, const float* __restrict__ W, int ldw,
    const float* __restrict__ bias, float* __restrict__ Y, int ldy, int M, int N, int K, int wide_store) {
    constexpr int TILES = RT * CT;
    constexpr int ITEMS = TILES > 8 ? TILES / 4 : 1;      // sums of four a thread: at least min(TILES, 8) wavefronts, 4 if TILES > 8
    extern __shared__ f32x4_t parts[];                    // [wavefront][tile][lane]
    const int wave = threadIdx.x / CELEG_WAVE, lane = threadIdx.x % CELEG_WAVE;
    const int n_waves = blockDim.x / CELEG_WAVE;
    const int qd = lane >> 4, r16 = lane & 15;
    const int row0 = blockIdx.y * (16 * RT), col0 = blockIdx.x * (16 * CT);
    // rows and columns past the end repeat the last one: an output depends on its own row and column only
    const float* x_row[RT];
    const float* w_row[CT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) x_row[rt] = X + static_cast<size_t>(min(row0 + rt * 16 + r16, M - 1)) * ldx;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) w_row[ct] = W + static_cast<size_t>(min(col0 + ct * 16 + r16, N - 1)) * ldw;

    auto four = [&](const float* row, int k, bool whole) __attribute__((always_inline)) {
        f32x4_t v = {0.f, 0.f, 0.f, 0.f};
        if (VEC) {
            if (whole || k < K) v = *reinterpret_cast<const f32x4_t*>(row + k);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (whole || k + i < K) v[i] = row[k + i];
        }
        return v;
    };
    auto load = [&](int k0, bool whole, f32x4_t (&wv)[CT][GROUP], f32x4_t (&xv)[RT][GROUP]) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < GROUP; ++s) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) wv[ct][s] = four(w_row[ct], k0 + 16 * s + 4 * qd, whole);
        }
#pragma unroll
        for (int s = 0; s < GROUP; ++s) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) xv[rt][s] = four(x_row[rt], k0 + 16 * s + 4 * qd, whole);
        }
    };
    f32x4_t acc[CT][RT];
    auto multiply = [&](const f32x4_t (&wv)[CT][GROUP], const f32x4_t (&xv)[RT][GROUP]) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < GROUP; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt)
                        acc[ct][rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[ct][s][i], xv[rt][s][i], acc[ct][rt], 0, 0, 0);
    };
    auto segment = [&](int k0, bool whole) __attribute__((always_inline)) {
        f32x4_t w0[CT][GROUP], x0[RT][GROUP];
        load(k0, whole, w0, x0);
        if (GROUP == F32_PIECES) {
            multiply(w0, x0);
            return;
        }
        f32x4_t w1[CT][GROUP], x1[RT][GROUP];
#pragma unroll
        for (int g = 0; g < F32_PIECES / GROUP; g += 2) {
            // (the order pinned: left alone the compiler asks for a group right ahead of the products that use it.  A value at a
            // time that is the better order: 424 x 1,024, K = 1,023 19.0 us, pinned 20.6; 200 x 3,072 34.7, 38.7)
            load(k0 + (g + 1) * 16 * GROUP, whole, w1, x1);
            if (VEC && CT > 1) __builtin_amdgcn_sched_barrier(0);
            multiply(w0, x0);
            if (VEC && CT > 1) __builtin_amdgcn_sched_barrier(0);
            if (g + 2 < F32_PIECES / GROUP) load(k0 + (g + 2) * 16 * GROUP, whole, w0, x0);
            if (VEC && CT > 1) __builtin_amdgcn_sched_barrier(0);
            multiply(w1, x1);
            if (VEC && CT > 1) __builtin_amdgcn_sched_barrier(0);
        }
    };

    f32x4_t total[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) total[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int segments = (K + F32_SEGMENT - 1) / F32_SEGMENT;
    for (int first = 0; first < segments; first += n_waves) {
        const int k0 = (first + wave) * F32_SEGMENT;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) acc[ct][rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (k0 + F32_SEGMENT <= K) segment(k0, true);
        else if (k0 < K) segment(k0, false);
        if (first) __syncthreads();                       // the sums before have been read
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) parts[(wave * TILES + ct * RT + rt) * CELEG_WAVE + lane] = acc[ct][rt];
        __syncthreads();
        const int n = min(n_waves, segments - first);
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const int item = static_cast<int>(threadIdx.x) + j * static_cast<int>(blockDim.x);
            if (item < TILES * CELEG_WAVE)
                for (int w = 0; w < n; ++w) total[j] += parts[w * TILES * CELEG_WAVE + item];
        }
    }
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const int item = static_cast<int>(threadIdx.x) + j * static_cast<int>(blockDim.x);
        if (item >= TILES * CELEG_WAVE) continue;
        const int tile = item / CELEG_WAVE, l = item % CELEG_WAVE;
        const int row = row0 + (tile % RT) * 16 + (l & 15), col = col0 + (tile / RT) * 16 + 4 * (l >> 4);
        if (row >= M) continue;
        float* y = Y + static_cast<size_t>(row) * ldy + col;
        if (wide_store && col + 3 < N) {
            f32x4_t v = total[j];
            if (bias) v += f32x4_t{bias[col], bias[col + 1], bias[col + 2], bias[col + 3]};
            *reinterpret_cast<f32x4_t*>(y) = v;
            continue;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (col + r < N) y[r] = total[j][r] + (bias ? bias[col + r] : 0.f);
    }
}

// What surrounds a product of few rows, folded into it (a decode step is a chain of short kernels, each of
// which costs 1.7 us empty): in front the RMSNorm of its rows (every workgroup normalises them for itself while its
// weights are on their way), behind it the addition into the residual stream, SwiGLU of a gate and an up stream,
// or the double-gated short convolution of a B, a C and an x stream for one new token per request with its state
// update.  Streams: rows [s N, (s + 1) N) of W.  An output is computed from the same 32-bit sums by the same
// operations as where these are kernels of their own, the squares of a row in the order of its norm's kernel.
// Reference semantics: RMSNorm src/backend/cpu/kernels/elementwise.cpp:56-76, SwiGLU elementwise.cpp:101-119, short
// convolution src/backend/cpu/kernels/convolution.cpp:7-28.
enum { F32_STORE = 0, F32_RESIDUAL = 2, F32_SWIGLU = 3, F32_CONV = 4 };      // (the numbers of the bfloat16 products)
#define F32_MAX_TAPS 8
struct F32Tail {
    const float* norm_w;        // [K]
    float eps;
    int taps;
    const float* conv_w;        // [N, taps]
    const float* conv_b;        // optional [N]
    float* state;               // [slots, taps, N]
    size_t state_slot_stride;
    const int* seq_slot;        // [M]
};
template <int EPI> constexpr int f32_streams() { return EPI == F32_SWIGLU ? 2 : EPI == F32_CONV ? 3 : 1; }

// The products of up to 16 rows.  The 16 x 16 tile of the instruction is cut into G x G blocks: its rows are
// (segment g of G, column j of 16 / G) of W, its columns (segment g', row m of 16 / G) of X, so the blocks
// g = g' on the diagonal are G segments' sums of the same outputs and the others are dropped.  A workgroup
// then owns 16 / G columns (of all streams together), and a matrix of few columns (w2: 1,024) is spread over G times
// as many workgroups; a segment's sum is formed by the same instructions, so the outputs keep their bits.
// 2 rows: 1024 x 4608 7.2 us (on 16 columns a workgroup 14.8), 1024 x 1024 3.3 (4.5).
// (a norm's rows are whole in one round of at most 16 / G wavefronts, K <= 2,048: the more registers are left to each)
template <int G, bool VEC, int EPI, bool NORM>
__global__ __launch_bounds__(NORM ? 1024 / G : 1024) void gemm_f32_slices_kernel(
    const float* __restrict__ X, int ldx, const float* __restrict__ W, int ldw,
    const float* __restrict__ bias, float* __restrict__ Y, int ldy, int M, int N, int K, int wide_store, int n_waves, const F32Tail f) {
    constexpr int MP = 16 / G, ITEMS = MP * MP / 4;      // sums of four neighbouring columns of a row
    constexpr int NS = f32_streams<EPI>(), OWN = MP / NS;      // columns of a stream that the workgroup owns
    extern __shared__ f32x4_t parts[];                    // [segment of the round][item], then the norm's weight, [row][256 values], [wavefront][piece][lane] and [row][column] floats
    const int wave = threadIdx.x / CELEG_WAVE, lane = threadIdx.x % CELEG_WAVE;
    // (n_waves comes beside the sizes: the launch's own count lies two lines behind the first arguments, a trip to memory of its
    // own: 2 rows, 3,072 x 1,024 4.90 us against 5.05)
    f32x4_t* const norm_w = parts + static_cast<size_t>(n_waves) * G * ITEMS;
    float* const row_squares = reinterpret_cast<float*>(norm_w + (NORM ? n_waves * CELEG_WAVE : 0));
    float* const chains = row_squares + (NORM ? 8 * MP : 0);
    float* const sums = chains + (NORM && G == 1 ? 8 * F32_PIECES * CELEG_WAVE : 0);
    const int qd = lane >> 4, r16 = lane & 15;
    const int col0 = blockIdx.x * OWN;
    const float* const x_row = X + static_cast<size_t>(min(r16 % MP, M - 1)) * ldx;
    const int tile_col = NS == 1 || r16 % MP < NS * OWN ? r16 % MP : 0;      // (what OWN x NS columns leave of the tile repeats the first)
    const float* const w_row = W + (static_cast<size_t>(tile_col / OWN) * N + min(col0 + tile_col % OWN, N - 1)) * ldw;
    // this lane's sums: row (lane % MP) and columns 4 (quad in its block) .. + 3, of segment `of`
    const int of = qd / (MP / 4), item = (qd % (MP / 4)) * MP + lane % MP;
    const bool on_diagonal = r16 / MP == of;
    const int segments = (K + F32_SEGMENT - 1) / F32_SEGMENT;
    f32x4_t total = {0.f, 0.f, 0.f, 0.f}, old = {0.f, 0.f, 0.f, 0.f};

    // ---- what the end needs from memory, asked for ahead of the products
    const int row = threadIdx.x % MP, col = col0 + 4 * (threadIdx.x / MP);      // of the item this thread adds up
    if (EPI == F32_RESIDUAL && threadIdx.x < ITEMS && row < M) {
        const float* y = Y + static_cast<size_t>(row) * ldy + col;
        if (wide_store && col + 3 < N) old = *reinterpret_cast<const f32x4_t*>(y);
        else
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (col + r < N) old[r] = y[r];
    }
    const int out_row = threadIdx.x / OWN, out_col = col0 + threadIdx.x % OWN;   // of the output this thread finishes (SwiGLU, convolution)
    const bool finishes = NS > 1 && threadIdx.x < MP * OWN && out_row < M && out_col < N;
    float taps[EPI == F32_CONV ? F32_MAX_TAPS : 1], state[EPI == F32_CONV ? F32_MAX_TAPS - 1 : 1], conv_b = 0.f;
    float* state_at = nullptr;
    const auto fetch_conv = [&]() __attribute__((always_inline)) {
        if (!finishes) return;
        state_at = f.state + static_cast<size_t>(f.seq_slot[out_row]) * f.state_slot_stride + out_col;
#pragma unroll
        for (int i = 0; i < F32_MAX_TAPS; ++i) taps[i] = f.conv_w[static_cast<size_t>(out_col) * f.taps + min(i, f.taps - 1)];
#pragma unroll
        for (int i = 0; i < F32_MAX_TAPS - 1; ++i) state[i] = state_at[static_cast<size_t>(min(i + 1, f.taps - 1)) * N];
        if (f.conv_b) conv_b = f.conv_b[out_col];
    };
    if constexpr (EPI == F32_CONV && G > 1) fetch_conv();      // (16 wavefronts have no registers to hold them)

    for (int first = 0; first < segments; first += n_waves * G) {
        const int mine = first + wave * G;                // this wavefront's segments: G of them from here
        const int k0 = (mine + r16 / MP) * F32_SEGMENT + 4 * qd;
        f32x4_t wv[F32_PIECES], xv[F32_PIECES], nw = {0.f, 0.f, 0.f, 0.f};
        const auto load_x = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < F32_PIECES; ++s) xv[s] = *reinterpret_cast<const f32x4_t*>(x_row + k0 + 16 * s);
        };
        // (the norm's weight goes by way of LDS, four values a thread, 256 a wavefront; held beside the operands, 32 registers)
        const auto load_norm = [&]() __attribute__((always_inline)) {
            if (4 * static_cast<int>(threadIdx.x) < K) nw = *reinterpret_cast<const f32x4_t*>(f.norm_w + 4 * threadIdx.x);
        };
        if (VEC && (mine + G) * F32_SEGMENT <= K) {
            if constexpr (NORM) {       // (the rows first: their squares are added up while the weights are on their way)
                load_x();
                load_norm();
            }
#pragma unroll
            for (int s = 0; s < F32_PIECES; ++s) wv[s] = *reinterpret_cast<const f32x4_t*>(w_row + k0 + 16 * s);
            if constexpr (!NORM) load_x();
        } else {
            if constexpr (NORM) load_norm();
#pragma unroll
            for (int s = 0; s < F32_PIECES; ++s) {
                const int k = k0 + 16 * s;
                wv[s] = xv[s] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                if (VEC) {
                    if (k < K) {
                        wv[s] = *reinterpret_cast<const f32x4_t*>(w_row + k);
                        xv[s] = *reinterpret_cast<const f32x4_t*>(x_row + k);
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (k + i < K) {
                            wv[s][i] = w_row[k + i];
                            xv[s][i] = x_row[k + i];
                        }
                }
            }
        }
        if constexpr (NORM) {           // (one round: the launch sees to it)
            norm_w[threadIdx.x] = nw;
            // The squares in the order of rmsnorm_vec_kernel (up to 1,024 values its own bits): chains over four neighbouring values,
            // the 64 chains of 256 values as a tree (128 values apart, 64, .. down to 4), these sums one after the other.
            const auto chain = [&](int s) __attribute__((always_inline)) { return squares_of_four(xv[s][0], xv[s][1], xv[s][2], xv[s][3]); };
            const auto tree = [&](auto&& of) __attribute__((always_inline)) {
                const float even = (of(0) + of(4)) + (of(2) + of(6));
                return sum_row16(sum_half32(even + ((of(1) + of(5)) + (of(3) + of(7)))));
            };
            static_assert(G <= 2 && F32_PIECES == 8, "256 values are a wavefront's two segments or those of two neighbouring wavefronts");
            float squares = 0.f;
            if constexpr (G == 2) {
                squares = tree([&](int s) __attribute__((always_inline)) { const float v = chain(s); return v + lane_move<LANES_ROTATE_8>(v); });
            } else {
                float* const theirs = chains + (wave / 2) * F32_PIECES * CELEG_WAVE + lane;
                if (wave % 2)
#pragma unroll
                    for (int s = 0; s < F32_PIECES; ++s) theirs[s * CELEG_WAVE] = chain(s);
                __syncthreads();
                if (wave % 2 == 0) {
                    const bool there = wave + 1 < n_waves;
                    squares = tree([&](int s) __attribute__((always_inline)) { return chain(s) + (there ? theirs[s * CELEG_WAVE] : 0.f); });
                }
            }
            constexpr int SUMS = 16 * F32_SEGMENT / 256;
            if (qd == 0 && (G == 2 ? r16 < MP : wave % 2 == 0)) row_squares[(r16 % MP) * SUMS + wave * G / 2] = squares;
            __syncthreads();
            float all = 0.f;
#pragma unroll
            for (int g = 0; g < SUMS; ++g)
                if (g * 256 < K) all += row_squares[(r16 % MP) * SUMS + g];
            const float inv = 1.0f / sqrtf(all / static_cast<float>(K) + f.eps);
#pragma unroll
            for (int s = 0; s < F32_PIECES; ++s) {
                const f32x4_t w4 = norm_w[k0 / 4 + 4 * s];
#pragma unroll
                for (int i = 0; i < 4; ++i) xv[s][i] = xv[s][i] * inv * w4[i];
            }
        }
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < F32_PIECES; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[s][i], xv[s][i], acc, 0, 0, 0);
        if (first) __syncthreads();                       // the sums before have been read
        if (on_diagonal) parts[(wave * G + of) * ITEMS + item] = acc;
        __syncthreads();
        const int n = min(n_waves * G, segments - first);
        if (threadIdx.x < ITEMS)
            for (int g = 0; g < n; ++g) total += parts[g * ITEMS + threadIdx.x];
    }
    if constexpr (NS > 1) {
        if constexpr (EPI == F32_CONV && G == 1) fetch_conv();
        if (threadIdx.x < ITEMS)
            *reinterpret_cast<f32x4_t*>(sums + row * MP + 4 * (threadIdx.x / MP)) = total;
        __syncthreads();
        if (!finishes) return;
        float v[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s)
            v[s] = sums[out_row * MP + s * OWN + threadIdx.x % OWN] + (bias ? bias[static_cast<size_t>(s) * N + out_col] : 0.f);
        float* const y = Y + static_cast<size_t>(out_row) * ldy + out_col;
        if constexpr (EPI == F32_SWIGLU) {
            *y = (v[0] / (1.0f + expf(-v[0]))) * v[1];
        } else {
            const float bx = v[0] * v[2];
            float conv = 0.f, last_tap = 0.f;
#pragma unroll
            for (int tap = 0; tap < F32_MAX_TAPS - 1; ++tap)
                if (tap + 1 < f.taps) {
                    conv = fmaf(taps[tap], state[tap], conv);
                    state_at[static_cast<size_t>(tap) * N] = state[tap];         // shift by one position
                }
#pragma unroll
            for (int tap = 0; tap < F32_MAX_TAPS; ++tap)
                if (tap == f.taps - 1) last_tap = taps[tap];
            conv = fmaf(last_tap, bx, conv);
            state_at[static_cast<size_t>(f.taps - 1) * N] = bx;
            *y = v[1] * (conv + conv_b);
        }
        return;
    }
    if (threadIdx.x >= ITEMS || row >= M) return;
    float* y = Y + static_cast<size_t>(row) * ldy + col;
    if (wide_store && col + 3 < N) {
        if (bias) total += f32x4_t{bias[col], bias[col + 1], bias[col + 2], bias[col + 3]};
        if (EPI == F32_RESIDUAL) total += old;
        *reinterpret_cast<f32x4_t*>(y) = total;
        return;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (col + r < N) {
            const float v = total[r] + (bias ? bias[col + r] : 0.f);
            y[r] = EPI == F32_RESIDUAL ? old[r] + v : v;
        }
}

template <int G, int EPI = F32_STORE, bool NORM = false>
static int launch_f32_slices(const float* X, int ldx, const float* W, int ldw, const float* bias, float* Y, int ldy,
                             int M, int N, int K, hipStream_t stream, const F32Tail& tail = F32Tail{}) {
    const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool vec = K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && aligned(X) && aligned(W);
    const int wide_store = ldy % 4 == 0 && aligned(Y);
    constexpr int MP = 16 / G, OWN = MP / f32_streams<EPI>();
    const int groups = ((K + F32_SEGMENT - 1) / F32_SEGMENT + G - 1) / G;
    const int rounds = (groups + 15) / 16, waves = (groups + rounds - 1) / rounds;     // as even as it goes: 36 are 3 rounds of 12
    // (all of a row is needed for its norm, and the end of a product with two or three streams takes a thread an output)
    if ((NORM && (rounds > 1 || !vec || !aligned(tail.norm_w))) || (EPI != F32_STORE && !vec)) return static_cast<int>(hipErrorInvalidValue);
    const int threads = max(waves * CELEG_WAVE, f32_streams<EPI>() > 1 ? (MP * OWN + CELEG_WAVE - 1) / CELEG_WAVE * CELEG_WAVE : 0);
    const dim3 grid((N + OWN - 1) / OWN), block(threads);
    const int waves_run = threads / CELEG_WAVE;
    const size_t lds = static_cast<size_t>(waves_run) * G * (MP * MP / 4) * sizeof(f32x4_t) + (NORM ? (4 * threads + 8 * MP + (G == 1 ? 8 * F32_PIECES * CELEG_WAVE : 0)) * sizeof(float) : 0) +
                       (f32_streams<EPI>() > 1 ? MP * MP * sizeof(float) : 0);
    if constexpr (EPI == F32_STORE && !NORM) {
        auto kernel = vec ? &gemm_f32_slices_kernel<G, true, EPI, NORM> : &gemm_f32_slices_kernel<G, false, EPI, NORM>;
        hipLaunchKernelGGL(kernel, grid, block, lds, stream, X, ldx, W, ldw, bias, Y, ldy, M, N, K, wide_store, waves_run, tail);
    } else {
        hipLaunchKernelGGL((gemm_f32_slices_kernel<G, true, EPI, NORM>), grid, block, lds, stream, X, ldx, W, ldw, bias, Y, ldy, M, N, K,
                           wide_store, waves_run, tail);
    }
    return CELEG_LAUNCH_RESULT();
}

template <int RT, int CT, int GROUP, int MAX_THREADS, int WAVES = 2>
static int launch_f32(const float* X, int ldx, const float* W, int ldw, const float* bias, float* Y, int ldy,
                      int M, int N, int K, hipStream_t stream) {
    const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool vec = K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && aligned(X) && aligned(W);
    const int wide_store = ldy % 4 == 0 && aligned(Y);
    constexpr int most = MAX_THREADS / CELEG_WAVE, least = RT * CT > 8 ? 4 : (RT * CT > 4 ? RT * CT : 4);
    const int segments = (K + F32_SEGMENT - 1) / F32_SEGMENT;
    const int rounds = (segments + most - 1) / most;      // as even as it goes: 36 segments are 3 rounds of 12
    const int waves = max(least, (segments + rounds - 1) / rounds);
    const dim3 grid((N + 16 * CT - 1) / (16 * CT), (M + 16 * RT - 1) / (16 * RT)), block(waves * CELEG_WAVE);
    const size_t lds = static_cast<size_t>(waves) * RT * CT * CELEG_WAVE * sizeof(f32x4_t);
    // (64 x 64 tiles are for rows that cannot be read 16 bytes at a time)
    if constexpr (RT * CT <= 8) {
        if (vec) {
            hipLaunchKernelGGL((gemm_f32_kernel<RT, CT, GROUP, MAX_THREADS, true, WAVES>), grid, block, lds, stream, X, ldx, W, ldw, bias, Y, ldy, M, N, K, wide_store);
            return CELEG_LAUNCH_RESULT();
        }
    }
    hipLaunchKernelGGL((gemm_f32_kernel<RT, CT, GROUP, MAX_THREADS, false, WAVES>), grid, block, lds, stream, X, ldx, W, ldw, bias, Y, ldy, M, N, K, wide_store);
    return CELEG_LAUNCH_RESULT();
}

// The products of many rows over a short K whose rows cannot be read 16 bytes at a time.  A wavefront has a tile of
// 16 RT x 16 CT outputs to itself and goes through the segments one after the other, each summed and added as above, so
// the outputs have the same bits; there is nothing to join, and a last segment that is not whole costs what it has.
// 2,048 x 4,096, K = 33 28 us (on the kernel above, most of whose wavefronts then wait, 128).
template <int RT, int CT>
__global__ __launch_bounds__(256) void gemm_f32_short_kernel(
    const float* __restrict__ X, int ldx, const float* __restrict__ W, int ldw,
    const float* __restrict__ bias, float* __restrict__ Y, int ldy, int M, int N, int K, int wide_store) {
    constexpr int GROUP = F32_PIECES / 2;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / CELEG_WAVE), lane = threadIdx.x % CELEG_WAVE;
    const int qd = lane >> 4, r16 = lane & 15;
    const int row0 = blockIdx.y * (16 * RT), col0 = (blockIdx.x * 4 + wave) * (16 * CT);
    if (col0 >= N) return;
    const float* x_row[RT];
    const float* w_row[CT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) x_row[rt] = X + static_cast<size_t>(min(row0 + rt * 16 + r16, M - 1)) * ldx;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) w_row[ct] = W + static_cast<size_t>(min(col0 + ct * 16 + r16, N - 1)) * ldw;
    auto four = [&](const float* row, int k) __attribute__((always_inline)) {
        f32x4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (k + i < K) v[i] = row[k + i];
        return v;
    };
    f32x4_t acc[CT][RT], total[CT][RT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) total[ct][rt] = acc[ct][rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < K; k0 += 16 * GROUP) {
        f32x4_t wv[CT][GROUP], xv[RT][GROUP];
#pragma unroll
        for (int s = 0; s < GROUP; ++s) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) wv[ct][s] = four(w_row[ct], k0 + 16 * s + 4 * qd);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) xv[rt][s] = four(x_row[rt], k0 + 16 * s + 4 * qd);
        }
#pragma unroll
        for (int s = 0; s < GROUP; ++s) {
            if (k0 + 16 * s >= K) break;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt)
                        acc[ct][rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[ct][s][i], xv[rt][s][i], acc[ct][rt], 0, 0, 0);
        }
        const int next = k0 + 16 * GROUP;
        if (next % F32_SEGMENT == 0 || next >= K) {        // the segment is done
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    total[ct][rt] += acc[ct][rt];
                    acc[ct][rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                }
        }
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int row = row0 + rt * 16 + r16;
        if (row >= M) continue;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const int col = col0 + ct * 16 + 4 * qd;
            float* y = Y + static_cast<size_t>(row) * ldy + col;
            f32x4_t v = total[ct][rt];
            if (wide_store && col + 3 < N) {
                if (bias) v += f32x4_t{bias[col], bias[col + 1], bias[col + 2], bias[col + 3]};
                *reinterpret_cast<f32x4_t*>(y) = v;
                continue;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (col + r < N) y[r] = v[r] + (bias ? bias[col + r] : 0.f);
        }
    }
}

template <int RT, int CT>
static int launch_f32_short(const float* X, int ldx, const float* W, int ldw, const float* bias, float* Y, int ldy,
                            int M, int N, int K, hipStream_t stream) {
    const int wide_store = ldy % 4 == 0 && (reinterpret_cast<uintptr_t>(Y) & 15) == 0;
    const dim3 grid((N + 64 * CT - 1) / (64 * CT), (M + 16 * RT - 1) / (16 * RT)), block(4 * CELEG_WAVE);
    hipLaunchKernelGGL((gemm_f32_short_kernel<RT, CT>), grid, block, 0, stream, X, ldx, W, ldw, bias, Y, ldy, M, N, K, wide_store);
    return CELEG_LAUNCH_RESULT();
}

// blocks of 4 or 8 columns while tiles of 16 would leave compute units without a second workgroup
static int f32_slices_of(int M, int weight_rows) { return weight_rows >= 512 * 16 || M > 8 ? 1 : M > 4 ? 2 : 4; }

// Up to 16 rows with what surrounds them (epi: the numbers above; N: columns of a stream; norm_w null: none).  X, W and
// norm_w on 16 bytes, ldx, ldw and K multiples of 4; with a norm K up to 2,048.
extern "C" int celeg_gemm_f32_fused(const float* X, int ldx, const float* W, int ldw, const float* bias, float* Y, int ldy, int M,
                                    int N, int K, int epi, const float* norm_w, float eps, const float* conv_w, const float* conv_b,
                                    float* state, size_t state_slot_stride, const int* seq_slot, int taps, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 16 || K <= 0 || (norm_w && K > 16 * F32_SEGMENT) ||
        (epi == F32_CONV && (taps < 1 || taps > F32_MAX_TAPS || !conv_w || !state || !seq_slot)))
        return static_cast<int>(hipErrorInvalidValue);
    F32Tail f{norm_w, eps, taps, conv_w, conv_b, state, state_slot_stride, seq_slot};
#define F32_FUSED(G, EPI, NORM) launch_f32_slices<G, EPI, NORM>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream, f)
#define F32_NORMED(EPI) (!norm_w ? static_cast<int>(hipErrorInvalidValue) : M > 8 ? F32_FUSED(1, EPI, true) : F32_FUSED(2, EPI, true))
    // (behind a norm blocks of 8 columns up to 8 rows, a wavefront two segments, the halves of 256 values: with the norm's weight still
    // in registers 2 rows by 1,024 took, w1 with w3 12.7 us, in_proj with the convolution 7.2, q/k/v 5.8; blocks of 16 columns 15.8, 8.4
    // and 7.8, of 4 12.4, 7.6 and 6.1; 4 rows 13.3, 7.5, 5.9; 15.9, 8.6, 7.9; 13.9, 8.2, 6.3.  By way of LDS w1 with w3 11.7.)
    switch (epi) {
        case F32_STORE: return F32_NORMED(F32_STORE);
        case F32_SWIGLU: return F32_NORMED(F32_SWIGLU);
        case F32_CONV: return F32_NORMED(F32_CONV);
        case F32_RESIDUAL: {
            if (norm_w) return static_cast<int>(hipErrorInvalidValue);
            const int g = f32_slices_of(M, N);
            return g == 4 ? F32_FUSED(4, F32_RESIDUAL, false) : g == 2 ? F32_FUSED(2, F32_RESIDUAL, false) : F32_FUSED(1, F32_RESIDUAL, false);
        }
        default: return static_cast<int>(hipErrorInvalidValue);
    }
#undef F32_NORMED
#undef F32_FUSED
}

// Products of many rows: a workgroup of four wavefronts (two by two) has all of k for a tile of BM x BN, the same sums in
// the same order.  The operands go through LDS, 32 values of k (a line of 128 bytes a row) at a time and three such steps deep: two
// are on their way while one is multiplied, so a wavefront waits once a step, for loads that it asked for two steps before,
// and an operand is read from the L2 once a tile instead of once a wavefront.  Straight from the caches (the kernel
// above, and one that kept all of k and read a piece ahead) the loads of rows 4 KiB apart met in the same channels:
// 55 to 82 TFLOP/s as soon as a SIMD had more than one wavefront.  Here the matrix cores are the bound: 2,048 rows, N = 9,216, K =
// 1,024 317 us (122 TFLOP/s of 153; before 564), N = 2,048 73 (117); 1,024 rows, N = 9,216 166 (286), N = 3,072 59
// (92); 424 rows, N = 9,216 75 (129), N = 3,072 34 (48); 200 rows, N = 9,216 46 (90); 2,048 rows, K = 256, N = 1,024 13.6 (23).
#define F32_STEP 32
#define F32_STEP_CHUNKS (F32_STEP / 4)

template <int N>
__device__ __forceinline__ void f32_wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int BM, int BN>
__global__ __launch_bounds__(256, 2) void gemm_f32_tile_kernel(
    const float* __restrict__ X, int ldx, const float* __restrict__ W, int ldw,
    const float* __restrict__ bias, float* __restrict__ Y, int ldy, int M, int N, int K, int wide_store) {
    constexpr int RT = BM / 32, CT = BN / 32, ROWS = BM + BN, LOADS = ROWS * F32_STEP_CHUNKS / 256, STAGES = 3;
    constexpr int STEPS_A_SEGMENT = F32_SEGMENT / F32_STEP;
    __shared__ __attribute__((aligned(128))) float stage[STAGES][ROWS * F32_STEP];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / CELEG_WAVE), lane = threadIdx.x % CELEG_WAVE;
    const int qd = lane >> 4, r16 = lane & 15;
    const int row0 = blockIdx.y * BM, col0 = blockIdx.x * BN;
    // chunk c of 16 bytes of a staged row lies at c ^ (row / 2 % 8): 16 lanes that read one chunk of 16 rows meet every bank once
    // (a thread's loads are of rows 32 apart: the same chunk; a chunk past the end of the row is the row's last one)
    const int my_chunk = (static_cast<int>(threadIdx.x) % F32_STEP_CHUNKS) ^ ((static_cast<int>(threadIdx.x) / (2 * F32_STEP_CHUNKS)) & 7);
    const float* src[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = (i * 256 + static_cast<int>(threadIdx.x)) / F32_STEP_CHUNKS;
        src[i] = row < BM ? X + static_cast<size_t>(min(row0 + row, M - 1)) * ldx : W + static_cast<size_t>(min(col0 + row - BM, N - 1)) * ldw;
    }
    auto issue = [&](int step) __attribute__((always_inline)) {
        float* to = stage[step % STAGES];
        const int k = min(step * F32_STEP + 4 * my_chunk, K - 4);
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + k),
                                             (__attribute__((address_space(3))) void*)(to + (i * 256 + wave * CELEG_WAVE) * 4), 16, 0, 0);
    };
    const int wr = (wave & 1) * (BM / 2), wc = (wave >> 1) * (BN / 2);
    f32x4_t acc[CT][RT], total[CT][RT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) total[ct][rt] = acc[ct][rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int steps = (K + F32_STEP - 1) / F32_STEP;
    auto multiply = [&](int step, bool whole) __attribute__((always_inline)) {
        const float* st = stage[step % STAGES];
#pragma unroll
        for (int s = 0; s < F32_STEP / 16; ++s) {
            const int chunk = 4 * s + qd, at = 4 * (chunk ^ ((r16 >> 1) & 7));
            f32x4_t x[RT], w[CT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) x[rt] = *reinterpret_cast<const f32x4_t*>(st + (wr + rt * 16 + r16) * F32_STEP + at);
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) w[ct] = *reinterpret_cast<const f32x4_t*>(st + (BM + wc + ct * 16 + r16) * F32_STEP + at);
            if (!whole) {
                const bool in = step * F32_STEP + 4 * chunk < K;
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[rt][i] = in ? x[rt][i] : 0.f;
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int i = 0; i < 4; ++i) w[ct][i] = in ? w[ct][i] : 0.f;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt)
                        acc[ct][rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[ct][i], x[rt][i], acc[ct][rt], 0, 0, 0);
        }
    };
    auto add_segment = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                total[ct][rt] += acc[ct][rt];
                acc[ct][rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            }
    };
    issue(0);
    if (steps > 1) issue(1);
    const int whole = K / F32_STEP;
    for (int step = 0; step < whole; ++step) {
        if (step + 1 < steps) f32_wait_loads<LOADS>();
        else f32_wait_loads<0>();
        __syncthreads();                                  // the step is here, and everyone has read the one before it
        if (step + 2 < steps) issue(step + 2);
        multiply(step, true);
        if ((step + 1) % STEPS_A_SEGMENT == 0) add_segment();
    }
    if (whole < steps) {
        f32_wait_loads<0>();
        __syncthreads();
        multiply(whole, false);
    }
    if (steps % STEPS_A_SEGMENT || whole < steps) add_segment();
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int row = row0 + wr + rt * 16 + r16;
        if (row >= M) continue;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const int col = col0 + wc + ct * 16 + 4 * qd;
            float* y = Y + static_cast<size_t>(row) * ldy + col;
            f32x4_t v = total[ct][rt];
            if (wide_store && col + 3 < N) {
                if (bias) v += f32x4_t{bias[col], bias[col + 1], bias[col + 2], bias[col + 3]};
                *reinterpret_cast<f32x4_t*>(y) = v;
                continue;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (col + r < N) y[r] = v[r] + (bias ? bias[col + r] : 0.f);
        }
    }
}

template <int BM, int BN>
static int launch_f32_tile(const float* X, int ldx, const float* W, int ldw, const float* bias, float* Y, int ldy,
                           int M, int N, int K, hipStream_t stream) {
    const int wide_store = ldy % 4 == 0 && (reinterpret_cast<uintptr_t>(Y) & 15) == 0;
    const dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM);
    hipLaunchKernelGGL((gemm_f32_tile_kernel<BM, BN>), grid, dim3(256), 0, stream, X, ldx, W, ldw, bias, Y, ldy, M, N, K, wide_store);
    return CELEG_LAUNCH_RESULT();
}

// The staged tile of a product whose rows lie on 16 bytes: 1 32 x 64, 2 64 x 64, 3 64 x 128, 0 none of them.
// Staged tiles once the smallest of them give every CU more than one, and below that where k is too short to be cut
// over eight wavefronts (200 rows, K = 1,024: N = 1,024 16.1 us against 15.9 cut, N = 3,072 24.4 against 30.3; N = 1,024,
// K = 4,608 89 against 64; K = 384, N = 2,048 7.9 against 8.5; 40 rows, K = 256 5.7 against 5.8, K = 384 7.6 against 6.8).  Cut
// products gain where rows are not whole lines apart (K % 32: other channels), staged ones pay a step for what is left of k, and
// columns that are stored one at a time: 33 to 64 rows, K = 160 4.1 against 4.9, K = 188 4.6 against 4.8, K = 196 5.0 against 4.75, K = 224
// 4.9 against 5.2, K = 252 5.4 against 4.8, N = 1,091, K = 160 5.1 against 5.5, K = 188 5.55 against 5.3, K = 256 6.35 against 5.85; 65 rows and more,
// K = 480 8.7 against 9.8, K = 496 9.2 against 8.3, K = 512 9.2 against 9.6.
// The tile by what a round of them over 256 CUs takes (in 0.1 us at K = 1,024, all in proportion to K: 64 x 128 tiles
// go two at a time through a CU): 424 rows, N = 9,216 75 us with 64 x 128, 78 with 64 x 64, 84 with 32 x 64;
// 424 rows, N = 3,072 42, 40 and 34; 1,024 rows, N = 9,216 179, 166 and 183.  (A grid has 65,535 rows of tiles.)
extern "C" int celeg_gemm_f32_staged_tile(int M, int N, int K) {
    const long long small = static_cast<long long>((M + 31) / 32) * ((N + 63) / 64);
    const bool lines = K % F32_STEP == 0, wide = N % 4 == 0;
    const bool few = M > 32 && (K <= 160 || (wide && (K <= 192 || (lines && K <= 2 * F32_SEGMENT))));
    const bool more = M > 64 && K < 8 * F32_SEGMENT && !(!lines && K > 15 * F32_STEP && K < 16 * F32_STEP);
    if (M <= 16 || !(small > 256 || few || more)) return 0;
    const auto rounds = [](long long m, long long n) { return (m * n + 255) / 256; };
    const long long c32 = 20 + 101 * rounds((M + 31) / 32, (N + 63) / 64), c64 = 40 + 185 * rounds((M + 63) / 64, (N + 63) / 64),
                    c128 = 70 + 350 * rounds((M + 63) / 64, (N + 127) / 128);
    return c128 < c64 && c128 < c32 ? 3 : c64 < c32 || M > 32 * 65535 ? 2 : 1;
}

extern "C" int celeg_gemm_f32(const float* X, int ldx, const float* W, int ldw, const float* bias,
                              float* Y, int ldy, int M, int N, int K, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0) return static_cast<int>(hipErrorInvalidValue);
    if (M <= 16) {
        const int g = f32_slices_of(M, N);
        return (g == 4 ? launch_f32_slices<4> : g == 2 ? launch_f32_slices<2> : launch_f32_slices<1>)(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream, F32Tail{});
    }
    const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool vec = K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && aligned(X) && aligned(W);
    switch (vec ? celeg_gemm_f32_staged_tile(M, N, K) : 0) {
        case 1: return launch_f32_tile<32, 64>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream);
        case 2: return launch_f32_tile<64, 64>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream);
        case 3: return launch_f32_tile<64, 128>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream);
    }
    if (M <= 32) return launch_f32<2, 1, 8, 512>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream);
    if (M <= 64) return launch_f32<4, 1, 4, 512>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream);
    if (!vec) {
        // Rows that cannot be read 16 bytes at a time.  One segment of k is one wavefront's work in the kernel above and the
        // others of its workgroup wait: a tile a wavefront (1,024 x 4,096, K = 33 16 us; 64 x 64 tiles 30, 32 x 64 66), with a little
        // more than one too once every CU has tiles (1,024 x 1,024, K = 129 13.9 against 15.0).  64 x 64 tiles from one a CU
        // on (1,024 x 1,024, K = 255 17.8 us, 32 x 64 21.4, a tile a wavefront 25.8; K = 1,023 34 and 40; 424 rows, 112
        // tiles, 32 and 21).
        const long long tiles = static_cast<long long>((M + 63) / 64) * ((N + 63) / 64);
        if (M <= 32 * 65535 && (K <= F32_SEGMENT || (K <= F32_SEGMENT + 16 && tiles >= 256)))
            return launch_f32_short<2, 2>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream);
        // Of these a CU holds two in 256 registers each, or one in what the compiler likes.  Two take 1.75 times as long as one, and a
        // rest of few tiles as long as one if K is long: by the rounds, then (600 x 4,096, K = 1,023 93 us by ones, 109 by twos; K = 4,095 321
        // and 297; 768 x 4,096, K = 2,047 175 and 198; 2,048 x 3,072, K = 1,025 227 and 180), and two up to 256 values of k, where
        // half of a tile's wavefronts wait (600 x 4,096, K = 255 51 and 39).
        if (tiles >= 256) {
            const long long rest = tiles % 512, ones = 100 * ((tiles + 255) / 256),
                            twos = 175 * (tiles / 512) + (rest == 0 ? 0 : rest <= 192 && K > 8 * F32_SEGMENT ? 100 : 175);
            return K <= 2 * F32_SEGMENT || twos <= ones ? launch_f32<4, 4, 2, 256, 2>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream)
                                                        : launch_f32<4, 4, 2, 256, 1>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream);
        }
    }
    return launch_f32<2, 4, 2, 512>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream);
}
