// True 32-bit matrix product for the 32-bit path: Y[M,N] = X[M,K] W[N,K]^T (+ bias).
// No reduced-precision matrix mode: the matrix cores' 32-bit instruction (16x16x4).  Every output
// element is summed in the same order whatever M, the tile or the batch is, so the logits of a row do
// not depend on how rows were batched: k in segments of 128, a segment as a chain of 32 instructions
// (instruction i of a piece of 16 takes the values i, 4 + i, 8 + i and 12 + i), then the segments'
// sums in order.
// The reference's projections: y = x W^T, weights [out, in] row-major
// (src/model/weight_plan.cpp:82-130).
//
// A workgroup owns a tile of 16 RT rows x 16 CT columns; its wavefronts take the segments in turn and
// leave their sums in LDS, where the workgroup adds them in order.  Few rows are bound by reading W: up to 16
// columns a workgroup, up to 16 wavefronts that each ask for 8 KiB at once, so
// that even a 1024 x 1024 matrix is asked for by 512 wavefronts in one trip to memory.  Many rows are bound
// by the matrix cores: larger tiles, operands straight from the caches (16 bytes a cycle and CU of them).
// Measured in a chain over different matrices (before: 64 x 64 tiles of vector instructions, k in order,
// 137 us for products of up to 64 rows and few columns with K = 1,024): 2 rows, 1024 x 1024 3.3 us, 3072 x 1024
// 5.5 us, 1024 x 4608 7.2 us (before 613), 65536 x 1024 54 us (5.0 TB/s; before 247); 64 rows, 3072 x 1024
// 13.7 us; 2,048 rows, 4608 x 1024 256 us (76 TFLOP/s).  Error against 64 bits 2.1e-7 of the result (2-norm), before 3 times that.
#include "common.h"

typedef float f32x4_t __attribute__((ext_vector_type(4)));

#define F32_SEGMENT 128
#define F32_PIECES (F32_SEGMENT / 16)

// GROUP: pieces of 16 values of k that are asked for together.  VEC: rows of X and W lie on 16 bytes
// and K is a multiple of 4; the same sums in the same order without it.
template <int RT, int CT, int GROUP, int MAX_THREADS, bool VEC>
__global__ __launch_bounds__(MAX_THREADS) void gemm_f32_kernel(
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
            load(k0 + (g + 1) * 16 * GROUP, whole, w1, x1);
            multiply(w0, x0);
            if (g + 2 < F32_PIECES / GROUP) load(k0 + (g + 2) * 16 * GROUP, whole, w0, x0);
            multiply(w1, x1);
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

// The products of up to 16 rows.  The 16 x 16 tile of the instruction is cut into G x G blocks: its rows are
// (segment g of G, column j of 16 / G) of W, its columns (segment g', row m of 16 / G) of X, so the blocks
// g = g' on the diagonal are G segments' sums of the same outputs and the others are dropped.  A workgroup
// then owns 16 / G columns, and a matrix of few columns (w2: 1,024) is spread over G times as many
// workgroups; a segment's sum is formed by the same instructions, so the outputs keep their bits.
// 2 rows: 1024 x 4608 7.2 us (on 16 columns a workgroup 14.8), 1024 x 1024 3.3 (4.5).
template <int G, bool VEC>
__global__ __launch_bounds__(1024) void gemm_f32_slices_kernel(
    const float* __restrict__ X, int ldx, const float* __restrict__ W, int ldw,
    const float* __restrict__ bias, float* __restrict__ Y, int ldy, int M, int N, int K, int wide_store) {
    constexpr int MP = 16 / G, ITEMS = MP * MP / 4;      // sums of four neighbouring columns of a row
    extern __shared__ f32x4_t parts[];                    // [segment of the round][item]
    const int wave = threadIdx.x / CELEG_WAVE, lane = threadIdx.x % CELEG_WAVE;
    const int n_waves = blockDim.x / CELEG_WAVE;
    const int qd = lane >> 4, r16 = lane & 15;
    const int col0 = blockIdx.x * MP;
    const float* const x_row = X + static_cast<size_t>(min(r16 % MP, M - 1)) * ldx;
    const float* const w_row = W + static_cast<size_t>(min(col0 + r16 % MP, N - 1)) * ldw;
    // this lane's sums: row (lane % MP) and columns 4 (quad in its block) .. + 3, of segment `of`
    const int of = qd / (MP / 4), item = (qd % (MP / 4)) * MP + lane % MP;
    const bool on_diagonal = r16 / MP == of;
    const int segments = (K + F32_SEGMENT - 1) / F32_SEGMENT;
    f32x4_t total = {0.f, 0.f, 0.f, 0.f};
    for (int first = 0; first < segments; first += n_waves * G) {
        const int mine = first + wave * G;                // this wavefront's segments: G of them from here
        const int k0 = (mine + r16 / MP) * F32_SEGMENT + 4 * qd;
        f32x4_t wv[F32_PIECES], xv[F32_PIECES];
        if (VEC && (mine + G) * F32_SEGMENT <= K) {
#pragma unroll
            for (int s = 0; s < F32_PIECES; ++s) wv[s] = *reinterpret_cast<const f32x4_t*>(w_row + k0 + 16 * s);
#pragma unroll
            for (int s = 0; s < F32_PIECES; ++s) xv[s] = *reinterpret_cast<const f32x4_t*>(x_row + k0 + 16 * s);
        } else {
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
    const int row = threadIdx.x % MP, col = col0 + 4 * (threadIdx.x / MP);
    if (threadIdx.x >= ITEMS || row >= M) return;
    float* y = Y + static_cast<size_t>(row) * ldy + col;
    if (wide_store && col + 3 < N) {
        if (bias) total += f32x4_t{bias[col], bias[col + 1], bias[col + 2], bias[col + 3]};
        *reinterpret_cast<f32x4_t*>(y) = total;
        return;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (col + r < N) y[r] = total[r] + (bias ? bias[col + r] : 0.f);
}

template <int G>
static int launch_f32_slices(const float* X, int ldx, const float* W, int ldw, const float* bias, float* Y, int ldy,
                             int M, int N, int K, hipStream_t stream) {
    const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool vec = K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && aligned(X) && aligned(W);
    const int wide_store = ldy % 4 == 0 && aligned(Y);
    constexpr int MP = 16 / G;
    const int groups = ((K + F32_SEGMENT - 1) / F32_SEGMENT + G - 1) / G;
    const int rounds = (groups + 15) / 16, waves = (groups + rounds - 1) / rounds;     // as even as it goes: 36 are 3 rounds of 12
    const dim3 grid((N + MP - 1) / MP), block(waves * CELEG_WAVE);
    const size_t lds = static_cast<size_t>(waves) * G * (MP * MP / 4) * sizeof(f32x4_t);
    auto kernel = vec ? &gemm_f32_slices_kernel<G, true> : &gemm_f32_slices_kernel<G, false>;
    hipLaunchKernelGGL(kernel, grid, block, lds, stream, X, ldx, W, ldw, bias, Y, ldy, M, N, K, wide_store);
    return CELEG_LAUNCH_RESULT();
}

template <int RT, int CT, int GROUP, int MAX_THREADS>
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
    if (vec)
        hipLaunchKernelGGL((gemm_f32_kernel<RT, CT, GROUP, MAX_THREADS, true>), grid, block, lds, stream, X, ldx, W, ldw, bias, Y, ldy, M, N, K, wide_store);
    else
        hipLaunchKernelGGL((gemm_f32_kernel<RT, CT, GROUP, MAX_THREADS, false>), grid, block, lds, stream, X, ldx, W, ldw, bias, Y, ldy, M, N, K, wide_store);
    return CELEG_LAUNCH_RESULT();
}

// The products of many rows over a short K.  A wavefront has a tile of 16 RT x 16 CT outputs to itself and goes
// through the segments one after the other, each summed and added as above, so the outputs have the same bits; there
// is nothing to join, and a last segment that is not whole costs what it has.  2,048 x 4,096: K = 32 18 us (on the
// kernel above, most of whose wavefronts then wait, 86; before that 26), K = 128 50 (95), K = 160 60 (100; 75).
template <int RT, int CT, bool VEC>
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
        if (VEC) {
            if (k < K) v = *reinterpret_cast<const f32x4_t*>(row + k);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (k + i < K) v[i] = row[k + i];
        }
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
    const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool vec = K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && aligned(X) && aligned(W);
    const int wide_store = ldy % 4 == 0 && aligned(Y);
    const dim3 grid((N + 64 * CT - 1) / (64 * CT), (M + 16 * RT - 1) / (16 * RT)), block(4 * CELEG_WAVE);
    auto kernel = vec ? &gemm_f32_short_kernel<RT, CT, true> : &gemm_f32_short_kernel<RT, CT, false>;
    hipLaunchKernelGGL(kernel, grid, block, 0, stream, X, ldx, W, ldw, bias, Y, ldy, M, N, K, wide_store);
    return CELEG_LAUNCH_RESULT();
}

extern "C" int celeg_gemm_f32(const float* X, int ldx, const float* W, int ldw, const float* bias,
                              float* Y, int ldy, int M, int N, int K, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0) return static_cast<int>(hipErrorInvalidValue);
    // (blocks of 4 or 8 columns while tiles of 16 would leave compute units without a second workgroup)
    if (M <= 16) {
        const int g = N >= 512 * 16 || M > 8 ? 1 : M > 4 ? 2 : 4;
        return (g == 4 ? launch_f32_slices<4> : g == 2 ? launch_f32_slices<2> : launch_f32_slices<1>)(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream);
    }
    if (M <= 32) return launch_f32<2, 1, 8, 512>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream);
    if (M <= 64) return launch_f32<4, 1, 4, 512>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream);
    // One segment of k is one wavefront's work in the kernel above and the others of its workgroup wait; with two, the
    // wavefront to itself is the faster one once there are tiles enough for every CU (K = 256: 1,024 x 1,024
    // 14.7 us against 16.9, 424 x 1,024 13.4 against 9.4; K = 384: 2,048 x 1,024 36 against 32).
    const long long tiles = static_cast<long long>((M + 63) / 64) * ((N + 63) / 64);
    if (M <= 32 * 65535 && (K <= F32_SEGMENT || (K <= 2 * F32_SEGMENT && tiles >= 256)))      // (a grid has 65,535 rows of tiles)
        return launch_f32_short<2, 2>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream);
    // 64 x 64 tiles (an operand from the caches serves four products) once there are two for every CU; below
    // that (350 rows: 96 of them at N = 1,024) half the tile and twice the wavefronts
    if (tiles >= 512)
        return launch_f32<4, 4, 2, 256>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream);
    return launch_f32<2, 4, 2, 512>(X, ldx, W, ldw, bias, Y, ldy, M, N, K, stream);
}
