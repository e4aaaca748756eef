// What holds a layer together besides its norms: activations with a bias, sums into the 32-bit
// residual stream, a per-layer token input, the mean of several normed branches, and the
// weighted sum over the results of all earlier layers, what a stream takes in before a run of a looped
// range, and logits bent by a tanh.  All arithmetic is 32-bit; T is the
// run's dtype of the branch rows.
#include "activations.h"
#include "common.h"

namespace {

// out = act(x + bias); act 0: gelu (tanh form), 1: square of relu, 2: none, 3: lg_bent with (p0, p1)
template <typename T>
__global__ void activation_bias_kernel(const T* __restrict__ x, int ldx, const float* __restrict__ bias, T* __restrict__ out,
                                       int ldo, int cols, int act, float p0, float p1) {
    const int t = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= cols) return;
    float z = to_float(x[static_cast<size_t>(t) * ldx + c]);
    if (bias) z += bias[c];
    out[static_cast<size_t>(t) * ldo + c] = from_float<T>(activated(z, act, p0, p1));
}

// The same without a bias on dense rows of the run's dtype that lie one after the other: eight values a thread.
template <typename T>
__global__ __launch_bounds__(256) void activation_dense_kernel(const T* __restrict__ x, T* __restrict__ out, size_t groups, int act, float p0,
                                                               float p1) {
    struct alignas(8 * sizeof(T)) Eight { T v[8]; };
    const size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= groups) return;
    Eight in = reinterpret_cast<const Eight*>(x)[i];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float z = to_float(in.v[e]);
        in.v[e] = from_float<T>(activated(z, act, p0, p1));
    }
    reinterpret_cast<Eight*>(out)[i] = in;
}

// h += a (+ b); copy (optional) receives the new rows in the run's dtype
template <typename T>
__global__ void residual_sum_kernel(float* __restrict__ h, const T* __restrict__ a, int lda, const T* __restrict__ b, int ldb,
                                    T* __restrict__ copy, int width) {
    const int t = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= width) return;
    float add = to_float(a[static_cast<size_t>(t) * lda + c]);
    if (b) add += to_float(b[static_cast<size_t>(t) * ldb + c]);
    const float v = h[static_cast<size_t>(t) * width + c] + add;
    h[static_cast<size_t>(t) * width + c] = v;
    if (copy) copy[static_cast<size_t>(t) * width + c] = from_float<T>(v);
}

// g[t, j] = gelu(z[t, j]) * table[token[t], offset + j]
template <typename T>
__global__ void token_gate_kernel(const T* __restrict__ z, int ldz, const T* __restrict__ table, int ld_table, int offset,
                                  const int* __restrict__ token_ids, T* __restrict__ g, int dim) {
    const int t = blockIdx.y;
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= dim) return;
    const float e = to_float(table[static_cast<size_t>(token_ids[t]) * ld_table + offset + j]);
    g[static_cast<size_t>(t) * dim + j] = from_float<T>(lg_gelu_tanh(to_float(z[static_cast<size_t>(t) * ldz + j])) * e);
}

// out[t] = factor * (a[t] / rms(a[t]) * wa + b[t] / rms(b[t]) * wb); one workgroup a row
template <typename T>
__global__ __launch_bounds__(256) void normed_mean_kernel(const T* __restrict__ a, int lda, const float* __restrict__ wa,
                                                          const T* __restrict__ b, int ldb, const float* __restrict__ wb, float eps,
                                                          float factor, T* __restrict__ out, int width) {
    __shared__ float scratch[16];
    const int t = blockIdx.x;
    const T* ar = a + static_cast<size_t>(t) * lda;
    const T* br = b + static_cast<size_t>(t) * ldb;
    float sa = 0.f, sb = 0.f;
    for (int c = threadIdx.x; c < width; c += blockDim.x) {
        const float x = to_float(ar[c]), y = to_float(br[c]);
        sa = fmaf(x, x, sa);
        sb = fmaf(y, y, sb);
    }
    sa = block_sum(sa, scratch);
    sb = block_sum(sb, scratch);
    const float ia = 1.0f / sqrtf(sa / static_cast<float>(width) + eps), ib = 1.0f / sqrtf(sb / static_cast<float>(width) + eps);
    for (int c = threadIdx.x; c < width; c += blockDim.x)
        out[static_cast<size_t>(t) * width + c] = from_float<T>(factor * (to_float(ar[c]) * ia * wa[c] + to_float(br[c]) * ib * wb[c]));
}

// history [n, rows_cap, width] 32-bit holds the results of the n - 1 entries before (the embedding's rows first);
// the stream's rows become entry n - 1, and the stream becomes sum_j w[j] history[j], j rising
__global__ void depth_mix_kernel(float* __restrict__ history, size_t entry_stride, float* __restrict__ h, const float* __restrict__ w,
                                 int n, int width) {
    const int t = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= width) return;
    const size_t at = static_cast<size_t>(t) * width + c;
    const float last = h[at];
    history[static_cast<size_t>(n - 1) * entry_stride + at] = last;
    float sum = 0.f;
    for (int j = 0; j < n - 1; ++j) sum = fmaf(w[j], history[static_cast<size_t>(j) * entry_stride + at], sum);
    h[at] = fmaf(w[n - 1], last, sum);
}

// Row rows[r] of h to row r of h_out and, where there is an a, its row likewise (in groups of 8 values k8_stride apart); one
// workgroup a row.  A thread takes four values of h and eight of a at a time: every load of 1,024 values of h and of 2,048 of a is
// asked for at once.  What bounds it is one trip to memory for the row's number and one for the row (one row of 1,024 values and 1,024
// of the branch: 3.0 us with its launch).
template <typename T, bool WIDE>
__global__ __launch_bounds__(256) void gather_rows_kernel(const int* __restrict__ rows, const float* __restrict__ h, float* __restrict__ h_out,
                                                          int width, const T* __restrict__ a, size_t lda, T* __restrict__ a_out,
                                                          size_t lda_out, size_t k8_stride, int inner) {
    const int r = blockIdx.x;
    const size_t from = rows[r];
    const float* const hr = h + from * width;
    float* const ho = h_out + static_cast<size_t>(r) * width;
    const T* const ar = a + from * lda;
    T* const ao = a_out + r * lda_out;
    if constexpr (WIDE) {
        typedef float f32x4 __attribute__((ext_vector_type(4)));
        struct alignas(16) Eight { T v[8]; };
        for (int i = threadIdx.x; i < width / 4; i += 256) reinterpret_cast<f32x4*>(ho)[i] = reinterpret_cast<const f32x4*>(hr)[i];
        for (int i = threadIdx.x; i < inner / 8; i += 256)
            *reinterpret_cast<Eight*>(ao + i * k8_stride) = *reinterpret_cast<const Eight*>(ar + 8 * i);
    } else {
        for (int i = threadIdx.x; i < width; i += 256) ho[i] = hr[i];
        for (int i = threadIdx.x; i < inner; i += 256) ao[(i >> 3) * k8_stride + (i & 7)] = ar[i];
    }
}

// h[t, :] += (rows[t, :] +) vec, all 32-bit: what a stream takes in before a run of a looped range
__global__ void stream_add_kernel(float* __restrict__ h, const float* __restrict__ rows, const float* __restrict__ vec, int width) {
    const int t = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= width) return;
    const size_t at = static_cast<size_t>(t) * width + c;
    float v = h[at];
    if (rows) v += rows[at];
    if (vec) v += vec[c];
    h[at] = v;
}

// x <- cap * tanh(x / cap), 32-bit
__global__ void softcap_kernel(float* __restrict__ x, size_t n, float cap) {
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) x[i] = cap * tanhf(x[i] / cap);
}

}  // namespace

#define LG_BY_DTYPE(kernel, grid, block, ...)                                                      \
    if (dtype == CELEG_F32) {                                                                      \
        using T = float;                                                                           \
        hipLaunchKernelGGL(kernel<T>, grid, block, 0, stream, __VA_ARGS__);                        \
    } else {                                                                                       \
        using T = bf16;                                                                            \
        hipLaunchKernelGGL(kernel<T>, grid, block, 0, stream, __VA_ARGS__);                        \
    }

// Few values, up to a workgroup of 256 on every compute unit, go one a thread: such a launch is a chain in
// which the code itself, 4.9 KB of it for eight values and 0.8 KB for one, is fetched anew (4 rows of 3,072,
// gelu: 3.1 -> 2.0 us).
#define LG_FEW_VALUES (256 * 256)

extern "C" int celeg_activation_bias(const void* x, int ldx, const float* bias, void* out, int ldo, int dtype, int rows, int cols,
                                     int act, float p0, float p1, hipStream_t stream) {
    if (rows <= 0 || cols <= 0) return 0;
    const size_t piece = 8 * (dtype == CELEG_F32 ? 4 : 2), count = static_cast<size_t>(rows) * cols;
    if (!bias && count > LG_FEW_VALUES && count % 8 == 0 && (rows == 1 || (ldx == cols && ldo == cols)) &&
        ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) & (piece - 1)) == 0) {
        dim3 grid(static_cast<unsigned>((count / 8 + 255) / 256)), block(256);
        LG_BY_DTYPE(activation_dense_kernel, grid, block, static_cast<const T*>(x), static_cast<T*>(out), count / 8, act, p0, p1);
        return CELEG_LAUNCH_RESULT();
    }
    dim3 grid((cols + 255) / 256, rows), block(256);
    LG_BY_DTYPE(activation_bias_kernel, grid, block, static_cast<const T*>(x), ldx, bias, static_cast<T*>(out), ldo, cols, act, p0, p1);
    return CELEG_LAUNCH_RESULT();
}

extern "C" int celeg_residual_sum(float* h, const void* a, int lda, const void* b, int ldb, void* copy, int dtype, int rows,
                                  int width, hipStream_t stream) {
    if (rows <= 0) return 0;
    dim3 grid((width + 255) / 256, rows), block(256);
    LG_BY_DTYPE(residual_sum_kernel, grid, block, h, static_cast<const T*>(a), lda, static_cast<const T*>(b), ldb,
                static_cast<T*>(copy), width);
    return CELEG_LAUNCH_RESULT();
}

extern "C" int celeg_token_gate(const void* z, int ldz, const void* table, int ld_table, int offset, const int* token_ids, void* g,
                                int dtype, int rows, int dim, hipStream_t stream) {
    if (rows <= 0) return 0;
    dim3 grid((dim + 63) / 64, rows), block(64);
    LG_BY_DTYPE(token_gate_kernel, grid, block, static_cast<const T*>(z), ldz, static_cast<const T*>(table), ld_table, offset,
                token_ids, static_cast<T*>(g), dim);
    return CELEG_LAUNCH_RESULT();
}

extern "C" int celeg_normed_mean(const void* a, int lda, const float* wa, const void* b, int ldb, const float* wb, float eps,
                                 float factor, void* out, int dtype, int rows, int width, hipStream_t stream) {
    if (rows <= 0) return 0;
    dim3 grid(rows), block(256);
    LG_BY_DTYPE(normed_mean_kernel, grid, block, static_cast<const T*>(a), lda, wa, static_cast<const T*>(b), ldb, wb, eps, factor,
                static_cast<T*>(out), width);
    return CELEG_LAUNCH_RESULT();
}

extern "C" int celeg_depth_mix(float* history, size_t entry_stride, float* h, const float* w, int n, int rows, int width,
                               hipStream_t stream) {
    if (rows <= 0 || n <= 0) return 0;
    dim3 grid((width + 255) / 256, rows), block(256);
    hipLaunchKernelGGL(depth_mix_kernel, grid, block, 0, stream, history, entry_stride, h, w, n, width);
    return CELEG_LAUNCH_RESULT();
}

extern "C" int celeg_stream_add(float* h, const float* rows, const float* vec, int n_rows, int width, hipStream_t stream) {
    if (n_rows <= 0 || (!rows && !vec)) return 0;
    dim3 grid((width + 255) / 256, n_rows), block(256);
    hipLaunchKernelGGL(stream_add_kernel, grid, block, 0, stream, h, rows, vec, width);
    return CELEG_LAUNCH_RESULT();
}

extern "C" int celeg_gather_rows(const int* rows, int n, const float* h, float* h_out, int width, const void* a, long long lda, void* a_out,
                                 long long lda_out, long long k8_stride, int inner, int dtype, hipStream_t stream) {
    if (n <= 0) return 0;
    if (width <= 0 || inner < 0 || (inner > 0 && (!a || !a_out))) return static_cast<int>(hipErrorInvalidValue);
    dim3 grid(n), block(256);
    const auto on16 = [](const void* p, long long row_bytes) { return ((reinterpret_cast<uintptr_t>(p) | static_cast<uintptr_t>(row_bytes)) & 15) == 0; };
    const long long size = dtype == CELEG_F32 ? 4 : 2;
    const bool wide = on16(h, width * 4LL) && on16(h_out, 0) && inner % 8 == 0 && on16(a, lda * size) && on16(a_out, lda_out * size) &&
                      on16(nullptr, k8_stride * size);
#define LG_GATHER(T, WIDE)                                                                                                     \
    hipLaunchKernelGGL((gather_rows_kernel<T, WIDE>), grid, block, 0, stream, rows, h, h_out, width, static_cast<const T*>(a),     \
                       static_cast<size_t>(lda), static_cast<T*>(a_out), static_cast<size_t>(lda_out), static_cast<size_t>(k8_stride), inner)
    if (dtype == CELEG_F32) {
        if (wide) LG_GATHER(float, true); else LG_GATHER(float, false);
    } else {
        if (wide) LG_GATHER(bf16, true); else LG_GATHER(bf16, false);
    }
#undef LG_GATHER
    return CELEG_LAUNCH_RESULT();
}

extern "C" int celeg_softcap(float* x, size_t n, float cap, hipStream_t stream) {
    if (n == 0) return 0;
    if (!(cap > 0.f)) return static_cast<int>(hipErrorInvalidValue);
    hipLaunchKernelGGL(softcap_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, stream, x, n, cap);
    return CELEG_LAUNCH_RESULT();
}
