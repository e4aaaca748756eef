// A sub-layer boundary of a block that norms a branch's output before adding it: for a row of
// the 32-bit residual stream h and the branch output y,
//     h += post(y)          (post: a layer norm, an RMS norm, or nothing but the addition)
//     out = pre(h)          (pre: the next sub-layer's norm; or no output at all)
// in one pass over the row, with every statistic and sum in 32-bit.  Either half may be absent,
// so the same kernel is a plain layer norm (with a gather of rows for the output head), the
// addition alone, or both.
//
// Layer norm: (x - mean) / sqrt(var + eps) * w + b with var the mean of the squared deviations
// from the mean (two passes over the row, which is staged in LDS).  RMS norm:
// x / sqrt(mean(x^2) + eps) * w.  The bias is optional in both.  "Dynamic tanh": tanh(alpha * x) * w + b
// with one number alpha, no statistic of the row at all.  A norm's `gain` multiplies what it gives
// as a whole (a block that adds m * post(y)).
#include "common.h"

#include "norm_params.h"

namespace {

// one value through a norm whose statistics are (shift, factor)
__device__ __forceinline__ float normed_value(float x, const CelegNorm& n, float shift, float factor, float w, float b) {
    const float v = n.mode == CELEG_NORM_TANH ? tanhf(n.alpha * x) : (x - shift) * factor;
    return (v * w + b) * n.gain;
}

// the statistics of `row` (LDS, width floats) for a norm of this mode: (shift, factor) such that
// the normalised value is (x - shift) * factor
__device__ __forceinline__ void row_stats(const float* row, int width, int mode, float eps, float* scratch, float& shift,
                                          float& factor) {
    shift = 0.f;
    factor = 1.f;
    if (mode == CELEG_NORM_LAYER) {
        float s = 0.f;
        for (int i = threadIdx.x; i < width; i += blockDim.x) s += row[i];
        shift = block_sum(s, scratch) / static_cast<float>(width);
    }
    if (mode == CELEG_NORM_LAYER || mode == CELEG_NORM_RMS) {
        float s = 0.f;
        for (int i = threadIdx.x; i < width; i += blockDim.x) {
            const float d = row[i] - shift;
            s += d * d;
        }
        factor = 1.0f / sqrtf(block_sum(s, scratch) / static_cast<float>(width) + eps);
    }
}

template <typename TY, typename TO>
__global__ __launch_bounds__(256) void norm_step_kernel(float* __restrict__ h, const TY* __restrict__ y, CelegNorm post,
                                                        CelegNorm pre, TO* __restrict__ out, const int* __restrict__ rows,
                                                        int width, int write_back) {
    extern __shared__ float row[];     // width floats
    __shared__ float scratch[16];
    const int r = blockIdx.x;
    const size_t src = static_cast<size_t>(rows ? rows[r] : r) * width;
    if (y) {
        for (int i = threadIdx.x; i < width; i += blockDim.x) row[i] = to_float(y[src + i]);
        __syncthreads();
        float shift, factor;
        row_stats(row, width, post.mode, post.eps, scratch, shift, factor);
        for (int i = threadIdx.x; i < width; i += blockDim.x) {
            float v = normed_value(row[i], post, shift, factor, post.w ? post.w[i] : 1.f, post.b ? post.b[i] : 0.f);
            v += h[src + i];
            row[i] = v;                 // (its own element: no other thread reads it before the barrier)
            if (write_back) h[src + i] = v;
        }
    } else {
        for (int i = threadIdx.x; i < width; i += blockDim.x) row[i] = h[src + i];
    }
    if (!out) return;
    __syncthreads();
    float shift, factor;
    row_stats(row, width, pre.mode, pre.eps, scratch, shift, factor);
    TO* dst = out + static_cast<size_t>(r) * width;
    for (int i = threadIdx.x; i < width; i += blockDim.x) {
        dst[i] = from_float<TO>(normed_value(row[i], pre, shift, factor, pre.w ? pre.w[i] : 1.f, pre.b ? pre.b[i] : 0.f));
    }
}

// The same for rows of up to 1024 * NG values, with the row in registers: a thread holds NG groups of four
// values, and everything that it reads (branch output, stream, both norms' weights and biases) is asked
// for at once, so that a row waits for memory once.  VEC: a group is four neighbours, read as one;
// otherwise (a row that is no whole number of groups, or an operand that is not on 16 bytes) it is four
// values 256 apart.
//
// A step of few rows runs this on as many workgroups, and its time is a chain: the launch, the loads, up to
// four sums over the row, and the fetching of the code itself, of which each launch has evicted the last.
// So the code is kept short (2.4 KB instead of 7.0): one load instead of four, no load under a condition
// whose result is converted inside it, one barrier a sum (each has its own four floats of LDS), and the
// tanh form is a kernel of its own.  4 rows of 1,024 values, two layer norms: 6.0 -> 3.0 us; a norm
// alone 3.1 -> 2.5, an addition alone 3.7 -> 2.5.
// the sum over the block of 256 in the order of block_sum; `slot` is used by this sum alone
__device__ __forceinline__ float row_sum(float v, float* slot) {
    v = wave_sum(v);
    if ((threadIdx.x & (CELEG_WAVE - 1)) == 0) slot[threadIdx.x / CELEG_WAVE] = v;
    __syncthreads();
    return slot[0] + slot[1] + slot[2] + slot[3];
}

// the place in the row of a thread's value e of group g
template <bool VEC>
__device__ __forceinline__ int value_at(int g, int e) {
    return VEC ? 4 * (static_cast<int>(threadIdx.x) + 256 * g) + e : static_cast<int>(threadIdx.x) + 256 * (4 * g + e);
}
template <bool VEC>
__device__ __forceinline__ bool in_row(int k, int width) {
    return value_at<VEC>(k / 4, VEC ? 0 : k % 4) < width;     // (a group read as one is in the row or not)
}

template <int NG, bool VEC, bool TANH>
__device__ __forceinline__ void reg_norm(float (&v)[4 * NG], int width, const CelegNorm& n, const float (&w)[4 * NG],
                                         const float (&b)[4 * NG], float* scratch) {
    float shift = 0.f, factor = 1.f;
    if (n.mode == CELEG_NORM_LAYER) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 4 * NG; ++i) s += in_row<VEC>(i, width) ? v[i] : 0.f;
        shift = row_sum(s, scratch) / static_cast<float>(width);
    }
    if (n.mode == CELEG_NORM_LAYER || n.mode == CELEG_NORM_RMS) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 4 * NG; ++i) {
            const float d = in_row<VEC>(i, width) ? v[i] - shift : 0.f;
            s += d * d;
        }
        factor = 1.0f / sqrtf(row_sum(s, scratch + 4) / static_cast<float>(width) + n.eps);
    }
#pragma unroll
    for (int i = 0; i < 4 * NG; ++i) {
        const float x = TANH && n.mode == CELEG_NORM_TANH ? tanhf(n.alpha * v[i]) : (v[i] - shift) * factor;
        v[i] = (x * w[i] + b[i]) * n.gain;
    }
}

__device__ __forceinline__ float to_raw(float x) { return x; }
__device__ __forceinline__ __bf16 to_raw(bf16 x) { return __builtin_bit_cast(__bf16, x.bits); }

// the row at p, or at `other` where there is none (its values are then not used: a load that always
// happens costs less than the branch round it); places past the row read its first values
template <typename T, int NG, bool VEC>
struct RowLoad {
    typename Vec4<T>::raw raw[NG];
    bool there;
    __device__ __forceinline__ RowLoad(const T* p, const void* other, int width) : there(p != nullptr) {
        const T* from = there ? p : static_cast<const T*>(other);
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            if (VEC) {
                const int i = value_at<true>(g, 0);
                raw[g] = *reinterpret_cast<const typename Vec4<T>::raw*>(from + (i < width ? i : 0));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int i = value_at<false>(g, e);
                    raw[g][e] = to_raw(from[i < width ? i : 0]);
                }
            }
        }
    }
    __device__ __forceinline__ void values(float none, float (&v)[4 * NG]) const {
#pragma unroll
        for (int k = 0; k < 4 * NG; ++k) v[k] = there ? static_cast<float>(raw[k / 4][k % 4]) : none;
    }
};

template <typename T, int NG, bool VEC>
__device__ __forceinline__ void row_store(T* p, int width, const float (&v)[4 * NG]) {
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        if (VEC) {
            const int i = value_at<true>(g, 0);
            const float o[4] = {v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
            if (i < width) Vec4<T>::store(p + i, o);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int i = value_at<false>(g, e);
                if (i < width) p[i] = from_float<T>(v[4 * g + e]);
            }
        }
    }
}

template <typename TY, typename TO, int NG, bool VEC, bool TANH>
__global__ __launch_bounds__(256) void norm_step_reg_kernel(float* __restrict__ h, const TY* __restrict__ y, CelegNorm post,
                                                            CelegNorm pre, TO* __restrict__ out, const int* __restrict__ rows,
                                                            int width, int write_back) {
    __shared__ float scratch[16];
    const int r = blockIdx.x;
    const size_t src = static_cast<size_t>(rows ? rows[r] : r) * width;
    float* row = h + src;
    const RowLoad<float, NG, VEC> h_row(row, row, width), post_w(post.w, row, width), post_b(post.b, row, width),
        pre_w(pre.w, row, width), pre_b(pre.b, row, width);
    const RowLoad<TY, NG, VEC> y_row(y ? y + src : nullptr, row, width);
    float hv[4 * NG], yv[4 * NG], w[4 * NG], b[4 * NG];
    y_row.values(0.f, yv);                  // (no branch output: the norm of it is skipped, and zeros are added)
    post_w.values(1.f, w);
    post_b.values(0.f, b);
    reg_norm<NG, VEC, TANH>(yv, width, post, w, b, scratch);
    h_row.values(0.f, hv);
#pragma unroll
    for (int k = 0; k < 4 * NG; ++k) hv[k] = yv[k] + hv[k];
    if (write_back) row_store<float, NG, VEC>(row, width, hv);
    if (!out) return;
    pre_w.values(1.f, w);
    pre_b.values(0.f, b);
    reg_norm<NG, VEC, TANH>(hv, width, pre, w, b, scratch + 8);
    row_store<TO, NG, VEC>(out + static_cast<size_t>(r) * width, width, hv);
}

template <typename TO>
__global__ void concat_rows_kernel(const float* __restrict__ a, const float* __restrict__ b, TO* __restrict__ out, size_t rows,
                                   int width) {
    const size_t idx = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= rows * 2 * width) return;
    const size_t r = idx / (2 * width);
    const int c = static_cast<int>(idx % (2 * width));
    out[idx] = from_float<TO>(c < width ? a[r * width + c] : b[r * width + c - width]);
}

}  // namespace

extern "C" int celeg_norm_step(float* h, const void* y, int y_dtype, CelegNorm post, CelegNorm pre, void* out, int out_dtype,
                               const int* rows, int n_rows, int width, int write_back, hipStream_t stream) {
    if (n_rows <= 0) return 0;
    const size_t lds = static_cast<size_t>(width) * sizeof(float);
    if (lds > 60 * 1024) return static_cast<int>(hipErrorInvalidValue);
    dim3 grid(n_rows), block(256);
    if (!y) post = CelegNorm{nullptr, nullptr, 0.f, CELEG_NORM_NONE, 1.f, 1.f};
    const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool vec = width % 4 == 0 && aligned(h) && aligned(y) && aligned(out) && aligned(post.w) && aligned(post.b) &&
                     aligned(pre.w) && aligned(pre.b);
    const bool tanh = post.mode == CELEG_NORM_TANH || (out && pre.mode == CELEG_NORM_TANH);
#define CELEG_NORM_STEP_REG(TY, TO, NG, VEC, TANH)                                                                         \
    hipLaunchKernelGGL((norm_step_reg_kernel<TY, TO, NG, VEC, TANH>), grid, block, 0, stream, h, static_cast<const TY*>(y), \
                       post, pre, static_cast<TO*>(out), rows, width, write_back)
#define CELEG_NORM_STEP_NG(TY, TO, NG)                                                                                     \
    if (vec && !tanh) { CELEG_NORM_STEP_REG(TY, TO, NG, true, false); }                                                    \
    else if (vec) { CELEG_NORM_STEP_REG(TY, TO, NG, true, true); }                                                         \
    else { CELEG_NORM_STEP_REG(TY, TO, NG, false, true); }
#define CELEG_NORM_STEP(TY, TO)                                                                                            \
    if (width <= 1024) {                                                                                                   \
        CELEG_NORM_STEP_NG(TY, TO, 1)                                                                                      \
    } else if (width <= 2048) {                                                                                            \
        CELEG_NORM_STEP_NG(TY, TO, 2)                                                                                      \
    } else                                                                                                                 \
        hipLaunchKernelGGL((norm_step_kernel<TY, TO>), grid, block, lds, stream, h, static_cast<const TY*>(y), post, pre,     \
                           static_cast<TO*>(out), rows, width, write_back)
    if (y_dtype == CELEG_F32 && out_dtype == CELEG_F32) { CELEG_NORM_STEP(float, float); }
    else if (y_dtype == CELEG_F32) { CELEG_NORM_STEP(float, bf16); }
    else if (out_dtype == CELEG_F32) { CELEG_NORM_STEP(bf16, float); }
    else { CELEG_NORM_STEP(bf16, bf16); }
#undef CELEG_NORM_STEP
#undef CELEG_NORM_STEP_NG
#undef CELEG_NORM_STEP_REG
    return CELEG_LAUNCH_RESULT();
}

// out [rows, 2 * width] = (a | b) row by row, both 32-bit, in the dtype of out
extern "C" int celeg_concat_rows(const float* a, const float* b, void* out, int out_dtype, int rows, int width,
                                 hipStream_t stream) {
    const size_t total = static_cast<size_t>(rows) * 2 * width;
    if (total == 0) return 0;
    dim3 grid(static_cast<unsigned>((total + 255) / 256)), block(256);
    if (out_dtype == CELEG_F32)
        hipLaunchKernelGGL(concat_rows_kernel<float>, grid, block, 0, stream, a, b, static_cast<float*>(out),
                           static_cast<size_t>(rows), width);
    else
        hipLaunchKernelGGL(concat_rows_kernel<bf16>, grid, block, 0, stream, a, b, static_cast<bf16*>(out),
                           static_cast<size_t>(rows), width);
    return CELEG_LAUNCH_RESULT();
}
