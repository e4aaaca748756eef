// Double-gated short causal convolution over the rows of a step, continuing each
// request from its saved state, and the state update that follows.
//
// bcx[t] = [B | C | x] (each `width` wide); bx = B*x;
// conv[t,ch] = sum_tap w[ch,tap] * bx[pos(t) - (taps-1-tap), ch] (+ bias), zero before
// position 0; y = C * conv.   Reference: src/backend/cpu/kernels/convolution.cpp:7-60;
// ragged CUDA form src/backend/cuda/kernels/shortconv.cuh:34-64.
//
// State per request [taps, width] in 32-bit: entry j holds bx at position
// (tokens seen) - taps + j.  The forward kernels read only the OLD state and the rows
// of the step; the update kernel runs after them on the same stream, except behind the
// kernel for long steps, which updates the state itself (the thread that read a request's
// old state writes its new one).  bx is kept as the unrounded 32-bit product both in the
// state and when read from rows, so cutting a sequence into steps changes nothing.
#include "common.h"

template <typename T>
__global__ void short_conv_fwd_kernel(
    const T* __restrict__ bcx, int ld_bcx, const float* __restrict__ w,
    const float* __restrict__ bias, const float* __restrict__ state, size_t state_slot_stride,
    T* __restrict__ out, const int* __restrict__ positions, const int* __restrict__ token_seq,
    const int* __restrict__ seq_start, const int* __restrict__ seq_slot,
    const int* __restrict__ cu_seqlens, int width, int taps) {
    const int ch = blockIdx.y * blockDim.x + threadIdx.x;
    if (ch >= width) return;
    const int t = blockIdx.x;
    const int s = token_seq[t];
    const int start = seq_start[s];
    const int row0 = cu_seqlens[s];
    const int pos = positions[t];
    const float* st = state + static_cast<size_t>(seq_slot[s]) * state_slot_stride;
    float conv = 0.f;
    for (int tap = 0; tap < taps; ++tap) {
        const int q = pos - (taps - 1 - tap);
        if (q < 0) continue;
        float bx;
        if (q >= start) {
            const T* row = bcx + static_cast<size_t>(row0 + (q - start)) * ld_bcx;
            bx = to_float(row[ch]) * to_float(row[2 * width + ch]);
        } else {
            bx = st[static_cast<size_t>(q - start + taps) * width + ch];
        }
        conv = fmaf(w[static_cast<size_t>(ch) * taps + tap], bx, conv);
    }
    if (bias) conv += bias[ch];
    const float c = to_float(bcx[static_cast<size_t>(t) * ld_bcx + width + ch]);
    out[static_cast<size_t>(t) * width + ch] = from_float<T>(c * conv);
}

// The same for groups of channels (16 bytes of a row per load): a thread takes VEC
// neighbouring channels of one token.  Tokens whose taps all lie in rows of this step (all
// but the first taps-1 of a portion) ask for every row at once; the others go the slower way
// through the state.
template <typename T> struct ConvVec;
template <> struct ConvVec<float> {
    static constexpr int n = 4;
    typedef float raw __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ float at(const raw& r, int i) { return r[i]; }
    static __device__ __forceinline__ void set(raw& r, int i, float v) { r[i] = v; }
};
template <> struct ConvVec<bf16> {
    static constexpr int n = 8;
    typedef __bf16 raw __attribute__((ext_vector_type(8)));
    static __device__ __forceinline__ float at(const raw& r, int i) { return static_cast<float>(r[i]); }
    static __device__ __forceinline__ void set(raw& r, int i, float v) { r[i] = static_cast<__bf16>(v); }
};
#define CONV_VEC_MAX_TAPS 8

template <typename T>
__device__ __forceinline__ void short_conv_token_vec(
    int t, int ch, const T* __restrict__ bcx, int ld_bcx, const float* __restrict__ w,
    const float* __restrict__ bias, const float* state, size_t state_slot_stride,
    T* __restrict__ out, const int* __restrict__ positions, const int* __restrict__ token_seq,
    const int* __restrict__ seq_start, const int* __restrict__ seq_slot,
    const int* __restrict__ cu_seqlens, int width, int taps) {
    constexpr int VEC = ConvVec<T>::n;
    typedef typename ConvVec<T>::raw raw;
    const int s = token_seq[t];
    const int start = seq_start[s];
    const int row0 = cu_seqlens[s];
    const int pos = positions[t];
    float conv[VEC];
#pragma unroll
    for (int i = 0; i < VEC; ++i) conv[i] = bias ? bias[ch + i] : 0.f;
    const raw cv = *reinterpret_cast<const raw*>(bcx + static_cast<size_t>(t) * ld_bcx + width + ch);
    if (pos - (taps - 1) >= start) {        // the same for the whole workgroup
        raw bv[CONV_VEC_MAX_TAPS], xv[CONV_VEC_MAX_TAPS];
#pragma unroll
        for (int tap = 0; tap < CONV_VEC_MAX_TAPS; ++tap) {
            // rows t - (taps-1-tap); taps beyond the kernel's length repeat the token's own row
            const int back = max(taps - 1 - tap, 0);
            const T* row = bcx + static_cast<size_t>(t - back) * ld_bcx;
            bv[tap] = *reinterpret_cast<const raw*>(row + ch);
            xv[tap] = *reinterpret_cast<const raw*>(row + 2 * width + ch);
        }
#pragma unroll
        for (int tap = 0; tap < CONV_VEC_MAX_TAPS; ++tap)
            if (tap < taps) {
#pragma unroll
                for (int i = 0; i < VEC; ++i)
                    conv[i] = fmaf(w[static_cast<size_t>(ch + i) * taps + tap],
                                   ConvVec<T>::at(bv[tap], i) * ConvVec<T>::at(xv[tap], i), conv[i]);
            }
    } else {
        const float* st = state + static_cast<size_t>(seq_slot[s]) * state_slot_stride;
        for (int tap = 0; tap < taps; ++tap) {
            const int q = pos - (taps - 1 - tap);
            if (q < 0) continue;
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                float bx;
                if (q >= start) {
                    const T* row = bcx + static_cast<size_t>(row0 + (q - start)) * ld_bcx;
                    bx = to_float(row[ch + i]) * to_float(row[2 * width + ch + i]);
                } else {
                    bx = st[static_cast<size_t>(q - start + taps) * width + ch + i];
                }
                conv[i] = fmaf(w[static_cast<size_t>(ch + i) * taps + tap], bx, conv[i]);
            }
        }
    }
    raw o;
#pragma unroll
    for (int i = 0; i < VEC; ++i) ConvVec<T>::set(o, i, ConvVec<T>::at(cv, i) * conv[i]);
    *reinterpret_cast<raw*>(out + static_cast<size_t>(t) * width + ch) = o;
}

template <typename T>
__global__ void short_conv_fwd_vec_kernel(
    const T* __restrict__ bcx, int ld_bcx, const float* __restrict__ w,
    const float* __restrict__ bias, const float* __restrict__ state, size_t state_slot_stride,
    T* __restrict__ out, const int* __restrict__ positions, const int* __restrict__ token_seq,
    const int* __restrict__ seq_start, const int* __restrict__ seq_slot,
    const int* __restrict__ cu_seqlens, int width, int taps) {
    const int ch = (blockIdx.y * blockDim.x + threadIdx.x) * ConvVec<T>::n;
    if (ch >= width) return;
    short_conv_token_vec<T>(blockIdx.x, ch, bcx, ld_bcx, w, bias, state, state_slot_stride, out, positions,
                            token_seq, seq_start, seq_slot, cu_seqlens, width, taps);
}

// The same for TT tokens in a row per thread: where they all belong to one request and every
// tap lies in rows of this step, a row's B and x are read once for all the tokens that use it
// (a window that slides down the rows) instead of once per tap.  The sums are formed in the
// same order as above, so the results are the same bits.  The rows are asked for before it is
// known whether the block is of that kind (their addresses do not depend on it).
// This kernel also updates the state, with no kernel behind it: the first taps-1 tokens of a
// request's rows, the only ones that read the old state, are all computed by the block that
// holds the request's first row (also those that lie in the next block, which skips them), and
// the same thread then writes the new state for its channels.  What a block needs beside its own rows
// where requests begin or end in it (their places, old states, last rows, the rows behind the block) is
// asked for without conditions, in two trips to memory: such blocks, one for every two decoding
// requests beside a prompt, set the kernel's time (2,048 rows of 1,024 channels: 20 decoding requests
// and a prompt 14.8 us with a load at a time there, now 7.0; one prompt 9.0, now 5.8; 24 rows 7.1, now 3.3; the taps,
// 16 bytes a load instead of 4, are in these too).
// (2,048 rows of one prompt 4.3 us, with 4 tokens a thread 5.8; beside 20 decoding requests 4.9 and 7.2; 64 decoding
// requests 4.1 and 6.6; 24 rows 3.5 and 5.2: 1,024 channels, three taps, bfloat16, the same rows again and again)
#define CONV_BLOCK_TOKENS 2
typedef float conv_f32x4 __attribute__((ext_vector_type(4)));
template <int VEC>
__device__ __forceinline__ void conv_load(float (&to)[VEC], const float* from) {
#pragma unroll
    for (int i = 0; i < VEC; i += 4) {
        const conv_f32x4 v = *reinterpret_cast<const conv_f32x4*>(from + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) to[i + e] = v[e];
    }
}

template <typename T, int TAPS, int TT>
__global__ __launch_bounds__(256) void short_conv_fwd_block_kernel(
    const T* __restrict__ bcx, int ld_bcx, const float* __restrict__ w,
    const float* __restrict__ bias, float* state, size_t state_slot_stride,
    T* __restrict__ out, const int* __restrict__ token_seq,
    const int* __restrict__ seq_start, const int* __restrict__ seq_slot,
    const int* __restrict__ cu_seqlens, int width, int n_tokens) {
    constexpr int VEC = ConvVec<T>::n;
    typedef typename ConvVec<T>::raw raw;
    const int ch = (blockIdx.y * blockDim.x + threadIdx.x) * VEC;
    if (ch >= width) return;
    // Workgroups go to the chip's 8 dies in turn, and each die has an L2 of its own: die d takes a
    // run of tokens, so that the rows two neighbouring workgroups both read (the taps before a
    // workgroup's first token) come from memory once, not once for each of two dies.  (The grid is
    // 8 runs of gridDim.x / 8 workgroups; those beyond the last token have nothing to do.)
    const int per_die = gridDim.x >> 3;
    const int t0 = ((blockIdx.x & 7) * per_die + (blockIdx.x >> 3)) * TT;
    if (t0 >= n_tokens) return;
    const int n = min(TT, n_tokens - t0);
    // (asked for ahead of the rows; what depends on it is asked for while the rows are on their way)
    int seq[TT];
#pragma unroll
    for (int j = 0; j < TT; ++j) seq[j] = token_seq[min(t0 + j, n_tokens - 1)];
    auto load_row = [&](int t, raw& bv, raw& xv) __attribute__((always_inline)) {
        const T* row = bcx + static_cast<size_t>(min(max(t, 0), n_tokens - 1)) * ld_bcx;
        bv = *reinterpret_cast<const raw*>(row + ch);
        xv = *reinterpret_cast<const raw*>(row + 2 * width + ch);
    };
    auto load_gate = [&](int t) __attribute__((always_inline)) {
        return *reinterpret_cast<const raw*>(bcx + static_cast<size_t>(min(t, n_tokens - 1)) * ld_bcx + width + ch);
    };
    raw bv[TT + TAPS - 1], xv[TT + TAPS - 1], cv[TT];
#pragma unroll
    for (int j = 0; j < TT + TAPS - 1; ++j) load_row(t0 - (TAPS - 1) + j, bv[j], xv[j]);
#pragma unroll
    for (int j = 0; j < TT; ++j) cv[j] = load_gate(t0 + j);
    float taps_flat[VEC * TAPS], b0[VEC];        // tap of channel ch + i: [i * TAPS + tap]
    conv_load<VEC * TAPS>(taps_flat, w + static_cast<size_t>(ch) * TAPS);
#pragma unroll
    for (int i = 0; i < VEC; ++i) b0[i] = bias ? bias[ch + i] : 0.f;
    auto store = [&](int t, const raw& gate, const float (&conv)[VEC]) __attribute__((always_inline)) {
        raw o;
#pragma unroll
        for (int i = 0; i < VEC; ++i) ConvVec<T>::set(o, i, ConvVec<T>::at(gate, i) * conv[i]);
        *reinterpret_cast<raw*>(out + static_cast<size_t>(t) * width + ch) = o;
    };
    // the same for the whole workgroup
    if (n < TT || seq[TT - 1] != seq[0] || t0 - (TAPS - 1) < cu_seqlens[seq[0]]) {
        // the requests of the block's rows
        int first[TT], last[TT], start[TT], slot[TT];
#pragma unroll
        for (int j = 0; j < TT; ++j) {
            first[j] = cu_seqlens[seq[j]];
            last[j] = cu_seqlens[seq[j] + 1];
            start[j] = seq_start[seq[j]];
            slot[j] = seq_slot[seq[j]];
        }
        // rows behind the block that may read an old state (rows 1 .. TAPS-2 of a request that begins at its end)
        constexpr int EXT = TAPS - 2;
        raw ebv[EXT > 0 ? EXT : 1], exv[EXT > 0 ? EXT : 1], ecv[EXT > 0 ? EXT : 1];
#pragma unroll
        for (int e = 0; e < EXT; ++e) {
            load_row(t0 + TT + e, ebv[e], exv[e]);
            ecv[e] = load_gate(t0 + TT + e);
        }
        // every row's request: its old state, and the last rows it brings
        float old[TT][TAPS][VEC];
        raw lbv[TT][TAPS], lxv[TT][TAPS];
#pragma unroll
        for (int j = 0; j < TT; ++j) {
            const float* st = state + static_cast<size_t>(slot[j]) * state_slot_stride + ch;
#pragma unroll
            for (int k = 0; k < TAPS; ++k) {
                conv_load<VEC>(old[j][k], st + static_cast<size_t>(k) * width);
                load_row(max(last[j] - TAPS + k, first[j]), lbv[j][k], lxv[j][k]);
            }
        }
        // B x at `back` rows before row `at` of the request of row j: a row of the step (row r of the window
        // t0 - (TAPS-1) ..), an old entry, or zero before position 0
        auto window = [&](int r, int i) __attribute__((always_inline)) {       // r is known when this is compiled
            return r < TT + TAPS - 1 ? ConvVec<T>::at(bv[r], i) * ConvVec<T>::at(xv[r], i)
                                     : ConvVec<T>::at(ebv[r - (TT + TAPS - 1) < EXT ? r - (TT + TAPS - 1) : 0], i) *
                                           ConvVec<T>::at(exv[r - (TT + TAPS - 1) < EXT ? r - (TT + TAPS - 1) : 0], i);
        };
        auto token = [&](int j, int u, const raw& gate) __attribute__((always_inline)) {     // row t0 + u, of row j's request
            const int at = t0 + u - first[j];
            float conv[VEC];
#pragma unroll
            for (int i = 0; i < VEC; ++i) conv[i] = b0[i];
#pragma unroll
            for (int tap = 0; tap < TAPS; ++tap) {
                const int from = at - (TAPS - 1 - tap);          // < 0: entry from + TAPS of the old state
                // (positions before 0 add nothing, not even a zero: the sum of a short sequence keeps its bits)
                if (start[j] + from < 0) continue;
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    float bx = window(u + tap, i);
#pragma unroll
                    for (int k = 1; k < TAPS; ++k) bx = from + TAPS == k ? old[j][k][i] : bx;
                    conv[i] = fmaf(taps_flat[i * TAPS + tap], bx, conv[i]);
                }
            }
            store(t0 + u, gate, conv);
        };
#pragma unroll
        for (int j = 0; j < TT; ++j) {
            if (j >= n) continue;
            // (the block of the request's first row has those of its rows that read the old state)
            if (first[j] >= t0 || t0 + j - first[j] >= TAPS - 1) token(j, j, cv[j]);
        }
#pragma unroll
        for (int j = 0; j < TT; ++j) {
            if (j >= n || first[j] != t0 + j) continue;          // requests that begin in this block:
#pragma unroll
            for (int e = 0; e < EXT; ++e)                        // their rows in the next block that read the old state,
                if (t0 + TT + e < min(t0 + j + TAPS - 1, last[j])) token(j, TT + e, ecv[e]);
            // then the new state: entry k is B x at position end - TAPS + k
            const int rows = last[j] - first[j];
            float* st = state + static_cast<size_t>(slot[j]) * state_slot_stride + ch;
#pragma unroll
            for (int k = 0; k < TAPS; ++k) {
                const int from = rows - TAPS + k;                // < 0: entry from + TAPS of the old state
                float v[VEC];
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    v[i] = ConvVec<T>::at(lbv[j][k], i) * ConvVec<T>::at(lxv[j][k], i);
#pragma unroll
                    for (int m = 1; m < TAPS; ++m) v[i] = from + TAPS == m && from < 0 ? old[j][m][i] : v[i];
                    if (start[j] + from < 0) v[i] = 0.f;
                }
#pragma unroll
                for (int i = 0; i < VEC; i += 4)
                    *reinterpret_cast<conv_f32x4*>(st + static_cast<size_t>(k) * width + i) = conv_f32x4{v[i], v[i + 1], v[i + 2], v[i + 3]};
            }
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < TT; ++j) {
        float conv[VEC];
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
            conv[i] = b0[i];
#pragma unroll
            for (int tap = 0; tap < TAPS; ++tap)
                conv[i] = fmaf(taps_flat[i * TAPS + tap], ConvVec<T>::at(bv[j + tap], i) * ConvVec<T>::at(xv[j + tap], i), conv[i]);
        }
        store(t0 + j, cv[j], conv);
    }
}

template <typename T>
__global__ void short_conv_state_kernel(
    const T* __restrict__ bcx, int ld_bcx, float* __restrict__ state, size_t state_slot_stride,
    const int* __restrict__ seq_start, const int* __restrict__ seq_slot,
    const int* __restrict__ cu_seqlens, int width, int taps) {
    const int ch = blockIdx.y * blockDim.x + threadIdx.x;
    if (ch >= width) return;
    const int s = blockIdx.x;
    const int start = seq_start[s];
    const int row0 = cu_seqlens[s];
    const int n = cu_seqlens[s + 1] - row0;
    const int end = start + n;
    float* st = state + static_cast<size_t>(seq_slot[s]) * state_slot_stride;
    // ascending j: an old entry is read at index j + n > j, before it is overwritten
    for (int j = 0; j < taps; ++j) {
        const int q = end - taps + j;
        float v = 0.f;
        if (q >= start) {
            const T* row = bcx + static_cast<size_t>(row0 + (q - start)) * ld_bcx;
            v = to_float(row[ch]) * to_float(row[2 * width + ch]);
        } else if (q >= 0) {
            v = st[static_cast<size_t>(q - start + taps) * width + ch];
        }
        st[static_cast<size_t>(j) * width + ch] = v;
    }
}

// For tests and tuning: 4 tokens a thread in the kernel for long steps instead of CONV_BLOCK_TOKENS (0: the default).
static int g_force_block_tokens = 0;
extern "C" void celeg_short_conv_force_block_tokens(int tokens) { g_force_block_tokens = tokens; }

extern "C" int celeg_short_conv(const void* bcx, int ld_bcx, int dtype, const float* w,
                                const float* bias, float* state, size_t state_slot_stride,
                                void* out, const int* positions, const int* token_seq,
                                const int* seq_start, const int* seq_slot, const int* cu_seqlens,
                                int n_tokens, int n_seqs, int width, int taps,
                                hipStream_t stream) {
    if (n_tokens <= 0 || n_seqs <= 0) return 0;
    dim3 block(256);
    dim3 grid_fwd(n_tokens, (width + 255) / 256), grid_state(n_seqs, (width + 255) / 256);
    const int vec = dtype == CELEG_F32 ? 4 : 8;
    const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    if (n_tokens >= 16 && taps <= CONV_VEC_MAX_TAPS && width % vec == 0 && ld_bcx % vec == 0 &&
        aligned(bcx) && aligned(out)) {
        const int threads = min(256, (width / vec + 63) / 64 * 64);
        dim3 vblock(threads), vgrid(n_tokens, (width / vec + threads - 1) / threads);
        if (taps >= 2 && taps <= 4 && aligned(w) && aligned(state) && state_slot_stride % 4 == 0) {      // (n_tokens >= 16 here)
            const int tt = g_force_block_tokens == 4 ? 4 : CONV_BLOCK_TOKENS;
            dim3 bgrid(((n_tokens + tt - 1) / tt + 7) / 8 * 8, vgrid.y);      // (8 runs of tokens, one a die)
#define CELEG_CONV_BLOCK(T_, TAPS_)                                                                \
    if (tt == 4) CELEG_CONV_BLOCK_TT(T_, TAPS_, 4); else CELEG_CONV_BLOCK_TT(T_, TAPS_, CONV_BLOCK_TOKENS)
#define CELEG_CONV_BLOCK_TT(T_, TAPS_, TT_)                                                        \
    hipLaunchKernelGGL((short_conv_fwd_block_kernel<T_, TAPS_, TT_>), bgrid, vblock, 0, stream,     \
                       static_cast<const T_*>(bcx), ld_bcx, w, bias, state, state_slot_stride,      \
                       static_cast<T_*>(out), token_seq, seq_start, seq_slot, cu_seqlens, width, n_tokens)
#define CELEG_CONV_BLOCK_T(T_)                                                                     \
    if (taps == 2) { CELEG_CONV_BLOCK(T_, 2); } else if (taps == 3) { CELEG_CONV_BLOCK(T_, 3); }     \
    else { CELEG_CONV_BLOCK(T_, 4); }
            if (dtype == CELEG_F32) { CELEG_CONV_BLOCK_T(float) } else { CELEG_CONV_BLOCK_T(bf16) }
#undef CELEG_CONV_BLOCK_T
#undef CELEG_CONV_BLOCK_TT
#undef CELEG_CONV_BLOCK
            return CELEG_LAUNCH_RESULT();
        }
        if (dtype == CELEG_F32) {
            hipLaunchKernelGGL(short_conv_fwd_vec_kernel<float>, vgrid, vblock, 0, stream,
                               static_cast<const float*>(bcx), ld_bcx, w, bias, state,
                               state_slot_stride, static_cast<float*>(out), positions, token_seq,
                               seq_start, seq_slot, cu_seqlens, width, taps);
            hipLaunchKernelGGL(short_conv_state_kernel<float>, grid_state, block, 0, stream,
                               static_cast<const float*>(bcx), ld_bcx, state, state_slot_stride,
                               seq_start, seq_slot, cu_seqlens, width, taps);
        } else {
            hipLaunchKernelGGL(short_conv_fwd_vec_kernel<bf16>, vgrid, vblock, 0, stream,
                               static_cast<const bf16*>(bcx), ld_bcx, w, bias, state,
                               state_slot_stride, static_cast<bf16*>(out), positions, token_seq,
                               seq_start, seq_slot, cu_seqlens, width, taps);
            hipLaunchKernelGGL(short_conv_state_kernel<bf16>, grid_state, block, 0, stream,
                               static_cast<const bf16*>(bcx), ld_bcx, state, state_slot_stride,
                               seq_start, seq_slot, cu_seqlens, width, taps);
        }
        return CELEG_LAUNCH_RESULT();
    }
    if (dtype == CELEG_F32) {
        hipLaunchKernelGGL(short_conv_fwd_kernel<float>, grid_fwd, block, 0, stream,
                           static_cast<const float*>(bcx), ld_bcx, w, bias, state,
                           state_slot_stride, static_cast<float*>(out), positions, token_seq,
                           seq_start, seq_slot, cu_seqlens, width, taps);
        hipLaunchKernelGGL(short_conv_state_kernel<float>, grid_state, block, 0, stream,
                           static_cast<const float*>(bcx), ld_bcx, state, state_slot_stride,
                           seq_start, seq_slot, cu_seqlens, width, taps);
    } else {
        hipLaunchKernelGGL(short_conv_fwd_kernel<bf16>, grid_fwd, block, 0, stream,
                           static_cast<const bf16*>(bcx), ld_bcx, w, bias, state,
                           state_slot_stride, static_cast<bf16*>(out), positions, token_seq,
                           seq_start, seq_slot, cu_seqlens, width, taps);
        hipLaunchKernelGGL(short_conv_state_kernel<bf16>, grid_state, block, 0, stream,
                           static_cast<const bf16*>(bcx), ld_bcx, state, state_slot_stride,
                           seq_start, seq_slot, cu_seqlens, width, taps);
    }
    return CELEG_LAUNCH_RESULT();
}
