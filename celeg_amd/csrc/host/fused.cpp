// Helpers of the fused path for steps of few rows (decode and small portions) and, with the
// tiled products, of many rows.  See parts.hpp.
#include "parts.hpp"

namespace celeg {
namespace fused {

// Whether products of `rows` rows that read a stream of this width take the fused path through
// the tiled products (otherwise they run the library's products with separate norm and activation
// kernels).  The choice is by the sizes of the products, not by the model: Runtime::tiled_max_width
// holds the widest stream for which the tiled products were measured faster.  (Whole prompts of wider models are faster on the tiles
// too at some numbers of rows, width 2,048 2 to 16 % up to 1,024 rows and from 1,600 on; but the weights with a norm's folded in
// are rounded to bfloat16 once more: logits of three prompts of 1,000 to 2,000 tokens 0.016 of the result away from 64 bits with
// them and 0.0147 without.  So they stay with the library.)
bool tiled_step(const Runtime& rt, int rows, long long width) {
    return rows > FUSED_MAX_ROWS && width <= rt.tiled_max_width && rt.dtype == DType::BF16 && rt.use_fused;
}

// Whether so many rows can take the fused path through products with these inner sizes.
bool rows_ok(const Runtime& rt, int rows, std::initializer_list<long long> inner) {
    long long widest = 0;
    for (long long k : inner) widest = std::max(widest, k);
    if (rows > FUSED_MAX_ROWS)
        // every inner size is also the width of some product's output
        // (the first inner size is the width of the stream)
        return inner.size() > 0 && tiled_step(rt, rows, *inner.begin()) && rt.ops.tiled_linear_ok(rows, 4, inner) &&
               widest <= 64 * TILED_MAX_STAT_BLOCKS;
    if (!(rt.dtype == DType::BF16 && rt.use_fused && rt.ops.fused_linear_ok(rows, inner))) return false;
    int limit = rt.fused_max_rows;
    if (limit < 0) limit = rt.ops.rows_kernel_ok(rows, inner) ? FUSED_MAX_ROWS : FUSED_MAX_ROWS_OLD_KERNEL;
    return rows <= limit;
}

// The same for the rows of a step.  Rows that are left of a step of many (Runtime::wanted) take it only where all of that step's rows
// do: the fused path multiplies a norm's weight into the product's, which rounds that to bfloat16 once more, and what a prompt's
// logits are made of does not hang on how many of them are wanted.
bool fused_rows_ok(const Runtime& rt, const StepBatch& batch, std::initializer_list<long long> inner) {
    if (rt.wanted.stream.defined() && !rows_ok(rt, rt.wanted.step_rows, inner)) return false;
    return rows_ok(rt, batch.n_tokens, inner);
}

bool fused_f32_ok(const Runtime& rt, const StepBatch& batch, std::initializer_list<long long> inner) {
    return rt.dtype == DType::F32 && rt.use_fused && Ops::fused_linear_f32_ok(batch.n_tokens, inner);
}

Tensor stream_stats(Runtime& rt, long long width, int rows) {
    if (rows > STAT_COLUMNS)     // a step of many rows: one partial sum per tile of columns
        return rt.ws.buf("stream_stats_many", DType::F32, {rows, TILED_MAX_STAT_BLOCKS});
    // up to one partial sum per 4 columns (the products for few rows use narrow workgroups)
    return rt.ws.buf("stream_stats", DType::F32, {STAT_COLUMNS, (width + 3) / 4});
}

// Room for a bfloat16 operand of the fused products, [rows, width] (up to 16 rows, or sizes the
// kernel for 9 to 64 rows does not take) or the view [rows, width/8, 8] of [width/8, 64, 8]: the
// rows side by side inside every group of 8 values, the layout that the kernel for 9 to 64 rows
// reads whole runs of memory from, where that kernel both reads it and, if a product writes it
// (inner size producer_inner), writes it.
Tensor operand_rows(Runtime& rt, const std::string& name, int rows, long long width,
                    std::initializer_list<long long> producer_inner) {
    if (rows > STAT_COLUMNS) return rt.ws.buf(name + "_many", DType::BF16, {rows, width});
    bool side_by_side = rt.ops.rows_kernel_ok(rows, {width});
    for (long long k : producer_inner) side_by_side = side_by_side && rt.ops.rows_kernel_ok(rows, {k});
    if (side_by_side) {
        Tensor t = rt.ws.buf(name + "_side_by_side", DType::BF16, {width / 8, STAT_COLUMNS, 8});
        Tensor view;
        view.data = t.data;
        view.dtype = DType::BF16;
        view.ndim = 3;
        view.shape[0] = rows;
        view.shape[1] = width / 8;
        view.shape[2] = 8;
        view.stride[0] = 8;
        view.stride[1] = STAT_COLUMNS * 8;
        view.stride[2] = 1;
        return view;
    }
    return rt.ws.buf(name, DType::BF16, {STAT_COLUMNS, width}).rows(0, rows);
}

// Both layouts of such an operand for up to 64 rows: made at one's first need, they would have recorded steps recorded again.
void operand_room(Runtime& rt, const std::string& name, long long width, std::initializer_list<long long> producer_inner) {
    operand_rows(rt, name, 1, width, producer_inner);
    operand_rows(rt, name, FUSED_MAX_ROWS, width, producer_inner);
}

// The bfloat16 copy of the residual stream that products behind a norm read.
Tensor stream_bf16(Runtime& rt, int rows, long long width) { return operand_rows(rt, "stream_bf16", rows, width, {}); }

// Whether a product of `rows` bfloat16 rows with this inner size takes the form with the norm
// folded into the weights (the kernels for up to 16 and for 9 to 64 rows).
bool sliced(const Runtime& rt, int rows, long long inner) {
    if (rt.ops.rows_kernel_ok(rows, {inner})) return true;
    return rows <= SLICED_MAX_ROWS && rt.ops.use_sliced;
}

namespace {
// w with the norm's weight multiplied into its columns, (x * nw) w^T = x (w * nw)^T, in the
// layout the products for few rows read best.  Made once per (weight, norm) pair and kept.
std::shared_ptr<DeviceTensor> folded_weight(Runtime& rt, const Tensor& w, const Tensor& norm_weight, bool* packed) {
    *packed = w.shape[1] % 32 == 0;
    const auto key = std::make_pair(static_cast<const void*>(w.data), static_cast<const void*>(norm_weight.data));
    auto it = rt.folded_weights.find(key);
    if (it == rt.folded_weights.end()) it = rt.folded_weights.emplace(key, rt.ops.fold_weight(w, &norm_weight, *packed)).first;
    return it->second;
}
std::shared_ptr<DeviceTensor> folded_plain_weight(Runtime& rt, const Tensor& w, const Tensor& norm_weight) {
    const auto key = std::make_pair(static_cast<const void*>(w.data), static_cast<const void*>(norm_weight.data));
    auto it = rt.folded_plain_weights.find(key);
    if (it == rt.folded_plain_weights.end())
        it = rt.folded_plain_weights.emplace(key, rt.ops.fold_weight(w, &norm_weight, false)).first;
    return it->second;
}
// a copy of w in the layout the products for few rows read best; made once
std::shared_ptr<DeviceTensor> packed_weight(Runtime& rt, const Tensor& w) {
    auto it = rt.packed_weights.find(w.data);
    if (it == rt.packed_weights.end()) it = rt.packed_weights.emplace(w.data, rt.ops.fold_weight(w, nullptr, true)).first;
    return it->second;
}
// the rows of a product that reads its weights as they are stored, behind their norm
Tensor rows_as_stored(Runtime& rt, long long width) { return rt.ws.buf("normed_as_stored", DType::BF16, {STAT_COLUMNS, width}); }
}  // namespace

bool qkv_tail_ok(const Runtime& rt, int rows, long long width) { return tiled_step(rt, rows, width); }

// (the two kernels that take the stream's bfloat16 copy; not the older form for very many columns)
bool activation_ok(const Runtime& rt, int rows, long long width, long long columns) {
    return rows <= FUSED_MAX_ROWS && !tiled_step(rt, rows, width) && sliced(rt, rows, width) &&
           (rt.ops.rows_kernel_ok(rows, {width}) || columns <= SLICED_MAX_COLUMNS);
}

void norm_linear(Runtime& rt, const Tensor& h, const Norm::Foldable& norm, const Tensor& w, const Tensor& out,
                 Epilogue epilogue, const LinearExtras& extras) {
    int blocks = rt.stream_stat_blocks;
    const int T = static_cast<int>(h.shape[0]);
    const long long width = h.shape[1];
    const int M = extras.n_rows >= 0 ? extras.n_rows : T;
    if (rt.dtype == DType::F32) {
        if (extras.rows || extras.qkv || w.dtype != DType::F32) throw KernelError("norm_linear: not a 32-bit product with a norm");
        FusedArgs args;
        args.epilogue = epilogue;
        args.norm_weight = norm.weight;
        args.eps = norm.eps;
        args.bias = extras.bias;
        args.conv = extras.conv;
        rt.ops.fused_linear_f32(h, w, out, args);
        return;
    }
    if (tiled_step(rt, T, width)) {
        if (extras.rows || (epilogue != Epilogue::Store && epilogue != Epilogue::Swiglu) || w.dtype != DType::BF16)
            throw KernelError("norm_linear: not a product of the path for many rows");
        Tensor stats = stream_stats(rt, width, T);
        Tensor xb = stream_bf16(rt, T, width);
        if (!(blocks > 0 && blocks <= TILED_MAX_STAT_BLOCKS && rt.stream_has_bf16)) {
            rt.ops.stream_prepare(h, xb, stats);
            rt.stream_stat_blocks = blocks = 1;
            rt.stream_has_bf16 = true;
        }
        rt.ops.tiled_linear(xb, folded_plain_weight(rt, w, norm.weight)->view, out, epilogue, norm.eps, &stats, blocks,
                            extras.bias.defined() ? &extras.bias : nullptr, nullptr, nullptr, extras.qkv);
        return;
    }
    if (extras.qkv) throw KernelError("norm_linear: the q/k/v tail goes with steps of many rows");
    const int streams = epilogue == Epilogue::Swiglu ? 2 : epilogue == Epilogue::Conv || epilogue == Epilogue::ConvRows ? 3 : 1;
    const bool streamed = rt.ops.rows_kernel_ok(M, {width});
    FusedArgs args;
    args.epilogue = epilogue;
    args.eps = norm.eps;
    args.rows = extras.rows;
    args.n_rows = extras.n_rows;
    args.bias = extras.bias;
    args.conv = extras.conv;
    args.activation = extras.activation;
    args.row_best = extras.row_best;
    args.row_best_ld = extras.row_best_ld;
    args.row_best_rows = extras.row_best_rows;
    rt.ops.last_best_parts = 0;
    const bool folds = sliced(rt, M, width) && w.dtype == DType::BF16 && (streamed || w.shape[0] / streams <= SLICED_MAX_COLUMNS);
    if (folds && extras.as_stored) {
        const Tensor normed = rows_as_stored(rt, width).rows(0, M);
        rt.ops.rmsnorm(h, norm.weight, norm.eps, normed, nullptr, extras.rows);
        args.rows = nullptr;
        args.plain = true;
        rt.ops.fused_linear(normed, w, out, args);
        return;
    }
    if (folds) {
        // the stream's bfloat16 copy times the weight with the norm's weight folded in, scaled
        // by the rows' 1/rms at the end
        Tensor stats = stream_stats(rt, width);
        Tensor xb = stream_bf16(rt, T, width);
        if (xb.ndim == 3 && !streamed) {
            // few wanted rows of a step of many: the kernel for few rows reads rows that lie one
            // after the other, so the stream gets such a copy too
            xb = rt.ws.buf("stream_bf16", DType::BF16, {STAT_COLUMNS, width}).rows(0, T);
            rt.ops.stream_prepare(h, xb, stats);
            rt.stream_stat_blocks = blocks = 1;
        } else if (!(blocks > 0 && blocks <= SLICED_MAX_STAT_BLOCKS && rt.stream_has_bf16)) {
            rt.ops.stream_prepare(h, xb, stats);
            rt.stream_stat_blocks = blocks = 1;
            rt.stream_has_bf16 = true;
        }
        bool packed = false;
        auto folded = folded_weight(rt, w, norm.weight, &packed);
        args.stats = stats;
        args.stat_blocks = blocks;
        args.packed = packed;
        rt.ops.fused_linear(xb, folded->view, out, args);
        return;
    }
    args.norm_weight = norm.weight;
    if (blocks) args.stats = stream_stats(rt, width);
    args.stat_blocks = blocks;
    if (w.dtype == DType::BF16 && w.ndim == 2 && w.shape[1] % 32 == 0 && w.shape[1] >= 2048 &&
        w.shape[0] / streams > SLICED_MAX_COLUMNS && !extras.as_stored) {
        // a product of very many long weight rows (the output head of a wide model): a copy of w in
        // blocks of 32 values of k with the rows side by side, which the kernel reads whole kilobytes
        // of; made once and kept (65,536 rows of 2,048 values at 8 rows: 54.6 against 62.4 us; of 1,024
        // values: 29.3 against 29.5, not worth a second copy of the table; nor is a prompt's one product)
        args.packed = true;
        rt.ops.fused_linear(h, packed_weight(rt, w)->view, out, args);
        return;
    }
    rt.ops.fused_linear(h, w, out, args);
}

// Leaves all rows but the wanted ones (Runtime::wanted): rt.wanted.stream gets theirs of h, and the result is theirs of `a`
// (nothing where there is no `a`), laid out as products of so few rows read them where `operand` says that one does.
Tensor keep_wanted_rows(Runtime& rt, const Tensor& h, const Tensor& a, bool operand) {
    Runtime::WantedRows& wanted = rt.wanted;
    wanted.pending = false;
    // Sizes that go by the step's rows, as those of all its buffers do, and not by how many are wanted: the first step of many rows
    // makes what later ones of no more rows need, and steps recorded behind it stay good.
    const long long width = h.shape[1], room = std::max<long long>(wanted.step_rows / 2, STAT_COLUMNS);
    wanted.stream = rt.ws.buf("wanted_stream", DType::F32, {room, width}).rows(0, wanted.n);
    rt.stream_stat_blocks = 0;
    rt.stream_has_bf16 = false;
    if (rt.dtype == DType::BF16) rows_as_stored(rt, width);      // (the head's)
    Tensor few;
    if (a.defined() && operand && rt.dtype == DType::BF16) {
        operand_room(rt, "wanted_operand", a.shape[1], {});
        operand_room(rt, "stream_bf16", width, {});
        stream_stats(rt, width);
        few = rt.ws.buf("wanted_operand_many", DType::BF16, {room, a.shape[1]}).rows(0, wanted.n);
        if (wanted.n <= FUSED_MAX_ROWS) few = operand_rows(rt, "wanted_operand", wanted.n, a.shape[1], {});
    } else if (a.defined()) {
        few = rt.ws.buf("wanted_branch", rt.dtype, {room, a.shape[1]}).rows(0, wanted.n);
    }
    rt.ops.gather_rows(h, a.defined() ? &a : nullptr, wanted.rows, wanted.n, wanted.stream, few.defined() ? &few : nullptr);
    return few;
}

void linear_into_stream(Runtime& rt, const Tensor& a, const Tensor& w, const Tensor& h, const Tensor* bias) {
    const int T = static_cast<int>(h.shape[0]);
    const long long width = h.shape[1];
    if (rt.wanted.pending && a.ndim == 2) {
        if (rt.wanted.n == 0) return;
        StepBatch few;
        few.n_tokens = rt.wanted.n;
        if (rows_ok(rt, few.n_tokens, {width, a.shape[1]}) || fused_f32_ok(rt, few, {width, a.shape[1]})) {
            const Tensor rows = keep_wanted_rows(rt, h, a, true);
            linear_into_stream(rt, rows, w, rt.wanted.stream, bias);
            return;
        }
    }
    if (rt.dtype == DType::F32) {
        FusedArgs args;
        args.epilogue = Epilogue::Residual;
        if (bias) args.bias = *bias;
        rt.ops.fused_linear_f32(a, w, h, args);
        rt.stream_stat_blocks = 0;
        rt.stream_has_bf16 = false;
        return;
    }
    if (tiled_step(rt, T, width)) {
        Tensor stats = stream_stats(rt, width, T);
        Tensor xb = stream_bf16(rt, T, width);
        const bool packed = w.dtype == DType::BF16 && Ops::tiled_packed(T, static_cast<int>(width), static_cast<int>(w.shape[1]));
        rt.ops.tiled_linear(a, packed ? packed_weight(rt, w)->view : w, h, Epilogue::Residual, 0.f, nullptr, 0, bias, &stats, &xb);
        rt.stream_stat_blocks = rt.ops.last_stat_blocks;
        rt.stream_has_bf16 = true;
        return;
    }
    Tensor stats = stream_stats(rt, width);
    const long long inner = a.ndim == 3 ? a.shape[1] * 8 : a.shape[1];
    const bool is_sliced = sliced(rt, T, inner);
    Tensor xb;
    if (is_sliced) {
        xb = stream_bf16(rt, T, width);
        // this product's kernel writes rows one after the other only: the next norm prepares the copy
        if (xb.ndim == 3 && !rt.ops.rows_kernel_ok(T, {inner})) xb = Tensor();
    }
    FusedArgs args;
    args.epilogue = Epilogue::Residual;
    if (bias) args.bias = *bias;
    args.stats_out = stats;
    args.out_bf16 = xb;
    const bool pack = is_sliced && w.shape[1] % 32 == 0;
    args.packed = pack;
    rt.ops.fused_linear(a, pack ? packed_weight(rt, w)->view : w, h, args);
    rt.stream_stat_blocks = rt.ops.last_stat_blocks;
    rt.stream_has_bf16 = xb.defined();
}

}  // namespace fused
}  // namespace celeg
