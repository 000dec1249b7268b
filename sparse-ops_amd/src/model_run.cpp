// SparseOnnxModel: buffer sizing and execution.  The reference walks the layers
// with a name->buffer map and allocates every output per call
// (src/model_run.cpp:3-140, src/layers/*.cpp); here every tensor has a fixed slot
// in one HBM arena, the chain is recorded once into a launch graph, and a call
// with an unchanged batch size allocates nothing.
#include "sparse_onnx.hpp"

#include <algorithm>
#include <cstdlib>
#include <stdexcept>

#include "model_impl.hpp"
#include "rbm_conv.hpp"

using namespace sparseops;

void SparseOnnxModel::resize_buffers(uint32_t batch)
{
    Impl &M = *impl_;
    if (batch == 0) throw std::runtime_error("resize_buffers: batch must be positive");
    so_ctx *ctx = context();
    std::lock_guard<std::mutex> lock(context_mutex());
    if (M.graph) { so_graph_free(ctx, M.graph); M.graph = nullptr; }
    M.has_conv = false;
    uint64_t pixels = 0;                       // of the largest convolution's output
    for (const LayerPlan &L : M.layers) {
        M.has_conv |= L.conv != nullptr;
        if (L.conv) pixels = std::max(pixels, uint64_t(L.cg.H_out) * L.cg.W_out);
    }
    // The convolutions work on batch tiles of 16, 8 or 4 entries, and the larger the tile the less a
    // batch entry costs: a batch is carried in rows of 4 (2 to 4 entries), 8 (up to 8) or the next
    // multiple of 16 (the extra columns are zeros on input and are never copied out; batch entries
    // do not interact).  Measured on a ResNet-18-shaped stack: 12 entries as 12 0.86 ms, as 16
    // 0.76 ms; 24 as 24 1.31 ms, as 32 1.24 ms.  One and two entries have a kernel of their own: one entry 0.35 ms as 4, 0.22
    // as 1; two as 4 / as 2, us, ResNet-18-shaped stacks: 224 x 224 of width 64 314 / 272, 48 273 / 219, 16 124 / 110, 64 x 64 of 16 102 / 91, but
    // 384 x 384 of 32 271 / 278, 448 x 448 of 64 632 / 672, 512 x 512 of 16 200 / 197: as 2 up to 128 x 128 outputs (a stride of two on 256 x 256).
    // Seven stacks of stride-1 layers and halvings (VGG-shaped, 32 x 32 to 128 x 128, width 16 to 64), layers alone: as 2 takes 0.76 to 0.95 of as 4, of
    // 256 x 256 1.09.  A single layer may lose, most where the gather kernel takes it at 2: 7x7/2 from 224 x 224, 32 channels, 20.5 / 11.4, 3x3 64
    // channels at 128 x 128 with rows of 58 35 / 21; by estimates of every layer nets of one to eight drawn layers would gain 0.3 %.
    uint32_t pbatch = batch;
    if (M.has_conv && batch > 1 && !(batch == 2 && pixels <= 128u * 128u)) pbatch = batch <= 4 ? 4u : batch <= 8 ? 8u : (batch + 15u) / 16u * 16u;
    // Slot offsets for this batch, 256-byte aligned.
    std::size_t total = 0;
    std::size_t widest = std::max(M.in_features, M.out_features);
    for (Slot &s : M.slots) {
        s.offset = total;
        total += (s.features * pbatch + 63) / 64 * 64;
    }
    M.arena.reserve(total * sizeof(float));
    M.stage_in.reserve(M.in_features * batch * sizeof(float));
    M.stage_out.reserve(M.out_features * batch * sizeof(float));
    if (pbatch != batch) M.stage_mid.reserve(widest * batch * sizeof(float));
    M.batch = batch;
    M.pbatch = pbatch;
    for (const LayerPlan &L : M.layers) {
        if (L.conv) check(so_conv_plan_tune(ctx, L.conv, pbatch), "so_conv_plan_tune");
        // whatever so_matmul would allocate at this batch is allocated now (run() allocates nothing, and a
        // launch graph cannot be recorded across an allocation)
        else if (L.op == Op::MatMul && L.dE) check(so_matmul_reserve(ctx, L.dE, pbatch), "so_matmul_reserve");
    }
    M.set_conv_rbm();
    if (!M.layers.empty() && M.record_pays()) {
        check(so_graph_begin(ctx), "so_graph_begin");
        try {
            M.enqueue_layers();
        } catch (...) {
            so_graph *g = nullptr;
            so_graph_end(ctx, &g);
            so_graph_free(ctx, g);
            throw;
        }
        check(so_graph_end(ctx, &M.graph), "so_graph_end");
    }
}

// The reference builds its row-block-merged plan for wide convolutions at load (src/sparse_onnx.cpp:499-502: Cout >= 32 and
// K >= 64, blocks of 8 channels) and never runs it.  Here it is built where SPARSEOPS_CONV_RBM=1 asks for its kernel, which the
// windowed one beats: looked at by the loader's and every later resize_buffers, as the other overrides are.
void SparseOnnxModel::Impl::set_conv_rbm()
{
    const char *env = std::getenv("SPARSEOPS_CONV_RBM");
    const bool asked = env && env[0] == '1';
    so_ctx *ctx = context();
    for (LayerPlan &L : layers) {
        if (!L.conv || L.cg.Cout < 32 || L.E->n < 64 || asked == (L.rbm != nullptr)) continue;
        if (asked) L.rbm = upload_rbm(build_rbm_from_ellpack(*L.E, nullptr, 8));
        check(so_conv_plan_set_rbm(ctx, L.conv, asked ? L.rbm : nullptr), "so_conv_plan_set_rbm");
        if (!asked) { so_rbm_free(ctx, L.rbm); L.rbm = nullptr; }
    }
}

bool SparseOnnxModel::recorded() const { return impl_->graph != nullptr; }

std::size_t SparseOnnxModel::Impl::output_layer() const
{
    for (std::size_t i = layers.size(); i > 0; --i)
        if (layers[i - 1].out == output_slot) return i - 1;
    return layers.size();
}

void SparseOnnxModel::Impl::enqueue_layers(const float *in, float *out) const
{
    so_ctx *ctx = context();
    const uint32_t B = pbatch;
    // Every layer reads and writes arena slots.  The input's slot holds nothing else.  A slot is shared by all tensors whose lifetimes do
    // not overlap, so the output's is the output only from the last layer that writes it on.
    const std::size_t made = output_layer();
    std::size_t at = 0;
    auto src = [&](int s) -> const float * { return in && s == input_slot ? in : out && at > made && s == output_slot ? out : slot_ptr(s); };
    auto dst = [&](int s) -> float * { return out && at == made ? out : slot_ptr(s); };
    // A convolution and the next layer, another one of the same input; neither makes the model's output in the caller's memory unless it is the second.
    const auto pairs = [&](std::size_t i) {
        if (i + 1 >= layers.size()) return false;
        const LayerPlan &L = layers[i], &N = layers[i + 1];
        return L.conv && N.conv && !L.residual && !N.residual && L.in0 == N.in0 && L.out != N.out && L.out != L.in0 && N.out != L.in0 && !(out && i >= made);
    };
    for (; at < layers.size(); ++at) {
        const LayerPlan &L = layers[at];
        const float *bias = L.has_bias ? bias_pool.f32() + L.bias_offset : nullptr;
        switch (L.op) {
        case Op::MatMul:
            check(so_matmul(ctx, L.dE, src(L.in0), B, bias, dst(L.out), L.act), "so_matmul");
            break;
        case Op::Conv:
            if (pairs(at)) {
                const LayerPlan &N = layers[++at];
                const float *bias2 = N.has_bias ? bias_pool.f32() + N.bias_offset : nullptr;
                check(so_conv2d_pair(ctx, L.conv, N.conv, src(L.in0), B, bias, slot_ptr(L.out), L.act, bias2, dst(N.out), N.act), "so_conv2d_pair");
            } else if (L.residual)
                check(so_conv2d_add(ctx, L.conv, src(L.in0), B, bias, src(L.in1), dst(L.out), L.act), "so_conv2d_add");
            else
                check(so_conv2d(ctx, L.conv, src(L.in0), B, bias, dst(L.out), L.act), "so_conv2d");
            break;
        case Op::Act:
            check(so_act(ctx, L.act, src(L.in0), L.out_features * B, dst(L.out)), "so_act");
            break;
        case Op::Add:
            check(so_add(ctx, src(L.in0), src(L.in1), L.out_features * B, dst(L.out)), "so_add");
            break;
        case Op::MaxPool:
            check(so_maxpool(ctx, &L.pg, src(L.in0), B, dst(L.out)), "so_maxpool");
            break;
        case Op::GlobalAveragePool:
            check(so_gap(ctx, L.pg.C, L.pg.H, L.pg.W, src(L.in0), B, dst(L.out)), "so_gap");
            break;
        }
    }
}

// A launch graph spares the host about 4 us a launch, but the GPU waits 4 to 10 us before and behind one and works on the arena's
// slots only, so that device callers' input and output are copied: it pays where the chain is shorter than the host needs to launch it.
// The chain's time: 4 us a layer and the longer of a row's chain at 10 ns an entry and the layer's work at 25 TFLOP/s; the line lies at 6.5 us a
// layer.  ResNet-18-shaped stacks, 23 layers in 20 launches (three projections share one), us with a graph / without, run_device: 64 x 64 of width 16 at batch 1 110 / 122, 4 121 / 132,
// 16 125 / 125; 96 x 96 of 32 at 8 158 / 159; 160 x 160 of 48 at 2 189 / 177, which the line still records; 128 x 128 of 32 at 32 268 / 257; 224 x 224 of 64 at 1 222 / 209, at 32
// 924 / 907.  From host arrays: 64 x 64 at batch 4 127 / 124, 96 x 96 at 8 188 / 192, 128 x 128 of 48 at 2 176 / 176; 160 x 160 of 32 at 11 369 / 365, 224 x 224 of 48 at 4 361 / 356, of 64 at 1
// 237 / 236.
// A 4-layer MLP: 111 / 102; chains of fewer than eight layers have no graph.
bool SparseOnnxModel::Impl::record_pays() const
{
    if (use_graph >= 0) return use_graph == 1;
    if (layers.size() < 8) return false;
    double us = 0.0;
    for (const LayerPlan &L : layers) {
        us += 4.0;
        if (!L.E || L.E->m == 0) continue;
        double nnz = 0.0;
        for (uint32_t c : L.E->nnz) nnz += c;
        const double columns = (L.op == Op::Conv ? double(L.cg.H_out) * L.cg.W_out : 1.0) * pbatch;
        us += std::max(0.010 * nnz / L.E->m, 2.0 * nnz * columns / 25e6);
    }
    return us < 6.5 * double(layers.size());
}

void SparseOnnxModel::Impl::launch_chain() const
{
    if (graph) check(so_graph_launch(context(), graph), "so_graph_launch");
    else enqueue_layers();
}

void SparseOnnxModel::Impl::rows_in(const float *d_rows) const
{
    check(so_copy_rows(context(), d_rows, batch, uint32_t(in_features), batch, slot_ptr(input_slot), pbatch, 1), "so_copy_rows(input)");
}

void SparseOnnxModel::Impl::rows_out(float *d_rows) const
{
    check(so_copy_rows(context(), slot_ptr(output_slot), pbatch, uint32_t(out_features), batch, d_rows, batch, 0), "so_copy_rows(output)");
}

void SparseOnnxModel::run(const float *input, uint32_t B, float *output) const
{
    Impl &M = *impl_;
    if (B != M.batch) const_cast<SparseOnnxModel *>(this)->resize_buffers(B);
    so_ctx *ctx = context();
    std::lock_guard<std::mutex> lock(context_mutex());
    if (!M.padded()) {
        check(so_stage_in(ctx, M.slot_ptr(M.input_slot), input, M.in_features * B * sizeof(float), nullptr, nullptr, 0), "so_stage_in(input)");
        M.launch_chain();
        check(so_stage_out(ctx, output, M.slot_ptr(M.output_slot), M.out_features * B * sizeof(float)), "so_stage_out(output)");
        return;
    }
    check(so_stage_in(ctx, M.stage_in.get(), input, M.in_features * B * sizeof(float), nullptr, nullptr, 0), "so_stage_in(input)");
    M.rows_in(M.stage_in.f32());
    M.launch_chain();
    M.rows_out(M.stage_out.f32());
    check(so_stage_out(ctx, output, M.stage_out.get(), M.out_features * B * sizeof(float)), "so_stage_out(output)");
}

void SparseOnnxModel::run_batch_major(const float *input, uint32_t B, float *output) const
{
    Impl &M = *impl_;
    if (B != M.batch) const_cast<SparseOnnxModel *>(this)->resize_buffers(B);
    if (B == 1) { run(input, B, output); return; }      // one sample is the same in either order
    so_ctx *ctx = context();
    std::lock_guard<std::mutex> lock(context_mutex());
    // Both ways through the staging memory as one pass each where it holds the arrays: transposed, and padded to the arena's rows,
    // as they cross the link.
    int done = 0;
    check(so_stage_in_transposed(ctx, M.slot_ptr(M.input_slot), M.pbatch, input, B, uint32_t(M.in_features), &done), "so_stage_in_transposed(input)");
    if (!done) {
        check(so_stage_in(ctx, M.stage_in.get(), input, M.in_features * B * sizeof(float), nullptr, nullptr, 0), "so_stage_in(input)");
        check(so_transpose(ctx, M.stage_in.f32(), B, uint32_t(M.in_features), M.padded() ? M.stage_mid.f32() : M.slot_ptr(M.input_slot)), "so_transpose(input)");
        if (M.padded()) M.rows_in(M.stage_mid.f32());
    }
    M.launch_chain();
    check(so_stage_out_transposed(ctx, output, M.slot_ptr(M.output_slot), M.pbatch, uint32_t(M.out_features), B, &done), "so_stage_out_transposed(output)");
    if (done) return;
    if (M.padded()) M.rows_out(M.stage_mid.f32());
    check(so_transpose(ctx, M.padded() ? M.stage_mid.f32() : M.slot_ptr(M.output_slot), uint32_t(M.out_features), B, M.stage_out.f32()), "so_transpose(output)");
    check(so_stage_out(ctx, output, M.stage_out.get(), M.out_features * B * sizeof(float)), "so_stage_out(output)");
}

void SparseOnnxModel::run_device(const float *dInput, uint32_t B, float *dOutput) const
{
    Impl &M = *impl_;
    if (B != M.batch) const_cast<SparseOnnxModel *>(this)->resize_buffers(B);
    if (!dInput || !dOutput) throw std::runtime_error("run_device: null device pointer");
    std::lock_guard<std::mutex> lock(context_mutex());
    if (M.layers.empty()) {
        check(so_d2d(context(), dOutput, dInput, M.in_features * B * sizeof(float)), "so_d2d");
        return;
    }
    if (M.padded()) {
        M.rows_in(dInput);
        M.launch_chain();
        M.rows_out(dOutput);
        return;
    }
    so_ctx *ctx = context();
    // Without a launch graph, the layers on the caller's memory, without a copy of the input and of the output, where it is aligned as the slots are for any kernel's
    // choice: the same kernels and bits.  Memory that overlaps is copied.
    const std::uintptr_t x = reinterpret_cast<std::uintptr_t>(dInput), y = reinterpret_cast<std::uintptr_t>(dOutput);
    const bool apart = x + M.in_features * B * sizeof(float) <= y || y + M.out_features * B * sizeof(float) <= x;
    if (((x | y) & 15u) == 0 && apart && !M.graph && M.output_layer() < M.layers.size()) {
        M.enqueue_layers(dInput, dOutput);
        return;
    }
    check(so_d2d(ctx, M.slot_ptr(M.input_slot), dInput, M.in_features * B * sizeof(float)), "so_d2d(input)");
    M.launch_chain();
    check(so_d2d(ctx, dOutput, M.slot_ptr(M.output_slot), M.out_features * B * sizeof(float)), "so_d2d(output)");
}

double SparseOnnxModel::time_device(int steps, int warmup) const
{
    Impl &M = *impl_;
    if (steps <= 0) throw std::runtime_error("time_device: steps must be positive");
    so_ctx *ctx = context();
    std::lock_guard<std::mutex> lock(context_mutex());
    for (int i = 0; i < warmup; ++i) M.launch_chain();
    check(so_timer_begin(ctx), "so_timer_begin");
    for (int i = 0; i < steps; ++i) M.launch_chain();
    float ms = 0.0f;
    check(so_timer_end(ctx, &ms), "so_timer_end");
    return double(ms) / steps;
}
