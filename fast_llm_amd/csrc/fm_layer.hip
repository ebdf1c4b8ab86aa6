// The MoE layer's forward and backward as one or two host calls each: the launches of the router, the sparse map, the copies, the
// activation and the grouped products in the order of a layer step, on the caller's stream and buffers.
//
// What bounds a small layer is the host: a step of 512 tokens, 256 x 512, runs 20 kernels that the device finishes in 166 us,
// and launching them one Python call at a time took 567 us. Through these calls it takes 300.
#include "fm_gemm_common.h"
#include "fm_router_layout.h"

namespace fm {

namespace {

struct Plan {
    int64_t experts, slots, rows, used_index_size;
    int index_dtype;
    size_t top_experts, scores, lse, statistics, sparse_rows, expert_ends, expert_pad_begins, router, routing_bytes;
    size_t workspace_bytes, router_linear_bytes;  // of a backward
    size_t forward_workspace_bytes;
};

constexpr int64_t kPad = 128;

int make_plan(const fm_moe_layer &layer, Plan &plan) {
    const char *name = "fm_moe_layer";
    FM_REQUIRE(layer.tokens > 0 && layer.hidden > 0 && layer.ffn > 0 && layer.routed_experts > 0 && layer.shared_experts >= 0 &&
                   layer.experts_per_token > 0,
               "%s: bad shape", name);
    FM_REQUIRE(valid_dtype(static_cast<int>(layer.dtype)), "%s: bad dtype", name);
    plan.experts = layer.routed_experts + layer.shared_experts;
    plan.slots = layer.experts_per_token + layer.shared_experts;
    const int64_t entries = layer.tokens * plan.slots;
    const int64_t most_rows = (entries + plan.experts * kPad) / kPad * kPad;
    FM_REQUIRE(layer.dynamic_rows >= 0 && layer.dynamic_rows <= most_rows, "%s: %lld rows of at most %lld", name,
               static_cast<long long>(layer.dynamic_rows), static_cast<long long>(most_rows));
    plan.rows = layer.dynamic_rows > 0 ? layer.dynamic_rows : most_rows;
    plan.index_dtype = most_rows < 32768 ? FM_INDEX_I16 : FM_INDEX_I32;
    plan.used_index_size = plan.index_dtype == FM_INDEX_I16 ? 2 : 4;
    size_t at = 0;
    const auto take = [&](size_t bytes) {
        const size_t offset = at;
        at += (bytes + 63) / 64 * 64;
        return offset;
    };
    plan.top_experts = take(8 * entries);
    plan.scores = take(4 * entries);
    plan.lse = take(8 * layer.tokens);
    plan.statistics = take(4 * RouterStats::size(static_cast<int>(layer.routed_experts)));
    plan.sparse_rows = take(plan.used_index_size * entries);
    plan.expert_ends = take(plan.used_index_size * plan.experts);
    plan.expert_pad_begins = take(plan.used_index_size * plan.experts);
    plan.router = take(fm_router_workspace_size(layer.tokens, layer.routed_experts));
    plan.routing_bytes = at;
    plan.router_linear_bytes = fm_router_linear_backward_workspace_size(layer.tokens, layer.routed_experts, layer.hidden, static_cast<int>(layer.dtype));
    plan.workspace_bytes = plan.forward_workspace_bytes = 0;  // see plan_workspace
    return FM_OK;
}

// The calls of one layer step: the first failure ends it, a remark (the generic kernel ran) is kept.
struct Step {
    const fm_moe_layer &layer;
    const Plan &plan;
    void *stream;
    int note = FM_OK;

    char *routing(size_t offset) const { return static_cast<char *>(layer.routing) + offset; }
    int dtype() const { return static_cast<int>(layer.dtype); }
    int64_t ffn_1() const { return layer.ffn * (layer.gated ? 2 : 1); }
    int keep(int status) {
        if (status > 0) note = status;
        return status < 0 ? status : FM_OK;
    }

    int dispatch(void *out) {
        return fm_copy_dense_to_sparse(layer.input, nullptr, routing(plan.sparse_rows), out, layer.tokens, layer.hidden, plan.slots,
                                       plan.rows, dtype(), FM_DTYPE_F32, plan.index_dtype, stream);
    }
    int combine(const void *in, const void *scores, void *out) {
        return fm_copy_sparse_to_dense(in, scores, routing(plan.sparse_rows), out, layer.tokens, layer.hidden, plan.slots, plan.rows,
                                       dtype(), FM_DTYPE_F32, plan.index_dtype, stream);
    }
    // The products compute the rows that tokens own: what the padding rows of an intermediate hold is nobody's.
    // out [rows, columns] = lhs [rows, inner] x (weight_e [columns, inner])^T
    GemmArgs output_sparse(const void *lhs, const void *weight, void *out, int64_t columns, int64_t inner) const {
        return GemmArgs{lhs, weight, out, routing(plan.expert_ends), routing(plan.expert_pad_begins), inner, 1, 1, inner, columns, 1,
                        plan.rows, columns, inner, columns, static_cast<int>(plan.experts), kOutputSparse, 0, plan.index_dtype, dtype()};
    }
    // out [rows, hidden] = lhs [rows, inner] x weight_e [inner, hidden]
    GemmArgs inner_sparse(const void *lhs, const void *weight, void *out, int64_t inner) const {
        const int64_t hidden = layer.hidden;
        return GemmArgs{lhs, weight, out, routing(plan.expert_ends), routing(plan.expert_pad_begins), inner, 1, hidden, 1, hidden, 1,
                        plan.rows, hidden, inner, inner, static_cast<int>(plan.experts), kInputInnerSparse, 0, plan.index_dtype, dtype()};
    }
    // out [experts * size, hidden] (+)= lhs^T x rhs, lhs [rows, size], rhs [rows, hidden]
    GemmArgs row_sparse(const void *lhs, const void *rhs, void *out, int64_t size, bool accumulate) const {
        const int64_t hidden = layer.hidden;
        return GemmArgs{lhs, rhs, out, routing(plan.expert_ends), routing(plan.expert_pad_begins), 1, size, hidden, 1, hidden, 1,
                        size * plan.experts, hidden, plan.rows, size, static_cast<int>(plan.experts), kInputRowSparse, accumulate,
                        plan.index_dtype, static_cast<int>(layer.grad_dtype)};
    }
    GemmArgs layer_1() const {
        GemmArgs args = output_sparse(layer.sparse_input, layer.weight_1, layer.layer_1_output, ffn_1(), layer.hidden);
        if (layer.gated && layer.layer_1_output == nullptr) {  // the activation in the product's epilogue
            args.fusion = kFusionGatedForward;
            args.activation = static_cast<int>(layer.activation);
            args.fused_out = layer.activation_output;
            args.fused_stride = args.half = layer.ffn;
            args.any_half = 1;
        }
        return args;
    }
    enum { kLayer1 = 0, kLayer2 = 1, kGradActivation = 1, kGradWeight2 = 2, kGradInput = 3, kGradWeight1 = 4 };
    // The products of a forward, and of a backward.
    void forward_products(GemmArgs *products) const {
        products[kLayer1] = layer_1();
        products[kLayer2] = inner_sparse(layer.activation_output, layer.weight_2, layer.layer_2_output, layer.ffn);
    }
    void backward_products(GemmArgs *products) const {
        products[kLayer1] = layer_1();
        products[kGradActivation] = output_sparse(layer.grad_layer_2_output, layer.weight_2, layer.grad_activation_output, layer.ffn, layer.hidden);
        products[kGradWeight2] = row_sparse(layer.activation_output, layer.grad_layer_2_output, layer.grad_weight_2, layer.ffn, layer.accumulate_2 != 0);
        products[kGradInput] = inner_sparse(layer.grad_layer_1_output, layer.weight_1, layer.grad_layer_2_output, ffn_1());
        products[kGradWeight1] = row_sparse(layer.grad_layer_1_output, layer.sparse_input, layer.grad_weight_1, ffn_1(), layer.accumulate_1 != 0);
    }
    // One launch for the tile tables of all products that are wanted: each launch of its own took 7 us.
    int plan_tables(GemmArgs *products, const bool *wanted, int count, size_t workspace_bytes) const {
        GemmArgs chosen[kMaxPlanned];
        int which[kMaxPlanned], num = 0;
        for (int i = 0; i < count; ++i)
            if (wanted[i]) chosen[num] = products[i], which[num++] = i;
        if (dtype() == FM_DTYPE_F32) return FM_OK;
        const int status = mfma_gemm_plan(chosen, num, dtype(), layer.workspace, workspace_bytes, static_cast<hipStream_t>(stream));
        for (int i = 0; i < num; ++i) products[which[i]] = chosen[i];
        return status;
    }
    int product(const GemmArgs &args) { return keep(run_gemm("fm_moe_layer", args, dtype(), nullptr, 0, stream)); }
    const void *rows_in_use() const { return routing(plan.expert_ends + (plan.experts - 1) * plan.used_index_size); }
};

// From the shape alone, whatever buffers the caller has filled in: it asks for the size before it has them. A forward runs layer
// 1 with or without its output, whose tables differ; a backward always has the output.
void plan_workspace(const fm_moe_layer &layer, Plan &plan) {
    fm_moe_layer kept = layer, fused = layer;
    kept.layer_1_output = kept.routing = &kept;  // any address: nothing is launched
    fused.layer_1_output = nullptr, fused.routing = &fused;
    const Step with_output{kept, plan, nullptr}, without{fused, plan, nullptr};
    const int dtype = with_output.dtype();
    GemmArgs products[kMaxPlanned];
    with_output.forward_products(products);
    plan.forward_workspace_bytes = max(fm_sparse_map_from_router_workspace_size(layer.tokens, plan.experts), mfma_gemm_plan_size(products, 2, dtype));
    without.forward_products(products);
    plan.forward_workspace_bytes = max(plan.forward_workspace_bytes, mfma_gemm_plan_size(products, 2, dtype));
    with_output.backward_products(products);
    plan.workspace_bytes = max(max(plan.router_linear_bytes, mfma_gemm_plan_size(products, kMaxPlanned, dtype)), size_t(256));
}

#define FM_STEP(call) \
    if (int status = (call)) return status

int route(const fm_moe_layer &layer, const Plan &plan, void *stream) {
    Step step{layer, plan, stream};
    const bool losses = layer.with_losses != 0;
    FM_REQUIRE(layer.logits && layer.routing && layer.workspace && (layer.losses || !losses), "fm_moe_layer_route: null tensor");
    FM_STEP(router_forward(layer.logits, layer.noise, step.routing(plan.top_experts), step.routing(plan.scores),
                           losses ? step.routing(plan.lse) : nullptr, losses ? step.routing(plan.statistics) : nullptr,
                           losses ? layer.losses : nullptr, step.routing(plan.router), plan.routing_bytes - plan.router, layer.tokens,
                           layer.routed_experts, layer.experts_per_token, layer.shared_experts, step.dtype(), false, stream));
    RouterFinish finish;
    if (losses)
        finish = router_finish_of(step.routing(plan.router), step.routing(plan.statistics), layer.losses, layer.tokens,
                                  layer.routed_experts, layer.shared_experts);
    FM_STEP(sparse_map_from_router(reinterpret_cast<const int64_t *>(step.routing(plan.top_experts)), step.routing(plan.router),
                                   plan.routing_bytes - plan.router, layer.tokens, plan.experts, layer.experts_per_token,
                                   layer.shared_experts, kPad, plan.index_dtype, step.routing(plan.sparse_rows),
                                   step.routing(plan.expert_ends), step.routing(plan.expert_pad_begins), layer.workspace,
                                   plan.forward_workspace_bytes, losses ? &finish : nullptr, stream));
    return FM_OK;
}

int forward(const fm_moe_layer &layer, const Plan &plan, void *stream) {
    Step step{layer, plan, stream};
    FM_REQUIRE(layer.input && layer.weight_1 && layer.weight_2 && layer.routing && layer.sparse_input && layer.activation_output &&
                   layer.layer_2_output && layer.output && layer.workspace,
               "fm_moe_layer_forward: null tensor");
    FM_REQUIRE(layer.gated || layer.layer_1_output, "fm_moe_layer_forward: layer 1 without a gate needs its output");
    GemmArgs products[2];
    step.forward_products(products);
    const bool wanted[2] = {true, true};
    FM_STEP(step.plan_tables(products, wanted, 2, plan.forward_workspace_bytes));
    FM_STEP(step.dispatch(layer.sparse_input));
    if (products[Step::kLayer1].fusion != kFusionNone) {
        // FM_ERR_UNSUPPORTED tells the caller to bring a layer-1 buffer.
        FM_STEP(run_fused_gemm("fm_moe_layer_forward", products[Step::kLayer1], step.dtype(), stream));
    } else {
        FM_STEP(step.product(products[Step::kLayer1]));
        FM_STEP(fm_mlp_activation_forward(layer.layer_1_output, layer.activation_output, plan.rows, layer.ffn,
                                          static_cast<int>(layer.gated), static_cast<int>(layer.activation), step.dtype(),
                                          step.rows_in_use(), plan.index_dtype, stream));
    }
    FM_STEP(step.product(products[Step::kLayer2]));
    FM_STEP(step.combine(layer.layer_2_output, step.routing(plan.scores), layer.output));
    return step.note;
}

// The gradients of layer 2's output and of the scores: the only step of a backward that reads layer 2's output.
int combine_backward(const fm_moe_layer &layer, const Plan &plan, void *stream) {
    const Step step{layer, plan, stream};
    FM_REQUIRE(layer.routing && layer.layer_2_output && layer.grad_output && layer.grad_layer_2_output && layer.grad_scores,
               "fm_moe_layer_backward: null tensor");
    return fm_copy_sparse_to_dense_backward(layer.layer_2_output, layer.grad_output, step.routing(plan.scores),
                                            step.routing(plan.sparse_rows), layer.grad_layer_2_output, layer.grad_scores,
                                            layer.tokens, layer.hidden, plan.slots, plan.rows, step.dtype(), FM_DTYPE_F32,
                                            FM_DTYPE_F32, plan.index_dtype, stream);
}

int rest_of_backward(const fm_moe_layer &layer, const Plan &plan, void *stream) {
    Step step{layer, plan, stream};
    FM_REQUIRE(layer.logits && layer.weight_1 && layer.weight_2 && layer.routing && layer.sparse_input && layer.layer_1_output &&
                   layer.activation_output && layer.grad_layer_2_output && layer.grad_activation_output &&
                   layer.grad_layer_1_output && layer.grad_scores && layer.grad_logits && layer.workspace &&
                   (layer.input || !(layer.recompute_input || layer.router)),
               "fm_moe_layer_backward: null tensor");
    GemmArgs products[kMaxPlanned];
    step.backward_products(products);
    const bool wanted[kMaxPlanned] = {layer.recompute_layer_1 != 0, true, layer.grad_weight_2 != nullptr, layer.grad_input != nullptr,
                                      layer.grad_weight_1 != nullptr};
    FM_STEP(step.plan_tables(products, wanted, kMaxPlanned, plan.workspace_bytes));
    // What the forward did not keep.
    if (layer.recompute_input) FM_STEP(step.dispatch(layer.sparse_input));
    if (layer.recompute_layer_1) FM_STEP(step.product(products[Step::kLayer1]));
    // Through layer 2 and the activation.
    FM_STEP(step.product(products[Step::kGradActivation]));
    FM_STEP(fm_mlp_activation_backward(layer.grad_activation_output, layer.grad_layer_1_output, layer.layer_1_output,
                                       layer.recompute_activation ? layer.activation_output : nullptr, plan.rows, layer.ffn,
                                       static_cast<int>(layer.gated), static_cast<int>(layer.activation), step.dtype(),
                                       step.rows_in_use(), plan.index_dtype, stream));
    if (layer.grad_weight_2) FM_STEP(step.product(products[Step::kGradWeight2]));
    // Through layer 1. The gradient of layer 2's output has been read for the last time: that of the sparse input takes
    // its place.
    if (layer.grad_input) FM_STEP(step.product(products[Step::kGradInput]));
    if (layer.grad_weight_1) FM_STEP(step.product(products[Step::kGradWeight1]));
    if (layer.grad_input) FM_STEP(step.combine(layer.grad_layer_2_output, nullptr, layer.grad_input));
    const bool losses = layer.with_losses != 0;
    FM_STEP(router_backward(layer.grad_scores, step.routing(plan.scores), step.routing(plan.top_experts), layer.logits, layer.noise,
                            losses ? step.routing(plan.lse) : nullptr, losses ? step.routing(plan.statistics) : nullptr,
                            layer.grad_logits, layer.auxiliary_loss_grad, layer.z_loss_grad, layer.tokens,
                            layer.routed_experts, layer.experts_per_token, layer.shared_experts, step.dtype(), true, stream));
    if (layer.router != nullptr)
        FM_STEP(step.keep(router_linear_backward(layer.grad_logits, layer.input, layer.router, layer.router_input_grad ? layer.grad_input : nullptr,
                                                 layer.grad_router, layer.router_input_grad == 2, layer.tokens, layer.routed_experts,
                                                 layer.hidden, step.dtype(), layer.workspace, plan.workspace_bytes, stream)));
    return step.note;
}

}  // namespace

}  // namespace fm

using namespace fm;

extern "C" int fm_moe_layer_sizes(fm_moe_layer *layer) {
    Plan plan;
    FM_REQUIRE(layer, "fm_moe_layer_sizes: null");
    if (int status = make_plan(*layer, plan)) return status;
    plan_workspace(*layer, plan);
    layer->rows = plan.rows;
    layer->routing_bytes = static_cast<int64_t>(plan.routing_bytes);
    layer->workspace_bytes = static_cast<int64_t>(plan.workspace_bytes);
    layer->forward_workspace_bytes = static_cast<int64_t>(plan.forward_workspace_bytes);
    layer->index_dtype = plan.index_dtype;
    layer->router_linear = plan.router_linear_bytes > 0;
    layer->used_rows_offset = static_cast<int64_t>(plan.expert_ends) + (plan.experts - 1) * plan.used_index_size;
    return FM_OK;
}

// The plan of a call, and that the caller's buffers are of the sizes which fm_moe_layer_sizes gave it for this very shape: the
// parts are told how large they are, so none of them would notice.
static int plan_call(const char *name, const fm_moe_layer *layer, Plan &plan) {
    FM_REQUIRE(layer, "%s: null", name);
    if (int status = make_plan(*layer, plan)) return status;
    plan_workspace(*layer, plan);
    FM_REQUIRE(layer->rows == plan.rows && layer->routing_bytes >= static_cast<int64_t>(plan.routing_bytes) &&
                   layer->workspace_bytes >= static_cast<int64_t>(plan.workspace_bytes) &&
                   layer->forward_workspace_bytes >= static_cast<int64_t>(plan.forward_workspace_bytes),
               "%s: %lld rows, %lld bytes of routing, %lld and %lld of workspace, needs %lld, %zu, %zu and %zu (fm_moe_layer_sizes, after "
               "the last change of the shape)", name, static_cast<long long>(layer->rows), static_cast<long long>(layer->routing_bytes),
               static_cast<long long>(layer->forward_workspace_bytes), static_cast<long long>(layer->workspace_bytes),
               static_cast<long long>(plan.rows), plan.routing_bytes, plan.forward_workspace_bytes, plan.workspace_bytes);
    FM_REQUIRE(reinterpret_cast<uintptr_t>(layer->routing) % 64 == 0 && reinterpret_cast<uintptr_t>(layer->workspace) % 64 == 0,
               "%s: routing and workspace must be 64-byte aligned", name);
    return FM_OK;
}

extern "C" int fm_moe_layer_route(const fm_moe_layer *layer, void *stream) {
    Plan plan;
    if (int status = plan_call("fm_moe_layer_route", layer, plan)) return status;
    return route(*layer, plan, stream);
}

extern "C" int fm_moe_layer_forward(const fm_moe_layer *layer, void *stream) {
    Plan plan;
    if (int status = plan_call("fm_moe_layer_forward", layer, plan)) return status;
    return forward(*layer, plan, stream);
}

extern "C" int fm_moe_layer_backward(const fm_moe_layer *layer, void *stream) {
    Plan plan;
    const char *name = "fm_moe_layer_backward";
    if (int status = plan_call(name, layer, plan)) return status;
    FM_REQUIRE(layer->backward_part >= 0 && layer->backward_part <= 2, "%s: part %lld", name, static_cast<long long>(layer->backward_part));
    if (layer->backward_part != 2) FM_STEP(combine_backward(*layer, plan, stream));
    return layer->backward_part != 1 ? rest_of_backward(*layer, plan, stream) : FM_OK;
}
