// The layer's host path: LookupFFN.forward and its backward from Python's call to the kernels' launches.
//
// A layer call at a few hundred tokens is one launch of a few microseconds, a training step of that size about twenty;
// through the interpreter (argument checks, the operator dispatcher, foreign-function calls, two autograd functions) a call
// took 15 us and a step 400 us whatever the kernels took (17 tokens, and 385 tokens at hidden 512).  Here a call
// looks up what the layer holds, allocates its result and launches; a
// training forward records one autograd node whose backward launches the whole chain.
//
// forward(layer, x, residual, ...) looks its modules and parameters up on every call and keeps nothing of them.  The answer is
// None whenever anything is not of a kind the kernels are built for: another module, sizes that do not fit together, a dtype,
// device or layout, a gradient wanted that this path does not compute.  Then the Python path runs, with its own checks and errors.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>

#include <dlfcn.h>

#include <array>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/lookupffn_hip.h"

namespace {

using at::Tensor;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// The kernel library is the one Python has loaded (bind gets its path): its entry points by name.
#define LFFN_ENTRIES(X)                     \
    X(lffn_error_string)                    \
    X(lffn_lookup_ffn_fused_layer_rows)     \
    X(lffn_lookup_gather_records_plan_rows) \
    X(lffn_ln_project_hash_records_f32)     \
    X(lffn_lookup_gather_records_rows)      \
    X(lffn_lookup_gather_parts_plan)        \
    X(lffn_lookup_gather_parts_rows)        \
    X(lffn_ln_project_hash_f32)             \
    X(lffn_lookup_gather_workspace_bytes)   \
    X(lffn_lookup_gather_ws_f32)            \
    X(lffn_lookup_gather_ws_bf16)           \
    X(lffn_lookup_gather_ws_f16)            \
    X(lffn_bh4_block_front_split_f32)       \
    X(lffn_bh4_block_front_train_split_f32) \
    X(lffn_bh4_fold_split_both_f32)         \
    X(lffn_bh4_fold_mode_f32)               \
    X(lffn_lookup_scatter_workspace_bytes)  \
    X(lffn_lookup_scatter_plan)             \
    X(lffn_lookup_backward_sums_f32)        \
    X(lffn_lookup_backward_sums_rows)       \
    X(lffn_lookup_inner_f32)                \
    X(lffn_lookup_scatter_f32)              \
    X(lffn_lookup_scatter_sorted_f32)       \
    X(lffn_ln_project_hash_bwd_f32)         \
    X(lffn_bh4_block_score_bwd_split_f32)   \
    X(lffn_ln_bh4_block_wgrad_f32)          \
    X(lffn_layer_norm_bwd_f32)              \
    X(lffn_sum_partials_f32)                \
    X(lffn_sum_many_f32)

struct Library {
#define X(name) decltype(&::name) name = nullptr;
    LFFN_ENTRIES(X)
#undef X
} lib;

void check(int rc, const char *what) { TORCH_CHECK(rc == LFFN_OK, what, ": ", lib.lffn_error_string(rc), " (code ", rc, ")"); }
#define CALL(name, ...) check(lib.name(__VA_ARGS__), #name)

enum Form { DIAG = 0, BLOCK = 1 };

// Sizes and constants of a layer.
struct Config {
    int64_t form, H, D, R, J, T, S, Do, fmt;
    bool one_launch, trainable;
    double eps, decay, residual;
};

// The Python operators' own (bind).
struct Thresholds {
    int64_t ln_partials, project_partials, sum_chunk_rows;
} limits;
PyTypeObject *layer_norm_type, *bh4_type;

// Which form the gather takes for a batch, a function of the sizes alone.
struct RecordPlan {
    std::array<int64_t, 6> sizes{-1};    // B, T, S, Do, row format, records possible
    int64_t stride = 0, bytes = 0, ws_bytes = 0;
    int32_t tokens = 0;
    lffn_gather_parts parts{};           // parts > 0: the tables shared out over several workgroups
};

// What the layer holds at this moment: its hash, the hash's projection and its LayerNorm as Python finds them on every access, the
// parameters in them (in the order of Input below) and their constants.  Borrowed references.
struct Parts {
    PyObject *norm, *hash, *projection;
    std::array<PyObject *, 6> params;
    double eps, decay;
    int64_t num_table, output_size;
};

PyObject *KEY_MODULES, *KEY_PARAMETERS, *KEY_LAYER_NORM, *KEY_HASH, *KEY_PROJECTION, *KEY_WEIGHT, *KEY_BIAS, *KEY_TABLES, *KEY_EPS,
    *KEY_DECAY, *KEY_NUM_TABLE, *KEY_OUTPUT_SIZE, *KEY_FOLDED;      // interned

PyObject *dict_of(PyObject *o) {
    PyObject **d = o ? _PyObject_GetDictPtr(o) : nullptr;
    return d ? *d : nullptr;
}

// (keys are strings: looking one up raises nothing)
PyObject *item(PyObject *dict, PyObject *key) { return dict && PyDict_Check(dict) ? PyDict_GetItemWithError(dict, key) : nullptr; }

bool number(PyObject *o, double &value) {
    if (!o || !(PyFloat_Check(o) || PyLong_Check(o))) return false;
    value = PyFloat_AsDouble(o);
    if (value == -1.0 && PyErr_Occurred()) {             // an integer beyond double
        PyErr_Clear();
        return false;
    }
    return true;
}

bool whole(PyObject *o, int64_t &value) {
    if (!o || !PyLong_Check(o)) return false;
    int overflow = 0;
    value = PyLong_AsLongLongAndOverflow(o, &overflow);
    return !overflow;
}

// False when something is not where a LookupFFN has it (a reparametrised weight is no parameter but computed on every access).
bool find_parts(PyObject *layer, Parts &found) {
    PyObject *own = dict_of(layer), *modules = item(own, KEY_MODULES);
    found.norm = item(modules, KEY_LAYER_NORM);
    found.hash = item(modules, KEY_HASH);
    PyObject *norm = dict_of(found.norm), *hash = dict_of(found.hash);
    found.projection = item(item(hash, KEY_MODULES), KEY_PROJECTION);
    if (!found.norm || !found.projection || !PyObject_TypeCheck(found.norm, layer_norm_type) || !PyObject_TypeCheck(found.projection, bh4_type))
        return false;
    PyObject *projection = dict_of(found.projection), *of_layer = item(own, KEY_PARAMETERS), *of_norm = item(norm, KEY_PARAMETERS),
             *of_projection = item(projection, KEY_PARAMETERS);
    found.params = {item(of_norm, KEY_WEIGHT),       item(of_norm, KEY_BIAS),    item(of_projection, KEY_WEIGHT),
                    item(of_projection, KEY_BIAS), item(of_layer, KEY_TABLES), item(of_layer, KEY_BIAS)};
    for (PyObject *o : found.params)
        if (!o || !THPVariable_Check(o)) return false;
    return number(item(norm, KEY_EPS), found.eps) && number(item(projection, KEY_DECAY), found.decay) &&
           whole(item(own, KEY_NUM_TABLE), found.num_table) && whole(item(own, KEY_OUTPUT_SIZE), found.output_size);
}

float *f32(const Tensor &t) { return t.defined() ? static_cast<float *>(t.data_ptr()) : nullptr; }

hipStream_t stream_on(const at::Device &d) { return c10::hip::getCurrentHIPStream(d.index()).stream(); }

Tensor empty_f32(at::IntArrayRef sizes, const at::Device &d) { return at::empty(sizes, at::TensorOptions().dtype(at::kFloat).device(d)); }
Tensor empty_bytes(int64_t n, const at::Device &d) { return at::empty({n}, at::TensorOptions().dtype(at::kByte).device(d)); }

RecordPlan plan_for(const Config &c, int64_t B, bool records) {
    // the last plans by their sizes
    static std::array<RecordPlan, 64> known;
    static std::mutex lock;
    const std::lock_guard<std::mutex> guard(lock);
    const std::array<int64_t, 6> sizes{B, c.T, c.S, c.Do, c.fmt, records && c.T % 2 == 0 && (c.form == BLOCK || c.D >= 16)};
    size_t slot = 0;
    for (int64_t n : sizes) slot = slot * 31 + (size_t)n;
    RecordPlan &p = known[(slot ^ slot >> 12) % known.size()];
    if (p.sizes != sizes) {
        RecordPlan made;
        CALL(lffn_lookup_gather_parts_plan, B, c.T, c.S, c.Do, (int32_t)c.fmt, (int32_t)sizes[5], &made.parts);
        if (made.parts.parts) {
            made.tokens = made.parts.tokens_per_workgroup;
            made.stride = made.parts.record_stride;
            made.ws_bytes = made.parts.bytes;
            if (sizes[5]) made.bytes = made.parts.bytes;
        } else if (sizes[5])
            CALL(lffn_lookup_gather_records_plan_rows, B, c.T, c.S, c.Do, (int32_t)c.fmt, &made.tokens, &made.stride, &made.bytes);
        if (made.bytes == 0 && made.ws_bytes == 0) CALL(lffn_lookup_gather_workspace_bytes, B, c.T, c.S, c.Do, (int32_t)c.fmt, &made.ws_bytes);
        made.sizes = sizes;
        p = made;
    }
    return p;
}

// Codes and scores [B, T] -> the gather, by whichever form the shape gets.
void gather(const Config &c, const Tensor &codes, const Tensor &scores, const Tensor &tables, const Tensor &obias, const float *residual,
            Tensor &out, int64_t B, const RecordPlan &plan, void *st) {
    const int64_t ws_bytes = plan.ws_bytes;
    Tensor ws;
    if (ws_bytes > 0) ws = empty_bytes(ws_bytes, out.device());
    void *wp = ws_bytes > 0 ? ws.data_ptr() : nullptr;
    const int32_t *cp = static_cast<const int32_t *>(codes.data_ptr());
    if (plan.parts.parts) {
        CALL(lffn_lookup_gather_parts_rows, &plan.parts, cp, f32(scores), tables.data_ptr(), f32(obias), residual, f32(out), wp, ws_bytes,
             B, c.T, c.S, c.Do, (int32_t)c.fmt, st);
        return;
    }
    if (c.fmt == 0)
        CALL(lffn_lookup_gather_ws_f32, cp, f32(scores), f32(tables), f32(obias), residual, f32(out), wp, ws_bytes, B, c.T, c.S, c.Do, st);
    else if (c.fmt == 1)
        CALL(lffn_lookup_gather_ws_bf16, cp, f32(scores), static_cast<const uint16_t *>(tables.data_ptr()), f32(obias), residual, f32(out),
             wp, ws_bytes, B, c.T, c.S, c.Do, st);
    else
        CALL(lffn_lookup_gather_ws_f16, cp, f32(scores), static_cast<const uint16_t *>(tables.data_ptr()), f32(obias), residual, f32(out),
             wp, ws_bytes, B, c.T, c.S, c.Do, st);
}

// The layer's parameters: LayerNorm's, the projection's, tables and output bias.
using Params = std::array<Tensor, 6>;

// Floats of the split weights (lffn_bh4_fold_split_f32).
int64_t split_words(const Config &c) { return c.R * c.J * (c.D * 65 + 1); }

// The front end of 64 x 64 blocks; split: their weights (lffn_bh4_fold_split_f32).  The kernel is the training forward's, so that a layer
// computes the same codes with gradients recorded and without (a checkpointed pass runs both).
lffn_block_front block_front(const Config &c, const Params &p, const Tensor &split) {
    lffn_block_front f{};
    f.ln_weight = f32(p[0]); f.ln_bias = f32(p[1]); f.w_split = f32(split); f.proj_bias = f32(p[3]);
    f.H = c.H; f.D = c.D; f.R = c.R; f.J = c.J; f.T = c.T;
    f.ln_eps = (float)c.eps; f.decay = (float)c.decay; f.residual = (float)c.residual;
    return f;
}

void infer(const Config &c, const Params &p, const Tensor &split, const Tensor &x, const float *residual, Tensor &out, int64_t B,
           int64_t fused_max) {
    const at::Device dev = x.device();
    void *st = stream_on(dev);
    // Rows of 16 bits are half the traffic of a form that reads every token's rows from memory, and so good for half as many tokens
    // more, and so are tables of which a token's rows are few.  One launch, two, us, tables not in the caches: fp32 768 tokens, 128
    // tables of 768 columns 45.5, 48.8, of 832 48.7, 51.5, of 896 52.4, 53.3, but of 960 55.3, 53.7, of 1024 59.0, 57.0 and 512 of 1024
    // 218, 187 (256 tables of 448 53.7, 63.7); bfloat16 1152 tokens, 128 of 768 37.8, 70, of 896 43.5, 45.2.
    if (c.fmt != 0) fused_max += fused_max / 2;
    if (c.T * c.Do <= 128 * 896) fused_max += fused_max / 2;
    if (c.one_launch && B <= fused_max) {
        const lffn_fused_layer layer{f32(p[0]), f32(p[1]), f32(p[2]), f32(p[3]), f32(p[4]), f32(p[5]), c.H, c.D, c.R, c.J, c.T,
                                     c.S, c.Do, (float)c.eps, (float)c.decay, (float)c.residual};
        CALL(lffn_lookup_ffn_fused_layer_rows, &layer, (int32_t)c.fmt, f32(x), residual, f32(out), B, st);
        return;
    }
    const float eps = (float)c.eps, decay = (float)c.decay, res = (float)c.residual;
    const RecordPlan plan = plan_for(c, B, true);
    if (plan.bytes > 0) {
        // some thousand tokens and more: the projection kernel writes the gather kernel's record stream directly
        Tensor records = empty_bytes(plan.bytes, dev);
        uint32_t *rp = static_cast<uint32_t *>(records.data_ptr());
        if (c.form == DIAG)
            CALL(lffn_ln_project_hash_records_f32, f32(x), f32(p[0]), f32(p[1]), eps, f32(p[2]), f32(p[3]), rp, plan.stride,
                 plan.tokens, B, c.H, c.D, c.R, c.J, c.T, decay, res, st);
        else {
            lffn_block_front front = block_front(c, p, split);
            front.records = rp;
            front.record_stride = plan.stride;
            front.tokens_per_workgroup = plan.tokens;
            CALL(lffn_bh4_block_front_split_f32, &front, f32(x), B, st);
        }
        if (plan.parts.parts)
            CALL(lffn_lookup_gather_parts_rows, &plan.parts, nullptr, nullptr, p[4].data_ptr(), f32(p[5]), residual, f32(out), rp, plan.bytes,
                 B, c.T, c.S, c.Do, (int32_t)c.fmt, st);
        else
            CALL(lffn_lookup_gather_records_rows, rp, plan.stride, p[4].data_ptr(), f32(p[5]), residual, f32(out), B, c.T, c.S, c.Do,
             (int32_t)c.fmt, plan.tokens, st);
        return;
    }
    Tensor codes = at::empty({B, c.T}, at::TensorOptions().dtype(at::kInt).device(dev)), scores = empty_f32({B, c.T}, dev);
    int32_t *cp = static_cast<int32_t *>(codes.data_ptr());
    if (c.form == DIAG)
        CALL(lffn_ln_project_hash_f32, f32(x), f32(p[0]), f32(p[1]), eps, f32(p[2]), f32(p[3]), nullptr, cp, f32(scores), B, c.H,
             c.D, c.R, c.J, c.T, decay, res, st);
    else {
        lffn_block_front front = block_front(c, p, split);
        front.codes = cp;
        front.scores = f32(scores);
        CALL(lffn_bh4_block_front_split_f32, &front, f32(x), B, st);
    }
    gather(c, codes, scores, p[4], p[5], residual, out, B, plan, st);
}

// Column sums of [P, n] arrays of partial sums, all in one launch at the end, fixed order of additions.  Very many rows go through a
// first pass over chunks of rows on many workgroups.
struct ColumnSums {
    std::array<lffn_sum, 8> sums{};
    int32_t count = 0;
    std::vector<Tensor> held;               // until finish(): what they are formed from, and results that nobody else may hold

    void add(const Tensor &parts, const float *a, const Tensor &out, int64_t n, int64_t P, const at::Device &dev, void *st) {
        held.push_back(parts);
        held.push_back(out);
        if (P > MANY_ROWS) {
            int64_t chunks = (P + limits.sum_chunk_rows - 1) / limits.sum_chunk_rows;
            const int64_t each = (P + chunks - 1) / chunks;
            chunks = (P + each - 1) / each;                    // no empty chunk
            held.push_back(empty_f32({chunks * n}, dev));
            float *mid = f32(held.back());
            CALL(lffn_sum_partials_f32, a, mid, n, nullptr, nullptr, 0, P, chunks, st);
            a = mid; P = chunks;
        }
        sums.at(count++) = {a, f32(out), n, P};
    }
    void finish(void *st) {
        if (count) CALL(lffn_sum_many_f32, sums.data(), count, st);
    }
    static constexpr int64_t MANY_ROWS = 4096;
};

// Inputs of the node, in the order of its gradients.
enum Input { X, LN_W, LN_B, WEIGHT, PBIAS, TABLES, OBIAS, RESIDUAL, INPUTS };

// What a graph through the layer's gradients (create_graph) ends in: the kernels compute them without one.
struct NoSecondDerivative : public torch::autograd::Node {
    std::string name() const override { return "LookupFFNNoSecondDerivative"; }
    variable_list apply(variable_list &&) override {
        TORCH_CHECK(false, "LookupFFN: the gradients of the layer cannot be differentiated (a graph through them was asked for with "
                           "create_graph)");
    }
};

struct LookupFFNBackward : public torch::autograd::Node {
    Config c{};
    int64_t B = 0;
    SavedVariable x, ln_w, ln_b, weight, tables, codes, scores, z, stage_in, stats, split_t;

    std::string name() const override { return "LookupFFNBackward"; }

    void release_variables() override {
        for (SavedVariable *v : {&x, &ln_w, &ln_b, &weight, &tables, &codes, &scores, &z, &stage_in, &stats, &split_t}) v->reset_data();
    }

    variable_list apply(variable_list &&grads) override {
        const bool graph = at::GradMode::is_enabled();
        variable_list out = gradients(grads);
        if (!graph) return out;
        auto end = std::shared_ptr<NoSecondDerivative>(new NoSecondDerivative(), torch::autograd::deleteNode);
        torch::autograd::edge_list edges = next_edges();                     // they depend on the inputs and on the gradient
        for (auto &e : torch::autograd::collect_next_edges(grads[0])) edges.push_back(std::move(e));
        end->set_next_edges(std::move(edges));
        for (int i = 0; i < INPUTS; ++i)
            if (i != RESIDUAL && out[i].defined()) torch::autograd::set_history(out[i], end);
        return out;
    }

    variable_list gradients(const variable_list &grads) {
        variable_list out(INPUTS);
        if (!grads[0].defined()) return out;
        at::AutoGradMode no_grad(false);
        const Tensor g = grads[0].contiguous();
        TORCH_CHECK(g.scalar_type() == at::kFloat, "LookupFFN: the gradient of the output is fp32");
        const auto self = shared_from_this();
        const Tensor x_ = x.unpack(self), lw = ln_w.unpack(self), lb = ln_b.unpack(self), w = weight.unpack(self),
                     tab = tables.unpack(self), code = codes.unpack(self), score = scores.unpack(self), z_ = z.unpack(self);
        const at::Device dev = x_.device();
        const c10::DeviceGuard guard(dev);
        void *st = stream_on(dev);
        const int64_t T = c.T, S = c.S, Do = c.Do, H = c.H, D = c.D, R = c.R, J = c.J;
        const int32_t *cp = static_cast<const int32_t *>(code.data_ptr());
        bool need[INPUTS];
        for (int i = 0; i < INPUTS; ++i) need[i] = task_should_compute_output(i);
        if (need[RESIDUAL]) out[RESIDUAL] = grads[0];
        ColumnSums column_sums;
        if (need[OBIAS]) out[OBIAS] = empty_f32({Do}, dev);
        bool bias_summed = !need[OBIAS];                        // in the scatter's copy of g
        const bool need_ln = need[X] || need[LN_W] || need[LN_B];
        const bool need_score = need_ln || need[WEIGHT] || need[PBIAS];
        // both gradients of the gather: one call with one workspace where the sorted scatter is the one to use
        Tensor g_score;
        if (need_score) g_score = empty_f32({B, T}, dev);
        if (need[TABLES]) out[TABLES] = at::empty_like(tab);
        if (need_score || need[TABLES]) {
            int64_t ws_bytes = 0;
            int32_t sorted = 0;
            CALL(lffn_lookup_scatter_plan, B, T, S, Do, &sorted);
            if (sorted) CALL(lffn_lookup_scatter_workspace_bytes, B, T, S, Do, &ws_bytes);
            if (need[TABLES] && ws_bytes > 0) {
                Tensor ws = empty_bytes(ws_bytes, dev);
                if (need_score) {
                    int64_t rows = 0;
                    CALL(lffn_lookup_backward_sums_rows, B, &rows);
                    Tensor parts = bias_summed ? Tensor() : empty_f32({rows * Do}, dev);
                    CALL(lffn_lookup_backward_sums_f32, cp, f32(score), f32(g), f32(tab), f32(g_score), f32(out[TABLES]),
                         bias_summed ? nullptr : f32(parts), ws.data_ptr(), ws_bytes, B, T, S, Do, 0, st);
                    if (!bias_summed) column_sums.add(parts, f32(parts), out[OBIAS], Do, rows, dev, st);
                    bias_summed = true;
                } else
                    CALL(lffn_lookup_scatter_sorted_f32, cp, f32(score), f32(g), f32(out[TABLES]), ws.data_ptr(), ws_bytes, B, T, S, Do, 0, st);
            } else {
                if (need_score) CALL(lffn_lookup_inner_f32, cp, f32(g), f32(tab), f32(g_score), B, T, S, Do, st);
                if (need[TABLES]) CALL(lffn_lookup_scatter_f32, cp, f32(score), f32(g), f32(out[TABLES]), B, T, S, Do, 0, st);
            }
        }
        if (!bias_summed) column_sums.add(g, f32(g), out[OBIAS], Do, B, dev, st);
        if (!need_score) {
            column_sums.finish(st);
            return out;
        }

        const float decay = (float)c.decay, res = (float)c.residual, eps = (float)c.eps;
        Tensor g_h = empty_f32({R, B, H}, dev);            // gradient of the LayerNorm output, one slab per repeat
        if (c.form == DIAG) {
            const int64_t n = std::max<int64_t>(1, std::min(limits.project_partials, (B + 3) / 4));
            Tensor parts = empty_f32({n * R * (J + 1) * D}, dev);
            float *pd = f32(parts), *pb = pd + n * R * J * D;
            CALL(lffn_ln_project_hash_bwd_f32, f32(x_), f32(lw), f32(lb), eps, f32(w), f32(z_), f32(g_score), f32(g_h), pd, pb, B, H, D, R, J,
                 T, n, decay, res, st);
            if (need[WEIGHT] || need[PBIAS]) {
                Tensor g_w = at::empty_like(w), g_b = empty_f32({R * D}, dev);
                column_sums.add(parts, pd, g_w, R * J * D, n, dev, st);
                column_sums.add(parts, pb, g_b, R * D, n, dev, st);
                if (need[WEIGHT]) out[WEIGHT] = g_w;
                if (need[PBIAS]) out[PBIAS] = g_b.narrow(0, 0, T * 8);
            }
        } else {
            const Tensor stage = stage_in.unpack(self), st_ = stats.unpack(self), split = split_t.unpack(self);
            const int64_t parts = (B + 15) / 16;               // of the projection bias's gradient
            Tensor g_b = need[PBIAS] ? empty_f32({parts * T * 8}, dev) : Tensor();
            Tensor stage_g = empty_f32({R * J, B, D}, dev), g_folded = need[WEIGHT] ? empty_f32({R * J * D * 64}, dev) : Tensor();
            const int64_t blocks = R * J * (D / 64);
            CALL(lffn_bh4_block_score_bwd_split_f32, f32(z_), f32(g_score), f32(split), f32(g_h), f32(stage_g), need[PBIAS] ? f32(g_b) : nullptr,
                 need[WEIGHT] ? f32(g_folded) : nullptr, need[WEIGHT] ? R * J * D * 64 : 0, B, H, D, R, J, T, 64, decay, res, st);
            if (need[WEIGHT]) {
                CALL(lffn_ln_bh4_block_wgrad_f32, f32(stage_g), f32(x_), f32(lw), f32(lb), f32(st_), J > 1 ? f32(stage) : nullptr, f32(g_folded),
                     B, H, D, R, J, 64, st);
                out[WEIGHT] = at::empty_like(w);
                CALL(lffn_bh4_fold_mode_f32, f32(g_folded), f32(out[WEIGHT]), blocks, 64, 2, st);
            }
            if (need[PBIAS]) {
                out[PBIAS] = empty_f32({T * 8}, dev);
                column_sums.add(g_b, f32(g_b), out[PBIAS], T * 8, parts, dev, st);
            }
        }
        if (need_ln) {
            const int64_t n = std::max<int64_t>(1, std::min(limits.ln_partials, (B + 3) / 4));
            Tensor parts = empty_f32({2 * n * H}, dev), g_x = at::empty_like(x_), g_lw = empty_f32({H}, dev), g_lb = empty_f32({H}, dev);
            CALL(lffn_layer_norm_bwd_f32, f32(x_), f32(lw), eps, f32(g_h), f32(g_x), f32(parts), f32(parts) + n * H, B, H, R, n, st);
            column_sums.add(parts, f32(parts), g_lw, H, n, dev, st);
            column_sums.add(parts, f32(parts) + n * H, g_lb, H, n, dev, st);
            if (need[X]) out[X] = g_x;
            if (need[LN_W]) out[LN_W] = g_lw;
            if (need[LN_B]) out[LN_B] = g_lb;
        }
        column_sums.finish(st);
        return out;
    }
};

void train(const Config &c, const Params &p, const Tensor &x, const Tensor &residual, Tensor &out, int64_t B) {
    const at::Device dev = x.device();
    void *st = stream_on(dev);
    auto node = std::shared_ptr<LookupFFNBackward>(new LookupFFNBackward(), torch::autograd::deleteNode);
    const auto int32 = at::TensorOptions().dtype(at::kInt).device(dev);
    Tensor codes = at::empty({B, c.T}, int32), scores = empty_f32({B, c.T}, dev), z = empty_f32({B, c.T * 8}, dev), stage, stats, split_t;
    int32_t *cp = static_cast<int32_t *>(codes.data_ptr());
    const float eps = (float)c.eps, decay = (float)c.decay, res = (float)c.residual;
    if (c.form == DIAG) {
        CALL(lffn_ln_project_hash_f32, f32(x), f32(p[0]), f32(p[1]), eps, f32(p[2]), f32(p[3]), f32(z), cp, f32(scores), B, c.H, c.D,
             c.R, c.J, c.T, decay, res, st);
    } else {
        stage = empty_f32({c.R, c.J - 1, B, c.D}, dev);
        stats = empty_f32({B, 2}, dev);
        Tensor split = empty_f32({split_words(c)}, dev);
        split_t = empty_f32({split_words(c)}, dev);             // the backward's
        CALL(lffn_bh4_fold_split_both_f32, f32(p[2]), f32(split), f32(split_t), c.R * c.J, c.D / 64, 64, st);
        lffn_block_front front = block_front(c, p, split);
        front.codes = cp;
        front.scores = f32(scores);
        CALL(lffn_bh4_block_front_train_split_f32, &front, f32(x), f32(z), c.J > 1 ? f32(stage) : nullptr, f32(stats), B, st);
    }
    gather(c, codes, scores, p[4], p[5], f32(residual), out, B, plan_for(c, B, false), st);

    node->c = c;
    node->B = B;
    node->set_next_edges(torch::autograd::collect_next_edges(x, p[0], p[1], p[2], p[3], p[4], p[5], residual));
    node->x = SavedVariable(x, false);                      // (every one an input of the node or no part of the graph)
    node->ln_w = SavedVariable(p[0], false);
    node->ln_b = SavedVariable(p[1], false);
    node->weight = SavedVariable(p[2], false);
    node->tables = SavedVariable(p[4], false);
    node->codes = SavedVariable(codes, false);
    node->scores = SavedVariable(scores, false);
    node->z = SavedVariable(z, false);
    node->stage_in = SavedVariable(stage, false);
    node->stats = SavedVariable(stats, false);
    node->split_t = SavedVariable(split_t, false);
    torch::autograd::set_history(out, node);
}

// ---------------------------------------------------------------- Python

// Tangents exist inside a forward-mode level only (asking a tensor for its own takes a lock).
bool forward_mode() { return torch::autograd::ForwardADLevel::try_get_by_idx(0) != nullptr; }

// An ordinary tensor: no transform of torch.func around it, nothing lazy.
bool ordinary(const Tensor &t) {
    constexpr c10::DispatchKeySet other({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Python,
                                         c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});
    return t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(other);
}

bool has_tangent(const Tensor &t) { return t.defined() && t._fw_grad(/*level=*/0).defined(); }

// and of no subclass
bool plain(PyObject *o) { return THPVariable_CheckExact(o) && ordinary(THPVariable_Unpack(o)); }

// Somebody watches the operators that are called: a tracer, a mode of torch.overrides or torch.utils._python_dispatch, a
// transform of torch.func.  They see them on the Python path.
bool watched_over() {
    return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer) ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Functionalize);
}

// bind(path of the kernel library, nn.LayerNorm, BH4, the operators' thresholds)
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 4 && PyType_Check(args[1]) && PyType_Check(args[2]) && PyTuple_Check(args[3]) && PyTuple_GET_SIZE(args[3]) == 3,
                "bind: a path, two types and three numbers");
    const char *p = PyUnicode_AsUTF8(args[0]);
    if (!p) return nullptr;
    void *h = dlopen(p, RTLD_NOW | RTLD_NOLOAD);
    if (!h) h = dlopen(p, RTLD_NOW);
    TORCH_CHECK(h, "cannot load ", p, ": ", dlerror());
    Library found;
#define X(name)                                                            \
    found.name = reinterpret_cast<decltype(&::name)>(dlsym(h, #name));     \
    TORCH_CHECK(found.name, p, " has no ", #name);
    LFFN_ENTRIES(X)
#undef X
    Thresholds t{};
    for (int i = 0; i < 3; ++i)
        TORCH_CHECK(whole(PyTuple_GET_ITEM(args[3], i), (&t.ln_partials)[i]), "bind: a threshold is no integer");
    Py_INCREF(args[1]);
    Py_INCREF(args[2]);
    lib = found;
    limits = t;
    layer_norm_type = reinterpret_cast<PyTypeObject *>(args[1]);
    bh4_type = reinterpret_cast<PyTypeObject *>(args[2]);
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// The layer's sizes from those of its parameters; false when they do not fit together or are not of a kind the kernels are built for.
bool configure(const Parts &parts, const Params &p, const at::Device &dev, Config &c) {
    for (int i = 0; i < 6; ++i)
        if (!ordinary(p[i]) || p[i].device() != dev || !p[i].is_contiguous() || (i != 4 && p[i].scalar_type() != at::kFloat)) return false;
    const Tensor &lw = p[0], &lb = p[1], &w = p[2], &pb = p[3], &tables = p[4], &ob = p[5];
    if (w.dim() != 5 || tables.dim() != 3) return false;
    const auto fmt = tables.scalar_type();
    if (fmt != at::kFloat && fmt != at::kBFloat16 && fmt != at::kHalf) return false;
    const int64_t bs = w.size(4);
    c.form = bs == 64 ? BLOCK : DIAG;
    c.fmt = fmt == at::kFloat ? 0 : fmt == at::kBFloat16 ? 1 : 2;
    c.H = lw.numel();
    c.R = w.size(0); c.J = w.size(1); c.D = w.size(2) * bs;
    c.T = tables.size(0); c.S = tables.size(1); c.Do = tables.size(2);
    c.eps = parts.eps; c.decay = parts.decay; c.residual = 1.0 - parts.decay;
    if ((bs != 1 && bs != 64) || w.size(3) != bs || c.D < (bs == 64 ? 64 : 8) || c.D > 1024 || c.J < 1 || c.T < 1 || c.Do < 1) return false;
    // (8 T values for T tables are codes of 8 bits)
    if (c.T != parts.num_table || c.Do != parts.output_size || c.Do % 64 != 0 || c.S < 1 || (c.S & (c.S - 1)) != 0) return false;
    // the projection as BH4 makes it for a hidden size of H and T codes: D the next power of two, as few repeats as give 8 T outputs
    if (c.H > c.D || 2 * c.H <= c.D || (c.D & (c.D - 1)) != 0 || c.R != (8 * c.T + c.D - 1) / c.D) return false;
    if (lb.numel() != c.H || pb.numel() != 8 * c.T || ob.numel() != c.Do || (c.form == BLOCK && c.H % 4 != 0)) return false;
    c.one_launch = c.form == DIAG && c.D >= 256 && c.T <= 512 && c.S == 256;
    c.trainable = c.fmt == 0 && c.H % 4 == 0 && (c.form == BLOCK || (c.D >= 256 && c.J <= 4));
    return true;
}

// hash._folded = ((version, address, device), split weights, what they were folded from, stream, event), as Hashing keeps them for 8-bit
// codes: the split weights if they are w's and of this stream, on which they come before whatever is launched now.
Tensor split_of(PyObject *hash, const Tensor &w, int64_t words) {
    PyObject *kept = item(dict_of(hash), KEY_FOLDED);
    if (!kept || !PyTuple_Check(kept) || PyTuple_GET_SIZE(kept) != 5) return {};
    PyObject *key = PyTuple_GET_ITEM(kept, 0), *split = PyTuple_GET_ITEM(kept, 1);
    int64_t version = 0, address = 0, made_on = 0;
    if (!PyTuple_Check(key) || PyTuple_GET_SIZE(key) != 3 || !whole(PyTuple_GET_ITEM(key, 0), version) ||
        !whole(PyTuple_GET_ITEM(key, 1), address) || !whole(PyTuple_GET_ITEM(kept, 3), made_on) || !THPVariable_Check(split))
        return {};
    const hipStream_t stream = stream_on(w.device());
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (reinterpret_cast<hipStream_t>(made_on) != stream || hipStreamIsCapturing(stream, &capture) != hipSuccess ||
        capture != hipStreamCaptureStatusNone)
        return {};
    const Tensor &f = THPVariable_Unpack(split);
    const bool same = w._version() == (uint32_t)version && w.data_ptr() == reinterpret_cast<void *>(address) && f.device() == w.device() &&
                      f.numel() == words;
    return same ? f : Tensor();
}

// Other threads run while this one allocates and launches: either may wait (for memory, for room in a full queue).
struct WithoutInterpreter {
    PyThreadState *state = PyEval_SaveThread();
    ~WithoutInterpreter() { PyEval_RestoreThread(state); }
};

// forward(layer, x, residual or None, tokens up to which the one-launch form is taken[, split weights]) -> a tensor; None: not for
// this path; False: the split weights (Hashing.split_weight) are wanted
PyObject *forward(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 4 || n == 5, "forward: 4 or 5 arguments");
    if (watched_over() || !plain(args[1])) Py_RETURN_NONE;
    Tensor x = THPVariable_Unpack(args[1]);
    const at::Device dev = x.device();
    const int64_t dims = x.dim();
    Parts parts;
    if (dims < 1 || x.numel() == 0 || x.scalar_type() != at::kFloat || c10::hip::current_device() != dev.index() ||
        !find_parts(args[0], parts))
        Py_RETURN_NONE;
    Params params;
    for (int i = 0; i < 6; ++i) params[i] = THPVariable_Unpack(parts.params[i]);
    Config c{};
    if (!configure(parts, params, dev, c) || x.size(dims - 1) != c.H) Py_RETURN_NONE;
    const int64_t B = x.numel() / c.H;
    c10::SmallVector<int64_t, 6> sizes(x.sizes().begin(), x.sizes().end());
    sizes[dims - 1] = c.Do;
    Tensor residual;
    if (args[2] != Py_None) {
        if (!plain(args[2])) Py_RETURN_NONE;
        residual = THPVariable_Unpack(args[2]);
        if (residual.device() != dev || residual.numel() != B * c.Do) Py_RETURN_NONE;
    }
    if (forward_mode()) {
        bool any = has_tangent(x) || has_tangent(residual);
        for (const Tensor &t : params) any = any || has_tangent(t);
        if (any) Py_RETURN_NONE;
    }
    bool grads = false;
    if (at::GradMode::is_enabled()) {
        grads = x.requires_grad() || (residual.defined() && residual.requires_grad());
        for (const Tensor &t : params) grads = grads || t.requires_grad();
    }
    if (grads && !c.trainable) Py_RETURN_NONE;
    Tensor split;
    if (!grads && c.form == BLOCK) {
        if (n == 4) {
            split = split_of(parts.hash, params[2], split_words(c));
            if (!split.defined()) Py_RETURN_FALSE;
        } else {
            if (!plain(args[4])) Py_RETURN_NONE;
            split = THPVariable_Unpack(args[4]);
            if (split.device() != dev || split.scalar_type() != at::kFloat || split.numel() != split_words(c) || !split.is_contiguous())
                Py_RETURN_NONE;
        }
    }
    const int64_t fused_max = PyLong_AsLongLong(args[3]);
    if (fused_max == -1 && PyErr_Occurred()) return nullptr;
    Tensor out;
    {
        // (from here on only what is owned here is used: x, the residual, the parameters and the split weights)
        const WithoutInterpreter unlocked;
        // any layout of x and any shape and type of the residual, as the Python path makes them
        x = x.contiguous();
        if (residual.defined() && !(residual.scalar_type() == at::kFloat && residual.is_contiguous() && residual.sizes().equals(sizes)))
            residual = residual.reshape(sizes).to(at::kFloat).contiguous();
        if (reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
            (!residual.defined() || reinterpret_cast<uintptr_t>(residual.data_ptr()) % 16 == 0)) {
            out = empty_f32(sizes, dev);
            if (grads) train(c, params, x, residual, out, B);
            else infer(c, params, split, x, f32(residual), out, B, fused_max);
        }
    }
    if (!out.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(bind)), METH_FASTCALL, nullptr},
    {"forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(forward)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
    const std::pair<PyObject **, const char *> keys[] = {
        {&KEY_MODULES, "_modules"}, {&KEY_PARAMETERS, "_parameters"}, {&KEY_LAYER_NORM, "LayerNorm"}, {&KEY_HASH, "hash"},
        {&KEY_PROJECTION, "projection"}, {&KEY_WEIGHT, "weight"}, {&KEY_BIAS, "bias"}, {&KEY_TABLES, "tables"},
        {&KEY_EPS, "eps"}, {&KEY_DECAY, "decay_coeff"}, {&KEY_NUM_TABLE, "num_table"},
        {&KEY_OUTPUT_SIZE, "output_size"}, {&KEY_FOLDED, "_folded"},
    };
    for (const auto &[key, name] : keys)
        if (!(*key = PyUnicode_InternFromString(name))) return nullptr;
    PyObject *made = PyModule_Create(&module);
    if (made && PyModule_AddStringConstant(made, "torch_version", LFFN_TORCH_VERSION) != 0) Py_CLEAR(made);
    return made;
}
