// The layer's host path: LookupFFN.forward and its backward from Python's call to the kernels' launches.
//
// A layer call at a few hundred tokens is one launch of a few microseconds, a training step of that size about twenty;
// through the interpreter (argument checks, the operator dispatcher, foreign-function calls, two autograd functions) a call
// took 15 us and a step 400 us whatever the kernels took (17 tokens, and 385 tokens at hidden 512).  Here a call
// checks what can have changed since the layer's parameters were last looked at, allocates its result and launches; a
// training forward records one autograd node whose backward launches the whole chain.
//
// Python builds a handle (make_layer) when the parameters are of a kind the kernels are built for, and calls
// forward(handle, layer, x, residual, ...).  The answer is None whenever anything is not as the handle expects: a module or a
// parameter of another kind, another parameter object (each looked up through the layer's modules on every call), storage, dtype, sizes or strides, an input of another type, dtype, device or layout, a gradient wanted that this path does not
// compute.  Then the Python path runs, with its own checks and errors.
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
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>

#include <dlfcn.h>

#include <array>
#include <atomic>
#include <memory>
#include <string>
#include <vector>

#include "../../include/lookupffn_hip.h"

namespace {

using at::Tensor;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// The kernel library is the one Python has loaded (bind_library gets its path): its entry points by name.
#define LFFN_ENTRIES(X)                     \
    X(lffn_error_string)                    \
    X(lffn_lookup_ffn_fused_layer_rows)     \
    X(lffn_lookup_gather_records_plan_rows) \
    X(lffn_ln_project_hash_records_f32)     \
    X(lffn_ln_bh4_block_hash_records_f32)   \
    X(lffn_lookup_gather_records_rows)      \
    X(lffn_ln_project_hash_f32)             \
    X(lffn_ln_bh4_block_hash_f32)           \
    X(lffn_lookup_gather_workspace_bytes)   \
    X(lffn_lookup_gather_ws_f32)            \
    X(lffn_lookup_gather_ws_bf16)           \
    X(lffn_lookup_gather_ws_f16)            \
    X(lffn_ln_bh4_block_hash_train_f32)     \
    X(lffn_bh4_fold_mode_f32)               \
    X(lffn_lookup_scatter_workspace_bytes)  \
    X(lffn_lookup_backward_f32)             \
    X(lffn_lookup_inner_f32)                \
    X(lffn_lookup_scatter_f32)              \
    X(lffn_lookup_scatter_sorted_f32)       \
    X(lffn_ln_project_hash_bwd_f32)         \
    X(lffn_code_score_bwd_f32)              \
    X(lffn_bh4_block_bwd_f32)               \
    X(lffn_ln_bh4_block_wgrad_f32)          \
    X(lffn_layer_norm_bwd_f32)              \
    X(lffn_sum_partials_f32)

struct Library {
#define X(name) decltype(&::name) name = nullptr;
    LFFN_ENTRIES(X)
#undef X
} lib;

void check(int rc, const char *what) { TORCH_CHECK(rc == LFFN_OK, what, ": ", lib.lffn_error_string(rc), " (code ", rc, ")"); }
#define CALL(name, ...) check(lib.name(__VA_ARGS__), #name)

enum Form { DIAG = 0, BLOCK = 1 };

// Sizes and constants of a layer; the thresholds are the Python operators' own.  The last three are what the modules hold
// at the call.
struct Config {
    int64_t form, one_launch, H, D, R, J, T, S, Do, fmt;
    int64_t sorted_min_work, ln_partials, project_partials, sum_chunk_rows, trainable;
    double eps, decay, residual;
};

struct RecordPlan {
    int64_t B = -1, stride = 0, bytes = 0, ws_bytes = 0;
    int32_t tokens = 0;
};

// A parameter, and what it was when the handle was made.
struct Watched {
    PyObject *object;
    const void *data;
    at::ScalarType dtype;
    std::vector<int64_t> sizes, strides;

    bool same(const Tensor &t) const {
        return t.data_ptr() == data && t.scalar_type() == dtype && t.sizes().equals(sizes) && t.strides().equals(strides);
    }
};

// What the layer holds at this moment: it, its LayerNorm, its hash and the hash's projection as Python finds them on every
// access, the parameters in them (in the order of Input below) and their constants.  Borrowed references.
struct Parts {
    std::array<PyObject *, 4> modules;
    std::array<PyObject *, 6> params;
    double eps, decay;
};

PyObject *KEY_MODULES, *KEY_PARAMETERS, *KEY_LAYER_NORM, *KEY_HASH, *KEY_PROJECTION, *KEY_WEIGHT, *KEY_BIAS, *KEY_TABLES, *KEY_EPS,
    *KEY_DECAY;                           // interned

PyObject *dict_of(PyObject *o) {
    PyObject **d = o ? _PyObject_GetDictPtr(o) : nullptr;
    return d ? *d : nullptr;
}

PyObject *item(PyObject *dict, PyObject *key) { return dict && PyDict_Check(dict) ? PyDict_GetItem(dict, key) : nullptr; }

bool number(PyObject *o, double &value) {
    if (!o || !(PyFloat_Check(o) || PyLong_Check(o))) return false;
    value = PyFloat_AsDouble(o);
    if (value == -1.0 && PyErr_Occurred()) {             // an integer beyond double
        PyErr_Clear();
        return false;
    }
    return true;
}

// False when something is not where a LookupFFN has it (a reparametrised weight is no parameter but computed on every access).
bool find_parts(PyObject *layer, Parts &found) {
    PyObject *own = dict_of(layer), *modules = item(own, KEY_MODULES);
    PyObject *norm = item(modules, KEY_LAYER_NORM), *hash = item(modules, KEY_HASH);
    PyObject *projection = item(item(dict_of(hash), KEY_MODULES), KEY_PROJECTION);
    PyObject *of_layer = item(own, KEY_PARAMETERS), *of_norm = item(dict_of(norm), KEY_PARAMETERS),
             *of_projection = item(dict_of(projection), KEY_PARAMETERS);
    found.modules = {layer, norm, hash, projection};
    found.params = {item(of_norm, KEY_WEIGHT),       item(of_norm, KEY_BIAS),      item(of_projection, KEY_WEIGHT),
                    item(of_projection, KEY_BIAS), item(of_layer, KEY_TABLES), item(of_layer, KEY_BIAS)};
    for (PyObject *o : found.modules)
        if (!o) return false;
    for (PyObject *o : found.params)
        if (!o) return false;
    return number(item(dict_of(norm), KEY_EPS), found.eps) && number(item(dict_of(projection), KEY_DECAY), found.decay);
}

struct Layer {
    Config c{};
    std::array<PyTypeObject *, 4> types;  // of the modules
    std::vector<Watched> watched;
    // lnw, lnb, weight, pbias, tables, obias (pbias may be undefined)
    std::array<Tensor, 6> p;
    Tensor folded;                       // BLOCK inference: the folded weights and the weight's version they belong to
    uint32_t folded_version = 0;
    PyObject *folded_dict = nullptr, *folded_key = nullptr, *folded_object = nullptr;
    std::array<RecordPlan, 8> plans;     // a few batch sizes in turn; guarded by the interpreter lock
    int next_plan = 0;
};

float *f32(const Tensor &t) { return t.defined() ? static_cast<float *>(t.data_ptr()) : nullptr; }

hipStream_t stream_on(const at::Device &d) { return c10::hip::getCurrentHIPStream(d.index()).stream(); }

Tensor empty_f32(at::IntArrayRef sizes, const at::Device &d) { return at::empty(sizes, at::TensorOptions().dtype(at::kFloat).device(d)); }
Tensor empty_bytes(int64_t n, const at::Device &d) { return at::empty({n}, at::TensorOptions().dtype(at::kByte).device(d)); }

const RecordPlan &plan_for(Layer &l, int64_t B) {
    for (const RecordPlan &p : l.plans)
        if (p.B == B) return p;
    RecordPlan &p = l.plans[l.next_plan];
    l.next_plan = (l.next_plan + 1) % (int)l.plans.size();
    const Config &c = l.c;
    p = RecordPlan{};
    if (c.T % 2 == 0 && (c.form == BLOCK || c.D >= 16))
        CALL(lffn_lookup_gather_records_plan_rows, B, c.T, c.S, c.Do, (int32_t)c.fmt, &p.tokens, &p.stride, &p.bytes);
    if (p.bytes == 0) CALL(lffn_lookup_gather_workspace_bytes, B, c.T, c.S, c.Do, (int32_t)c.fmt, &p.ws_bytes);
    p.B = B;
    return p;
}

// Codes and scores [B, T] -> the gather, by whichever form the shape gets.
void gather(const Config &c, const Tensor &codes, const Tensor &scores, const Tensor &tables, const Tensor &obias, const float *residual,
            Tensor &out, int64_t B, int64_t ws_bytes, void *st) {
    Tensor ws;
    if (ws_bytes > 0) ws = empty_bytes(ws_bytes, out.device());
    void *wp = ws_bytes > 0 ? ws.data_ptr() : nullptr;
    const int32_t *cp = static_cast<const int32_t *>(codes.data_ptr());
    if (c.fmt == 0)
        CALL(lffn_lookup_gather_ws_f32, cp, f32(scores), f32(tables), f32(obias), residual, f32(out), wp, ws_bytes, B, c.T, c.S, c.Do, st);
    else if (c.fmt == 1)
        CALL(lffn_lookup_gather_ws_bf16, cp, f32(scores), static_cast<const uint16_t *>(tables.data_ptr()), f32(obias), residual, f32(out),
             wp, ws_bytes, B, c.T, c.S, c.Do, st);
    else
        CALL(lffn_lookup_gather_ws_f16, cp, f32(scores), static_cast<const uint16_t *>(tables.data_ptr()), f32(obias), residual, f32(out),
             wp, ws_bytes, B, c.T, c.S, c.Do, st);
}

void infer(Layer &l, const Config &c, const Tensor &x, const float *residual, Tensor &out, int64_t B, int64_t fused_max) {
    const at::Device dev = x.device();
    void *st = stream_on(dev);
    // (rows of 16 bits are half the traffic of a form that reads every token's rows from memory, and so good for half
    // as many tokens more: 768 tokens, 128 tables of 768 columns 34 us against 55 in two launches, 512 of 1024 113 against 120)
    if (c.one_launch && B <= (c.fmt == 0 ? fused_max : fused_max + fused_max / 2)) {
        const lffn_fused_layer layer{f32(l.p[0]), f32(l.p[1]), f32(l.p[2]), f32(l.p[3]), f32(l.p[4]), f32(l.p[5]), c.H, c.D, c.R, c.J, c.T,
                                     c.S, c.Do, (float)c.eps, (float)c.decay, (float)c.residual};
        CALL(lffn_lookup_ffn_fused_layer_rows, &layer, (int32_t)c.fmt, f32(x), residual, f32(out), B, st);
        return;
    }
    const float eps = (float)c.eps, decay = (float)c.decay, res = (float)c.residual;
    const RecordPlan plan = plan_for(l, B);
    if (plan.bytes > 0) {
        // many tokens: the projection kernel writes the gather kernel's record stream directly
        Tensor records = empty_bytes(plan.bytes, dev);
        uint32_t *rp = static_cast<uint32_t *>(records.data_ptr());
        if (c.form == DIAG)
            CALL(lffn_ln_project_hash_records_f32, f32(x), f32(l.p[0]), f32(l.p[1]), eps, f32(l.p[2]), f32(l.p[3]), rp, plan.stride,
                 plan.tokens, B, c.H, c.D, c.R, c.J, c.T, decay, res, st);
        else
            CALL(lffn_ln_bh4_block_hash_records_f32, f32(x), f32(l.p[0]), f32(l.p[1]), eps, f32(l.folded), f32(l.p[3]), rp, plan.stride,
                 plan.tokens, B, c.H, c.D, c.R, c.J, c.T, 64, decay, res, st);
        CALL(lffn_lookup_gather_records_rows, rp, plan.stride, l.p[4].data_ptr(), f32(l.p[5]), residual, f32(out), B, c.T, c.S, c.Do,
             (int32_t)c.fmt, plan.tokens, st);
        return;
    }
    Tensor codes = at::empty({B, c.T}, at::TensorOptions().dtype(at::kInt).device(dev)), scores = empty_f32({B, c.T}, dev);
    int32_t *cp = static_cast<int32_t *>(codes.data_ptr());
    if (c.form == DIAG)
        CALL(lffn_ln_project_hash_f32, f32(x), f32(l.p[0]), f32(l.p[1]), eps, f32(l.p[2]), f32(l.p[3]), nullptr, cp, f32(scores), B, c.H,
             c.D, c.R, c.J, c.T, decay, res, st);
    else
        CALL(lffn_ln_bh4_block_hash_f32, f32(x), f32(l.p[0]), f32(l.p[1]), eps, f32(l.folded), f32(l.p[3]), cp, f32(scores), B, c.H, c.D,
             c.R, c.J, c.T, 64, decay, res, st);
    gather(c, codes, scores, l.p[4], l.p[5], residual, out, B, plan.ws_bytes, st);
}

// Column sums of one or two [P, n] arrays of partial sums, fixed order of additions; many rows go through a first
// pass over chunks of rows on many workgroups.
void column_sums(const Config &c, const float *a, float *out_a, int64_t na, const float *b, float *out_b, int64_t nb, int64_t P,
                 const at::Device &dev, void *st) {
    Tensor mid;
    if (P > 4 * c.sum_chunk_rows) {
        int64_t chunks = (P + c.sum_chunk_rows - 1) / c.sum_chunk_rows;
        const int64_t each = (P + chunks - 1) / chunks;
        chunks = (P + each - 1) / each;                    // no empty chunk
        mid = empty_f32({chunks * (na + nb)}, dev);
        float *ma = f32(mid), *mb = nb ? ma + chunks * na : nullptr;
        CALL(lffn_sum_partials_f32, a, ma, na, b, mb, nb, P, chunks, st);
        a = ma; b = mb; P = chunks;
    }
    CALL(lffn_sum_partials_f32, a, out_a, na, b, out_b, nb, P, 1, st);
}

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
    SavedVariable x, ln_w, ln_b, weight, tables, codes, scores, z, stage_in, stats;

    std::string name() const override { return "LookupFFNBackward"; }

    void release_variables() override {
        for (SavedVariable *v : {&x, &ln_w, &ln_b, &weight, &tables, &codes, &scores, &z, &stage_in, &stats}) v->reset_data();
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
        if (need[OBIAS]) {
            out[OBIAS] = empty_f32({Do}, dev);
            column_sums(c, f32(g), f32(out[OBIAS]), Do, nullptr, nullptr, 0, B, dev, st);
        }
        const bool need_ln = need[X] || need[LN_W] || need[LN_B];
        const bool need_score = need_ln || need[WEIGHT] || need[PBIAS];
        // both gradients of the gather: one call with one workspace where the sorted scatter is the one to use
        Tensor g_score;
        if (need_score) g_score = empty_f32({B, T}, dev);
        if (need[TABLES]) out[TABLES] = at::empty_like(tab);
        if (need_score || need[TABLES]) {
            int64_t ws_bytes = 0;
            CALL(lffn_lookup_scatter_workspace_bytes, B, T, S, Do, &ws_bytes);
            if (B <= LFFN_SCATTER_LIST_TOKENS || B * T * Do < c.sorted_min_work) ws_bytes = 0;
            if (need[TABLES] && ws_bytes > 0) {
                Tensor ws = empty_bytes(ws_bytes, dev);
                if (need_score)
                    CALL(lffn_lookup_backward_f32, cp, f32(score), f32(g), f32(tab), f32(g_score), f32(out[TABLES]), ws.data_ptr(), ws_bytes, B,
                         T, S, Do, 0, st);
                else
                    CALL(lffn_lookup_scatter_sorted_f32, cp, f32(score), f32(g), f32(out[TABLES]), ws.data_ptr(), ws_bytes, B, T, S, Do, 0, st);
            } else {
                if (need_score) CALL(lffn_lookup_inner_f32, cp, f32(g), f32(tab), f32(g_score), B, T, S, Do, st);
                if (need[TABLES]) CALL(lffn_lookup_scatter_f32, cp, f32(score), f32(g), f32(out[TABLES]), B, T, S, Do, 0, st);
            }
        }
        if (!need_score) return out;

        const float decay = (float)c.decay, res = (float)c.residual, eps = (float)c.eps;
        Tensor g_h = empty_f32({R, B, H}, dev);            // gradient of the LayerNorm output, one slab per repeat
        if (c.form == DIAG) {
            const int64_t n = std::max<int64_t>(1, std::min(c.project_partials, (B + 3) / 4));
            Tensor parts = empty_f32({n * R * (J + 1) * D}, dev);
            float *pd = f32(parts), *pb = pd + n * R * J * D;
            CALL(lffn_ln_project_hash_bwd_f32, f32(x_), f32(lw), f32(lb), eps, f32(w), f32(z_), f32(g_score), f32(g_h), pd, pb, B, H, D, R, J,
                 T, n, decay, res, st);
            if (need[WEIGHT] || need[PBIAS]) {
                Tensor g_w = at::empty_like(w), g_b = empty_f32({R * D}, dev);
                column_sums(c, pd, f32(g_w), R * J * D, pb, f32(g_b), R * D, n, dev, st);
                if (need[WEIGHT]) out[WEIGHT] = g_w;
                if (need[PBIAS]) out[PBIAS] = g_b.narrow(0, 0, T * 8);
            }
        } else {
            const Tensor stage = stage_in.unpack(self), st_ = stats.unpack(self);
            Tensor g_z = empty_f32({B, T * 8}, dev), stage_g = empty_f32({R * J, B, D}, dev), folded = at::empty_like(w);
            CALL(lffn_code_score_bwd_f32, f32(z_), f32(g_score), f32(g_z), B * T, 8, st);
            const int64_t blocks = R * J * (D / 64);
            CALL(lffn_bh4_fold_mode_f32, f32(w), f32(folded), blocks, 64, 1, st);
            CALL(lffn_bh4_block_bwd_f32, f32(g_z), f32(folded), f32(g_h), f32(stage_g), B, H, D, R, J, T, 64, decay, res, st);
            if (need[WEIGHT]) {
                Tensor g_folded = at::zeros({R * J, D / 64, 64, 64}, at::TensorOptions().dtype(at::kFloat).device(dev));
                CALL(lffn_ln_bh4_block_wgrad_f32, f32(stage_g), f32(x_), f32(lw), f32(lb), f32(st_), J > 1 ? f32(stage) : nullptr, f32(g_folded),
                     B, H, D, R, J, 64, st);
                out[WEIGHT] = at::empty_like(w);
                CALL(lffn_bh4_fold_mode_f32, f32(g_folded), f32(out[WEIGHT]), blocks, 64, 2, st);
            }
            if (need[PBIAS]) {
                out[PBIAS] = empty_f32({T * 8}, dev);
                column_sums(c, f32(g_z), f32(out[PBIAS]), T * 8, nullptr, nullptr, 0, B, dev, st);
            }
        }
        if (need_ln) {
            const int64_t n = std::max<int64_t>(1, std::min(c.ln_partials, (B + 3) / 4));
            Tensor parts = empty_f32({2 * n * H}, dev), g_x = at::empty_like(x_), g_lw = empty_f32({H}, dev), g_lb = empty_f32({H}, dev);
            CALL(lffn_layer_norm_bwd_f32, f32(x_), f32(lw), eps, f32(g_h), f32(g_x), f32(parts), f32(parts) + n * H, B, H, R, n, st);
            column_sums(c, f32(parts), f32(g_lw), H, f32(parts) + n * H, f32(g_lb), H, n, dev, st);
            if (need[X]) out[X] = g_x;
            if (need[LN_W]) out[LN_W] = g_lw;
            if (need[LN_B]) out[LN_B] = g_lb;
        }
        return out;
    }
};

void train(Layer &l, const Config &c, const Tensor &x, const Tensor &residual, Tensor &out, int64_t B) {
    const at::Device dev = x.device();
    void *st = stream_on(dev);
    auto node = std::shared_ptr<LookupFFNBackward>(new LookupFFNBackward(), torch::autograd::deleteNode);
    const auto int32 = at::TensorOptions().dtype(at::kInt).device(dev);
    Tensor codes = at::empty({B, c.T}, int32), scores = empty_f32({B, c.T}, dev), z = empty_f32({B, c.T * 8}, dev), stage, stats;
    int32_t *cp = static_cast<int32_t *>(codes.data_ptr());
    const float eps = (float)c.eps, decay = (float)c.decay, res = (float)c.residual;
    if (c.form == DIAG) {
        CALL(lffn_ln_project_hash_f32, f32(x), f32(l.p[0]), f32(l.p[1]), eps, f32(l.p[2]), f32(l.p[3]), f32(z), cp, f32(scores), B, c.H, c.D,
             c.R, c.J, c.T, decay, res, st);
    } else {
        stage = empty_f32({c.R, c.J - 1, B, c.D}, dev);
        stats = empty_f32({B, 2}, dev);
        Tensor folded = at::empty_like(l.p[2]);
        CALL(lffn_bh4_fold_mode_f32, f32(l.p[2]), f32(folded), c.R * c.J * (c.D / 64), 64, 0, st);
        CALL(lffn_ln_bh4_block_hash_train_f32, f32(x), f32(l.p[0]), f32(l.p[1]), eps, f32(folded), f32(l.p[3]), cp, f32(scores), f32(z),
             c.J > 1 ? f32(stage) : nullptr, f32(stats), B, c.H, c.D, c.R, c.J, c.T, 64, decay, res, st);
    }
    int64_t ws_bytes = 0;
    CALL(lffn_lookup_gather_workspace_bytes, B, c.T, c.S, c.Do, (int32_t)c.fmt, &ws_bytes);
    gather(c, codes, scores, l.p[4], l.p[5], f32(residual), out, B, ws_bytes, st);

    node->c = c;
    node->B = B;
    node->set_next_edges(torch::autograd::collect_next_edges(x, l.p[0], l.p[1], l.p[2], l.p[3], l.p[4], l.p[5], residual));
    node->x = SavedVariable(x, false);                      // (every one an input of the node or no part of the graph)
    node->ln_w = SavedVariable(l.p[0], false);
    node->ln_b = SavedVariable(l.p[1], false);
    node->weight = SavedVariable(l.p[2], false);
    node->tables = SavedVariable(l.p[4], false);
    node->codes = SavedVariable(codes, false);
    node->scores = SavedVariable(scores, false);
    node->z = SavedVariable(z, false);
    node->stage_in = SavedVariable(stage, false);
    node->stats = SavedVariable(stats, false);
    torch::autograd::set_history(out, node);
}

// ---------------------------------------------------------------- Python

const char *CAPSULE = "lookupffn_amd.layer";

void free_layer(PyObject *capsule) {
    Layer *l = static_cast<Layer *>(PyCapsule_GetPointer(capsule, CAPSULE));
    if (!l) return;
    for (Watched &w : l->watched) Py_XDECREF(w.object);
    for (PyTypeObject *t : l->types) Py_XDECREF(t);
    Py_XDECREF(l->folded_dict);
    Py_XDECREF(l->folded_key);
    Py_XDECREF(l->folded_object);
    delete l;
}

// An ordinary tensor: no transform of torch.func around it, nothing lazy, no tangent.
bool ordinary(const Tensor &t) {
    constexpr c10::DispatchKeySet other({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Python,
                                         c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});
    return t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(other) && !t._fw_grad(/*level=*/0).defined();
}

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

PyObject *bind_library(PyObject *, PyObject *path) {
    HANDLE_TH_ERRORS
    const char *p = PyUnicode_AsUTF8(path);
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
    lib = found;
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// make_layer(config: 15 ints, layer, folded: (dict, key, object, tensor, version) or None) -> handle, or None when the
// layer has not the parameters it was made with
PyObject *make_layer(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 3, "make_layer: 3 arguments");
    Parts parts;
    if (!find_parts(args[1], parts)) Py_RETURN_NONE;
    for (PyObject *o : parts.params)
        if (o != Py_None && !(THPVariable_Check(o) && ordinary(THPVariable_Unpack(o)))) Py_RETURN_NONE;
    auto l = std::make_unique<Layer>();
    int64_t *ints = &l->c.form;
    TORCH_CHECK(PyTuple_GET_SIZE(args[0]) == 15, "make_layer: sizes");
    for (int i = 0; i < 15; ++i) ints[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(args[0], i));
    if (PyErr_Occurred()) return nullptr;
    for (int i = 0; i < 4; ++i) {
        l->types[i] = Py_TYPE(parts.modules[i]);
        Py_INCREF(l->types[i]);
    }
    for (int i = 0; i < 6; ++i) {
        PyObject *o = parts.params[i];
        if (o != Py_None) l->p[i] = THPVariable_Unpack(o);
        Py_INCREF(o);
        Watched w{o, nullptr, at::kFloat, {}, {}};
        if (const Tensor &t = l->p[i]; t.defined()) {
            w.data = t.data_ptr();
            w.dtype = t.scalar_type();
            w.sizes = t.sizes().vec();
            w.strides = t.strides().vec();
        }
        l->watched.push_back(std::move(w));
    }
    if (args[2] != Py_None) {
        l->folded_dict = PyTuple_GET_ITEM(args[2], 0);
        l->folded_key = PyTuple_GET_ITEM(args[2], 1);
        l->folded_object = PyTuple_GET_ITEM(args[2], 2);
        for (PyObject *k : {l->folded_dict, l->folded_key, l->folded_object}) Py_INCREF(k);
        l->folded = THPVariable_Unpack(PyTuple_GET_ITEM(args[2], 3));
        l->folded_version = (uint32_t)PyLong_AsUnsignedLong(PyTuple_GET_ITEM(args[2], 4));
    }
    PyObject *capsule = PyCapsule_New(l.get(), CAPSULE, free_layer);
    if (capsule) l.release();
    return capsule;
    END_HANDLE_TH_ERRORS
}

// forward(handle, layer, x, residual or None, tokens up to which the one-launch form is taken) -> tensor or None
PyObject *forward(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 5, "forward: 5 arguments");
    Layer *l = static_cast<Layer *>(PyCapsule_GetPointer(args[0], CAPSULE));
    if (!l) return nullptr;
    Parts parts;
    if (!find_parts(args[1], parts)) Py_RETURN_NONE;
    Config c = l->c;
    c.eps = parts.eps;
    c.decay = parts.decay;
    c.residual = 1.0 - parts.decay;
    if (watched_over() || !plain(args[2])) Py_RETURN_NONE;
    const Tensor &x = THPVariable_Unpack(args[2]);
    const at::Device dev = l->p[4].device();
    const int64_t dims = x.dim();
    if (dims < 1 || x.size(dims - 1) != c.H || x.numel() == 0 || x.scalar_type() != at::kFloat || !x.is_contiguous() || x.device() != dev ||
        c10::hip::current_device() != dev.index())
        Py_RETURN_NONE;
    const int64_t B = x.numel() / c.H;
    if (reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 != 0) Py_RETURN_NONE;
    c10::SmallVector<int64_t, 6> sizes(x.sizes().begin(), x.sizes().end());
    sizes[dims - 1] = c.Do;
    Tensor residual;
    if (args[3] != Py_None) {
        if (!plain(args[3])) Py_RETURN_NONE;
        residual = THPVariable_Unpack(args[3]);
        if (residual.scalar_type() != at::kFloat || residual.device() != dev || !residual.is_contiguous() || !residual.sizes().equals(sizes) ||
            reinterpret_cast<uintptr_t>(residual.data_ptr()) % 16 != 0)
            Py_RETURN_NONE;
    }
    bool grads = false;
    const bool grad_mode = at::GradMode::is_enabled();
    if (grad_mode) grads = x.requires_grad() || (residual.defined() && residual.requires_grad());
    for (size_t i = 0; i < l->types.size(); ++i)
        if (Py_TYPE(parts.modules[i]) != l->types[i]) Py_RETURN_NONE;
    for (size_t i = 0; i < l->watched.size(); ++i) {
        const Watched &w = l->watched[i];
        if (parts.params[i] != w.object) Py_RETURN_NONE;
        const Tensor &p = l->p[i];
        if (!p.defined()) continue;
        if (!ordinary(p) || !w.same(p)) Py_RETURN_NONE;
        if (grad_mode) grads = grads || p.requires_grad();
    }
    if (grads && !c.trainable) Py_RETURN_NONE;
    if (!grads && c.form == BLOCK &&
        (!l->folded.defined() || PyDict_GetItem(l->folded_dict, l->folded_key) != l->folded_object || l->p[2]._version() != l->folded_version))
        Py_RETURN_NONE;
    Tensor out = empty_f32(sizes, dev);
    if (grads) train(*l, c, x, residual, out, B);
    else infer(*l, c, x, f32(residual), out, B, PyLong_AsLongLong(args[4]));
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"bind_library", bind_library, METH_O, nullptr},
    {"make_layer", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(make_layer)), METH_FASTCALL, nullptr},
    {"forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(forward)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
    const std::pair<PyObject **, const char *> keys[] = {
        {&KEY_MODULES, "_modules"}, {&KEY_PARAMETERS, "_parameters"}, {&KEY_LAYER_NORM, "LayerNorm"}, {&KEY_HASH, "hash"},
        {&KEY_PROJECTION, "projection"}, {&KEY_WEIGHT, "weight"}, {&KEY_BIAS, "bias"}, {&KEY_TABLES, "tables"},
        {&KEY_EPS, "eps"}, {&KEY_DECAY, "decay_coeff"},
    };
    for (const auto &[key, name] : keys)
        if (!(*key = PyUnicode_InternFromString(name))) return nullptr;
    return PyModule_Create(&module);
}
