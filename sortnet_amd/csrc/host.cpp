// Host side of the autograd front-end: argument checks, output allocation, graph nodes and the calls into the C ABI
// (include/sortdist.h), one C++ function per op of sortnet_amd/functional.py.
//
// Why native: a small layer (128 x 3072 x 1024) keeps the device busy for 50 us per forward and backward, and the same
// calls made from Python (autograd.Function, a device context, a dozen checked ctypes arguments per entry point, the
// backward once more through the interpreter) took 120 us of host time, so the host set the pace.  Here a call
// is a few tensor headers, one graph node and the launches; the backward runs on autograd's own thread without the
// interpreter.  Tensors stay torch's: outputs come from its caching allocator and work is queued on its current
// stream.
#include <cmath>
#include <mutex>
#include <stdexcept>
#include <string>

#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/utils/pybind.h>

#include "../../include/sortdist.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::collect_next_edges;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::set_history;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

namespace {

// ---- arguments --------------------------------------------------------------------------------------------------
template <class T>
T* data(const Tensor& t, const char* name, at::ScalarType type) {
    if (!t.is_cuda()) throw std::runtime_error(std::string(name) + " must be a CUDA tensor");
    if (!t.is_contiguous()) throw std::runtime_error(std::string(name) + " must be contiguous");
    if (t.scalar_type() != type)
        throw std::runtime_error(std::string(name) + " must have dtype " + (type == at::kFloat ? "torch.float32" : "torch.int32"));
    return static_cast<T*>(t.data_ptr());
}
float* floats(const Tensor& t, const char* name) { return data<float>(t, name, at::kFloat); }
int* ints(const Tensor& t, const char* name) { return data<int>(t, name, at::kInt); }
int* ints(const OptTensor& t, const char* name) { return t && t->defined() ? ints(*t, name) : nullptr; }

void require(int rc, const char* who) {
    if (rc == 0) return;
    const char* msg = sd_last_error();
    throw std::runtime_error(std::string(who) + " failed (status " + std::to_string(rc) + "): " + (msg ? msg : "?"));
}

// torch's current stream on t's GPU (queried while the arguments of an entry point are formed, perhaps before t is checked)
sd_stream_t stream_of(const Tensor& t) {
    if (!t.is_cuda()) throw std::runtime_error("input must be a CUDA tensor");
    return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// sizes of a layer call on x (B, C, HW)
struct Dims {
    int B, CI, HW, CO, G;
    Dims(const Tensor& x, int64_t groups, int64_t channels)
        : B((int)x.size(0)), CI((int)x.size(1)), HW((int)x.size(2)), CO((int)channels), G((int)groups) {}
};

Tensor new_floats(const Tensor& like, at::IntArrayRef size) { return at::empty(size, like.options().dtype(at::kFloat)); }
Tensor new_ints(const Tensor& like, at::IntArrayRef size) { return at::empty(size, like.options().dtype(at::kInt)); }
Tensor new_out(const Tensor& x, int64_t channels) { return new_floats(x, {x.size(0), channels, x.size(2)}); }

// The nodes below hold backward formulas and nothing else.  An input with a forward-mode tangent would come out without
// one, which a caller reads as a zero derivative, and the kernels know nothing of the wrapped tensors of torch.func: both
// are refused, as an autograd function without `jvp` and `setup_context` refuses them.
template <class... T>
void reverse_mode_only(const char* who, const T&... t) {
    if (c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))   // inside a transform
        throw std::runtime_error(std::string("sortnet_amd.") + who + " does not support the transforms of torch.func (vmap, grad, jvp, ...)");
    TORCH_CHECK_NOT_IMPLEMENTED(!(... || (t.defined() && t._fw_grad(0).defined())),
                                "sortnet_amd.", who, " does not support forward mode AD: an input carries a tangent");
}

template <class... T>
bool want_grad(const T&... t) { return at::GradMode::is_enabled() && (t.requires_grad() || ...); }

// Every node takes its mutex_ while it reads or frees what it saved: two threads may run backward through a graph that they
// share.  Saved tensors are unpacked before autograd is switched off, since the caller's unpack hooks run inside.
using Locked = std::lock_guard<std::mutex>;

// The gradient that flows into output `i` of a node, zeros where none does (an op behind it that has no gradient to give):
// the inputs then get zeros and not nothing.
Tensor incoming(const Node& node, const variable_list& grads, int i) {
    return grads[i].defined() ? grads[i].contiguous() : node.input_metadata(i).zeros_like();
}

template <class N>
std::shared_ptr<N> new_node() { return std::shared_ptr<N>(new N(), torch::autograd::deleteNode); }

// ---- l-inf, masked and l-p layers: x, weight -> y -----------------------------------------------------------------
// A node has two edges, x and weight; `kind` names the backward entry points.
struct DistNode : Node {
    enum Kind { MAX, SORT, POWER } kind;
    SavedVariable x, weight, state;            // state: positions (MAX, SORT) or the output (POWER)
    SavedVariable ci, co;
    int groups, truncate = 0;
    double p = 0, q = 0;

    variable_list apply(variable_list&& grads) override {
        const Locked lock(mutex_);
        variable_list out(2);
        const bool want_w = task_should_compute_output(1), want_x = task_should_compute_output(0);
        if (!want_w && !want_x) return out;
        const Tensor xs = x.unpack(), ws = weight.unpack(), st = state.unpack(shared_from_this());
        const Tensor cis = ci.unpack(), cos = co.unpack();
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor g = incoming(*this, grads, 0);
        const c10::DeviceGuard guard(g.device());
        const int B = (int)g.size(0), CO = (int)g.size(1), HW = (int)g.size(2), CI = (int)xs.size(1), G = groups;
        const int W_CO = (int)ws.size(0), W_CI = (int)ws.size(1) * G;
        Tensor gx = at::empty(xs.sizes(), xs.options()), gw;
        const float* gp = floats(g, "grad_output");
        const int *cip = cis.defined() ? ints(cis, "w_index_ci") : nullptr, *cop = cos.defined() ? ints(cos, "w_index_co") : nullptr;
        const sd_stream_t s = stream_of(g);
        if (want_w) gw = at::empty(ws.sizes(), ws.options());
        float *gxp = floats(gx, "grad_input"), *gwp = want_w ? floats(gw, "grad_weight") : nullptr;
        if (kind == MAX) {
            const int* pos = ints(st, "pos");
            if (want_w) require(sd_inf_dist_backward_input_weight(gp, pos, B, CO, CI, G, HW, gxp, gwp, cip, cop, W_CO, W_CI, s),
                                "sd_inf_dist_backward_input_weight");
            else require(sd_inf_dist_backward_input(gp, pos, B, CO, CI, G, HW, gxp, s), "sd_inf_dist_backward_input");
        } else if (kind == SORT) {
            const int* pos = ints(st, "pos");
            if (want_w) require(sd_sort_neuron_backward_input_weight(gp, pos, B, CO, CI, G, HW, gxp, gwp, (float)q, truncate, s),
                                "sd_sort_neuron_backward_input_weight");
            else require(sd_sort_neuron_backward_input(gp, pos, B, CO, CI, G, HW, gxp, (float)q, truncate, s),
                         "sd_sort_neuron_backward_input");
        } else {
            const float *xp = floats(xs, "input"), *wp = floats(ws, "weight"), *yp = floats(st, "output");
            if (want_w) require(sd_norm_dist_backward_input_weight(gp, xp, wp, yp, B, CO, CI, G, HW, gxp, gwp, (float)p, cip, cop,
                                                                   W_CO, W_CI, s), "sd_norm_dist_backward_input_weight");
            else require(sd_norm_dist_backward_input(gp, xp, wp, yp, B, CO, CI, G, HW, gxp, (float)p, cip, cop, W_CO, W_CI, s),
                         "sd_norm_dist_backward_input");
        }
        if (want_x) out[0] = gx;
        if (want_w) out[1] = gw;
        return out;
    }
    void release_variables() override {
        const Locked lock(mutex_);
        x.reset_data(); weight.reset_data(); state.reset_data(); ci.reset_data(); co.reset_data();
    }
    std::string name() const override { return "DistNode"; }
};

// makes y the output of a node over (x, weight); the caller adds what its kind needs
std::shared_ptr<DistNode> attach(const Tensor& x, const Tensor& w, int64_t groups, DistNode::Kind kind) {
    auto node = new_node<DistNode>();
    node->set_next_edges(collect_next_edges(x, w));
    node->kind = kind;
    node->groups = (int)groups;
    node->x = SavedVariable(x, false);
    node->weight = SavedVariable(w, false);
    return node;
}

Tensor norm_dist_lists(const Tensor& x, const Tensor& w, const OptTensor& ci, const OptTensor& co, int64_t groups, double p,
                       bool lists) {
    reverse_mode_only("norm_dist", x, w);
    const bool grad = want_grad(x, w);
    const int64_t channels = co && co->defined() ? co->size(-1) * groups : w.size(0);
    Tensor y, pos;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(x.device());
        y = new_out(x, channels);
        const Dims d(x, groups, channels);
        const float *xp = floats(x, "input"), *wp = floats(w, "weight");
        const int *cip = ints(ci, "w_index_ci"), *cop = ints(co, "w_index_co");
        const int W_CO = (int)w.size(0), W_CI = (int)(w.size(1) * groups);
        if (std::isinf(p)) {
            if (grad || lists) {
                pos = new_ints(x, y.sizes());
                require(sd_inf_dist_forward(xp, wp, d.B, d.CO, d.CI, d.G, d.HW, floats(y, "output"), ints(pos, "pos"), cip, cop,
                                            W_CO, W_CI, stream_of(x)), "sd_inf_dist_forward");
            } else
                require(sd_inf_dist_forward_nograd(xp, wp, d.B, d.CO, d.CI, d.G, d.HW, floats(y, "output"), stream_of(x)),
                        "sd_inf_dist_forward_nograd");
        } else
            require(sd_norm_dist_forward(xp, wp, d.B, d.CO, d.CI, d.G, d.HW, floats(y, "output"), (float)p, cip, cop, W_CO, W_CI,
                                         stream_of(x)), "sd_norm_dist_forward");
    }
    if (grad) {
        const bool power = !std::isinf(p);
        auto node = attach(x, w, groups, power ? DistNode::POWER : DistNode::MAX);
        node->p = p;
        if (ci && ci->defined()) node->ci = SavedVariable(*ci, false);
        if (co && co->defined()) node->co = SavedVariable(*co, false);
        set_history(y, node);
        node->state = power ? SavedVariable(y, true) : SavedVariable(pos, false);
    }
    return y;
}

Tensor norm_dist(const Tensor& x, const Tensor& w, int64_t groups, double p) {
    return norm_dist_lists(x, w, {}, {}, groups, p, false);
}
Tensor norm_dist_dropout(const Tensor& x, const Tensor& w, const OptTensor& ci, const OptTensor& co, int64_t groups, double p) {
    return norm_dist_lists(x, w, ci, co, groups, p, true);
}

Tensor masked_inf_dist(const Tensor& x, const Tensor& w, int64_t groups, double q, uint32_t seed, int mode) {
    reverse_mode_only("masked_inf_dist", x, w);
    const bool grad = want_grad(x, w);
    Tensor y, pos;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(x.device());
        y = new_out(x, w.size(0));
        if (grad) pos = new_ints(x, y.sizes());
        const Dims d(x, groups, w.size(0));
        require(sd_masked_inf_dist_forward(floats(x, "input"), floats(w, "weight"), d.B, d.CO, d.CI, d.G, d.HW, floats(y, "output"),
                                           grad ? ints(pos, "pos") : nullptr, (float)q, seed, mode, stream_of(x)),
                "sd_masked_inf_dist_forward");
    }
    if (grad) {
        auto node = attach(x, w, groups, DistNode::MAX);
        set_history(y, node);
        node->state = SavedVariable(pos, false);
    }
    return y;
}

Tensor sort_neuron(const Tensor& x, const Tensor& w, int64_t groups, double q, int truncate) {
    reverse_mode_only("sort_neuron", x, w);
    const bool grad = want_grad(x, w);
    Tensor y, pos;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(x.device());
        y = new_out(x, w.size(0));
        const Dims d(x, groups, w.size(0));
        const float *xp = floats(x, "input"), *wp = floats(w, "weight");
        if (grad) {
            pos = new_ints(x, {(int64_t)truncate, x.size(0), w.size(0), x.size(2)});
            require(sd_sort_neuron_forward(xp, wp, d.B, d.CO, d.CI, d.G, d.HW, floats(y, "output"), ints(pos, "pos"), (float)q,
                                           truncate, stream_of(x)), "sd_sort_neuron_forward");
        } else
            require(sd_sort_neuron_forward_nograd(xp, wp, d.B, d.CO, d.CI, d.G, d.HW, floats(y, "output"), (float)q, truncate,
                                                  stream_of(x)), "sd_sort_neuron_forward_nograd");
    }
    if (grad) {
        auto node = attach(x, w, groups, DistNode::SORT);
        node->q = q; node->truncate = truncate;
        set_history(y, node);
        node->state = SavedVariable(pos, false);
    }
    return y;
}

// ---- interval bounds: lower, upper, weight -> lower, upper -----------------------------------------------------------
struct BoundNode : Node {
    SavedVariable xl, xu, weight, pl, pu;
    int groups = 1;

    variable_list apply(variable_list&& grads) override {
        const Locked lock(mutex_);
        variable_list out(3);
        const bool want_l = task_should_compute_output(0), want_u = task_should_compute_output(1), want_w = task_should_compute_output(2);
        if (!want_l && !want_u && !want_w) return out;
        const Tensor l = xl.unpack(), u = xu.unpack(), w = weight.unpack(), posl = pl.unpack(), posu = pu.unpack();
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor gl = incoming(*this, grads, 0), gu = incoming(*this, grads, 1);
        const c10::DeviceGuard guard(l.device());
        const int B = (int)gl.size(0), CO = (int)gl.size(1), HW = (int)gl.size(2), CI = (int)l.size(1);
        // One bound alone, with a frozen weight, gets no gradient from this op (core/norm_dist.py:157-173: zeros).  What
        // counts is which inputs require a gradient (should_compute_output: the graph's edges), not which of them this
        // backward pass asks for (task_should_compute_output).
        if (!should_compute_output(2) && !(should_compute_output(0) && should_compute_output(1))) {
            if (want_l) out[0] = at::zeros_like(l);
            if (want_u) out[1] = at::zeros_like(u);
            return out;
        }
        // the entry points write every element of the three gradients
        Tensor gxl = at::empty(l.sizes(), l.options()), gxu = at::empty(u.sizes(), u.options());
        const float *glp = floats(gl, "grad_outputL"), *gup = floats(gu, "grad_outputU");
        const int *plp = ints(posl, "posL"), *pup = ints(posu, "posU");
        if (want_w) {
            out[2] = at::empty(w.sizes(), w.options());
            require(sd_bound_inf_dist_backward_input_weight(glp, gup, plp, pup, B, CO, CI, groups, HW, floats(gxl, "grad_inputL"),
                                                            floats(gxu, "grad_inputU"), floats(out[2], "grad_weight"), stream_of(l)),
                    "sd_bound_inf_dist_backward_input_weight");
        } else
            require(sd_bound_inf_dist_backward_input(glp, gup, plp, pup, B, CO, CI, groups, HW, floats(gxl, "grad_inputL"),
                                                     floats(gxu, "grad_inputU"), stream_of(l)), "sd_bound_inf_dist_backward_input");
        if (want_l) out[0] = gxl;
        if (want_u) out[1] = gxu;
        return out;
    }
    void release_variables() override {
        const Locked lock(mutex_);
        xl.reset_data(); xu.reset_data(); weight.reset_data(); pl.reset_data(); pu.reset_data();
    }
    std::string name() const override { return "BoundNode"; }
};

std::pair<Tensor, Tensor> bound_inf_dist(const Tensor& xl, const Tensor& xu, const Tensor& w, int64_t groups) {
    reverse_mode_only("bound_inf_dist", xl, xu, w);
    const bool grad = want_grad(xl, xu, w);
    Tensor lo, up, pl, pu;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(xl.device());
        lo = new_out(xl, w.size(0));
        up = new_out(xl, w.size(0));
        const Dims d(xl, groups, w.size(0));
        const float *lp = floats(xl, "inputL"), *upp = floats(xu, "inputU"), *wp = floats(w, "weight");
        if (grad) {
            pl = new_ints(xl, lo.sizes());
            pu = new_ints(xl, lo.sizes());
            require(sd_bound_inf_dist_forward(lp, upp, wp, d.B, d.CO, d.CI, d.G, d.HW, floats(lo, "outputL"), floats(up, "outputU"),
                                              ints(pl, "posL"), ints(pu, "posU"), stream_of(xl)), "sd_bound_inf_dist_forward");
        } else
            require(sd_bound_inf_dist_forward_nograd(lp, upp, wp, d.B, d.CO, d.CI, d.G, d.HW, floats(lo, "outputL"),
                                                     floats(up, "outputU"), stream_of(xl)), "sd_bound_inf_dist_forward_nograd");
    }
    if (grad) {
        auto node = new_node<BoundNode>();
        node->set_next_edges(collect_next_edges(xl, xu, w));
        node->groups = (int)groups;
        node->xl = SavedVariable(xl, false); node->xu = SavedVariable(xu, false); node->weight = SavedVariable(w, false);
        node->pl = SavedVariable(pl, false); node->pu = SavedVariable(pu, false);
        set_history(variable_list{lo, up}, node);
    }
    return {lo, up};
}

std::pair<Tensor, Tensor> bound_sort_neuron(const Tensor& xl, const Tensor& xu, const Tensor& w, int64_t groups, double q,
                                            int truncate) {
    reverse_mode_only("bound_sort_neuron", xl, xu, w);
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(xl.device());
    Tensor lo = new_out(xl, w.size(0)), up = new_out(xl, w.size(0));
    const Dims d(xl, groups, w.size(0));
    require(sd_bound_sort_neuron_forward(floats(xl, "inputL"), floats(xu, "inputU"), floats(w, "weight"), d.B, d.CO, d.CI, d.G, d.HW,
                                         floats(lo, "outputL"), floats(up, "outputU"), (float)q, truncate, stream_of(xl)),
            "sd_bound_sort_neuron_forward");
    return {lo, up};
}

// ---- mean shift: the gradient of the centring is the centring of the gradient ----------------------------------------
void shift_kernels(const Tensor& x, const Tensor& index, int64_t channels, const Tensor& mean, const OptTensor& running,
                   double momentum, const Tensor& y) {
    float* rp = running && running->defined() ? floats(*running, "running_mean") : nullptr;
    if (index.defined()) {
        const int G = (int)index.size(-2), cnt = (int)index.size(-1);
        if (G == 0) throw std::runtime_error("index names no groups: its size must be (sub-batches, groups, channels)");
        require(sd_mean_shift_index_forward(floats(x, "input"), ints(index, "index"), (int)x.size(0), G, cnt, (int)(channels / G),
                                            (int)x.size(2), floats(mean, "mean"), rp, (float)momentum, floats(y, "output"),
                                            stream_of(x)), "sd_mean_shift_index_forward");
    } else
        require(sd_mean_shift_forward(floats(x, "input"), (int)x.size(0), (int)x.size(1), (int)x.size(2), floats(mean, "mean"), rp,
                                      (float)momentum, floats(y, "output"), stream_of(x)), "sd_mean_shift_forward");
}

struct ShiftNode : Node {
    SavedVariable index;
    int64_t channels = 0;

    variable_list apply(variable_list&& grads) override {
        const Locked lock(mutex_);
        variable_list out(1);
        if (!task_should_compute_output(0)) return out;
        const Tensor idx = index.unpack();
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor g = incoming(*this, grads, 0);
        const c10::DeviceGuard guard(g.device());
        out[0] = at::empty(g.sizes(), g.options());
        shift_kernels(g, idx, channels, new_floats(g, {channels}), {}, 0.0, out[0]);
        return out;
    }
    void release_variables() override {
        const Locked lock(mutex_);
        index.reset_data();
    }
    std::string name() const override { return "ShiftNode"; }
};

std::pair<Tensor, Tensor> mean_shift_index(const Tensor& x_in, const OptTensor& index, int64_t channels, const OptTensor& running,
                                           double momentum) {
    reverse_mode_only("mean_shift", x_in);
    const bool grad = want_grad(x_in);
    Tensor y, mean, idx = index ? *index : Tensor();
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(x_in.device());
        const Tensor x = x_in.contiguous();
        y = at::empty(x.sizes(), x.options());
        mean = new_floats(x, {channels});
        shift_kernels(x, idx, channels, mean, running, momentum, y);
    }
    if (grad) {
        auto node = new_node<ShiftNode>();
        node->set_next_edges(collect_next_edges(x_in));
        node->channels = channels;
        if (idx.defined()) node->index = SavedVariable(idx, false);
        set_history(y, node);
    }
    return {y, mean};
}

std::pair<Tensor, Tensor> mean_shift(const Tensor& x, const OptTensor& running, double momentum) {
    return mean_shift_index(x, {}, x.size(1), running, momentum);
}

// (sub_batches, groups, count) ascending kept channels, drawn on the current stream of `device`
Tensor sample_index_lists(int64_t seed, int64_t sub_batches, int64_t groups, int64_t channels, int64_t count, at::Device device) {
    const c10::DeviceGuard guard(device);
    const Tensor out = at::empty({sub_batches, groups, count}, at::TensorOptions().dtype(at::kInt).device(device));
    if (count > 0)
        require(sd_sample_index_lists((uint32_t)seed, (int)sub_batches, (int)groups, (int)channels, (int)count, ints(out, "index"),
                                      stream_of(out)), "sd_sample_index_lists");
    return out;
}

// z + sign * vec[channel], outside any graph
Tensor channel_shift(const Tensor& z_in, const Tensor& vec_in, double sign) {
    reverse_mode_only("channel_shift", z_in, vec_in);
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(z_in.device());
    const Tensor z = z_in.contiguous(), vec = vec_in.contiguous();
    Tensor out = at::empty(z.sizes(), z.options());
    require(sd_channel_shift(floats(z, "input"), floats(vec, "shift"), (int)z.size(0), (int)z.size(1), (int)z.size(2), (float)sign,
                             floats(out, "output"), stream_of(z)), "sd_channel_shift");
    return out;
}

// ---- evaluation pass: a layer's values or bounds with sign * shift[channel] added, outside any graph ------------------
Tensor norm_dist_shifted(const Tensor& x, const Tensor& w, int64_t groups, const Tensor& shift_in, double sign) {
    reverse_mode_only("norm_dist", x, w, shift_in);
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x.device());
    Tensor y = new_out(x, w.size(0));
    const Tensor shift = shift_in.contiguous();
    const Dims d(x, groups, w.size(0));
    require(sd_inf_dist_forward_shifted(floats(x, "input"), floats(w, "weight"), d.B, d.CO, d.CI, d.G, d.HW, floats(y, "output"),
                                        floats(shift, "shift"), (float)sign, stream_of(x)), "sd_inf_dist_forward_shifted");
    return y;
}

Tensor sort_neuron_shifted(const Tensor& x, const Tensor& w, int64_t groups, double q, int truncate, const Tensor& shift_in, double sign) {
    reverse_mode_only("sort_neuron", x, w, shift_in);
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x.device());
    Tensor y = new_out(x, w.size(0));
    const Tensor shift = shift_in.contiguous();
    const Dims d(x, groups, w.size(0));
    require(sd_sort_neuron_forward_shifted(floats(x, "input"), floats(w, "weight"), d.B, d.CO, d.CI, d.G, d.HW, floats(y, "output"), (float)q,
                                           truncate, floats(shift, "shift"), (float)sign, stream_of(x)), "sd_sort_neuron_forward_shifted");
    return y;
}

std::pair<Tensor, Tensor> bound_inf_dist_shifted(const Tensor& xl, const Tensor& xu, const Tensor& w, int64_t groups, const Tensor& shift_in,
                                                 double sign) {
    reverse_mode_only("bound_inf_dist", xl, xu, w, shift_in);
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(xl.device());
    Tensor lo = new_out(xl, w.size(0)), up = new_out(xl, w.size(0));
    const Tensor shift = shift_in.contiguous();
    const Dims d(xl, groups, w.size(0));
    require(sd_bound_inf_dist_forward_shifted(floats(xl, "inputL"), floats(xu, "inputU"), floats(w, "weight"), d.B, d.CO, d.CI, d.G, d.HW,
                                              floats(lo, "outputL"), floats(up, "outputU"), floats(shift, "shift"), (float)sign, stream_of(xl)),
            "sd_bound_inf_dist_forward_shifted");
    return {lo, up};
}

std::pair<Tensor, Tensor> bound_sort_neuron_shifted(const Tensor& xl, const Tensor& xu, const Tensor& w, int64_t groups, double q, int truncate,
                                                    const Tensor& shift_in, double sign) {
    reverse_mode_only("bound_sort_neuron", xl, xu, w, shift_in);
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(xl.device());
    Tensor lo = new_out(xl, w.size(0)), up = new_out(xl, w.size(0));
    const Tensor shift = shift_in.contiguous();
    const Dims d(xl, groups, w.size(0));
    require(sd_bound_sort_neuron_forward_shifted(floats(xl, "inputL"), floats(xu, "inputU"), floats(w, "weight"), d.B, d.CO, d.CI, d.G, d.HW,
                                                 floats(lo, "outputL"), floats(up, "outputU"), (float)q, truncate, floats(shift, "shift"),
                                                 (float)sign, stream_of(xl)), "sd_bound_sort_neuron_forward_shifted");
    return {lo, up};
}

// values and bounds of a layer together
std::tuple<Tensor, Tensor, Tensor> sort_neuron_box_shifted(const Tensor& x, const Tensor& xl, const Tensor& xu, const Tensor& w, int64_t groups,
                                                           double q, int truncate, const Tensor& shift_in, double sign) {
    reverse_mode_only("sort_neuron", x, xl, xu, w, shift_in);
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x.device());
    Tensor y = new_out(x, w.size(0)), lo = new_out(xl, w.size(0)), up = new_out(xl, w.size(0));
    const Tensor shift = shift_in.contiguous();
    const Dims d(x, groups, w.size(0));
    require(sd_sort_neuron_box_forward(floats(x, "input"), floats(xl, "inputL"), floats(xu, "inputU"), floats(w, "weight"), d.B, d.CO, d.CI, d.G,
                                       d.HW, floats(y, "output"), floats(lo, "outputL"), floats(up, "outputU"), (float)q, truncate,
                                       floats(shift, "shift"), (float)sign, stream_of(x)), "sd_sort_neuron_box_forward");
    return {y, lo, up};
}

// ---- windows of a convolutional layer as columns; the gradient is the sum back into the image --------------------------
struct UnfoldNode : Node {   // saves sizes only, which nothing changes or frees
    int B, C, H, W, KH, KW, stride, pad, dil;

    variable_list apply(variable_list&& grads) override {
        at::AutoDispatchBelowADInplaceOrView below;
        variable_list out(1);
        if (!grads[0].defined() || !task_should_compute_output(0)) return out;
        const Tensor g = grads[0].contiguous();
        const c10::DeviceGuard guard(g.device());
        out[0] = new_floats(g, {B, C, H, W});
        require(sd_fold(floats(g, "grad_output"), B, C, H, W, KH, KW, stride, pad, dil, floats(out[0], "grad_input"), stream_of(g)),
                "sd_fold");
        return out;
    }
    std::string name() const override { return "UnfoldNode"; }
};

Tensor unfold(const Tensor& x_in, int kh, int kw, int dil, int pad, int stride) {
    reverse_mode_only("unfold", x_in);
    const bool grad = want_grad(x_in);
    const int B = (int)x_in.size(0), C = (int)x_in.size(1), H = (int)x_in.size(2), W = (int)x_in.size(3);
    Tensor y;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(x_in.device());
        const Tensor x = x_in.contiguous();
        if (stride < 1) throw std::runtime_error("unfold: stride=" + std::to_string(stride) + " must be positive");
        const int64_t oh = (H + 2 * pad - dil * (kh - 1) - 1) / stride + 1, ow = (W + 2 * pad - dil * (kw - 1) - 1) / stride + 1;
        y = new_floats(x, {B, (int64_t)C * kh * kw, oh > 0 && ow > 0 ? oh * ow : 1});   // a window that does not fit is refused below
        require(sd_unfold(floats(x, "input"), B, C, H, W, kh, kw, stride, pad, dil, floats(y, "output"), stream_of(x)), "sd_unfold");
    }
    if (grad) {
        auto node = new_node<UnfoldNode>();
        node->set_next_edges(collect_next_edges(x_in));
        node->B = B; node->C = C; node->H = H; node->W = W; node->KH = kh; node->KW = kw;
        node->stride = stride; node->pad = pad; node->dil = dil;
        set_history(y, node);
    }
    return y;
}

}  // namespace

PYBIND11_MODULE(_host, m) {
    m.doc() = "Autograd front-end of libsortdist.so";
    using released = py::call_guard<py::gil_scoped_release>;
    m.def("norm_dist", &norm_dist, released());
    m.def("norm_dist_dropout", &norm_dist_dropout, released());
    m.def("masked_inf_dist", &masked_inf_dist, released());
    m.def("sort_neuron", &sort_neuron, released());
    m.def("bound_sort_neuron", &bound_sort_neuron, released());
    m.def("bound_inf_dist", &bound_inf_dist, released());
    m.def("mean_shift", &mean_shift, released());
    m.def("mean_shift_index", &mean_shift_index, released());
    m.def("channel_shift", &channel_shift, released());
    m.def("sample_index_lists", &sample_index_lists, released());
    m.def("norm_dist_shifted", &norm_dist_shifted, released());
    m.def("sort_neuron_shifted", &sort_neuron_shifted, released());
    m.def("bound_inf_dist_shifted", &bound_inf_dist_shifted, released());
    m.def("bound_sort_neuron_shifted", &bound_sort_neuron_shifted, released());
    m.def("sort_neuron_box_shifted", &sort_neuron_box_shifted, released());
    m.def("unfold", &unfold, released());
}
