// The layer as one autograd node in C++: allocation of a call's buffers, the argument block of mole_layer_fwd /
// mole_layer_bwd, and the node autograd records.  Built into mole_torch.so beside libmole_hip.so, which it calls through the
// C ABI; there is no GPU code here.
//
// Why it exists: with the same two calls made from Python a training step of a small layer spent 250 us on the host, 50 of
// them in the library.  The rest was an autograd.Function and its context in Python, tensor allocations through the
// interpreter and argument blocks through ctypes, half of it on autograd's own thread.
#include <torch/extension.h>
#include <ATen/TracerMode.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <atomic>
#include <limits>

#include "mole_hip.h"

namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void check(int rc, const char *what) {
    TORCH_CHECK(rc == 0, what, " failed (code ", rc, "): ", mole_last_error_string());
}
int64_t up256(int64_t v) { return (v + 255) & ~(int64_t)255; }

// Passes a layer has been through backward, shared with the Python side (MOLECore.step)
struct Counter {
    std::atomic<int64_t> value;
    explicit Counter(int64_t v) : value(v) {}
};

// Sizes of one layer call, shared by every call of the same shape: the kept rows' bound, and where each intermediate lies
// in the buffers of a call - route (the routing, which the layer also keeps as last_route), act (xd, a, out and h, kept for
// the backward, as the scores are) and grad (the backward's temporaries and scratch).  The forward's scratch is no part of what
// is kept: it has a buffer of its own, or in a pass without autograd, which keeps nothing and stores no h, the place of h, with
// the scores behind it (every allocation is a microsecond of the host's).  Holds no device memory.
struct Plan {
    mole_layer head{};
    at::ScalarType dtype;
    int gelu_bwd;
    enum { GATES, IDX, LOC, ROW, COUNTS, KEPT, OFFSETS, CAPACITY, N_ROUTE };
    enum { XD, A, OUT, H, N_ACT };
    enum { D_O, T, GXD, DLOGITS, GRAD_WS, N_GRAD };
    int64_t route_off[N_ROUTE], act_off[N_ACT], grad_off[N_GRAD];
    int64_t route_bytes, act_bytes, grad_bytes, ws_fwd, ws_bwd;

    template <int N> static int64_t carve(const int64_t (&bytes)[N], int64_t (&off)[N]) {
        int64_t at = 0;
        for (int i = 0; i < N; ++i) {
            off[i] = at;
            at += up256(bytes[i]);
        }
        return at;
    }

    Plan(int dtype_code, int64_t S, int64_t M, int64_t E, int64_t k, int64_t F, double cf, int layout, bool normalize, int gelu)
        : dtype(dtype_code == MOLE_BF16 ? at::kBFloat16 : at::kFloat), gelu_bwd(gelu) {
        TORCH_CHECK(S >= 1 && M >= 1 && E >= 1 && k >= 1 && F >= 1 && S * k < (1ll << 31), "bad layer sizes");
        const int64_t es = dtype_code == MOLE_BF16 ? 2 : 4;
        int64_t rows = S * k;
        if (cf > 0) {
            // the reference's integer: k * int(cf * ceil(S / E)), the product in double precision.  A factor whose product
            // no int64 holds would come out of the conversion negative, and the buffers a row long: 2^31 per choice is
            // more than the S k rows there are (and more than the padded layout takes)
            TORCH_CHECK(cf <= std::numeric_limits<double>::max(), "the capacity factor must be finite");
            const int64_t cap = k * (int64_t)std::min(cf * (double)((S + E - 1) / E), 2147483648.0);
            rows = layout == MOLE_LAYOUT_PADDED ? E * cap : std::min(rows, E * cap);
        }
        rows = std::max<int64_t>(rows, 1);
        TORCH_CHECK(rows < (1ll << 31), "too many rows");
        head.dtype = dtype_code; head.S = (int)S; head.M = (int)M; head.E = (int)E; head.k = (int)k; head.F = (int)F;
        head.rows = (int)rows; head.layout = layout; head.normalize_gate = normalize; head.capacity_factor = cf;
        ws_fwd = (int64_t)mole_layer_workspace_bytes(&head, 0);
        ws_bwd = (int64_t)mole_layer_workspace_bytes(&head, 1);
        route_bytes = carve({k * S * 4, k * S * 4, k * S * 4, k * S * 4, k * E * 4, E * 4, (E + 1) * 4, 4}, route_off);
        act_bytes = carve({rows * M * es, rows * F * es, rows * M * es, rows * F * es}, act_off);
        grad_bytes = carve({rows * M * es, rows * F * es, rows * M * es, S * E * 4, ws_bwd}, grad_off);
    }
    std::vector<int64_t> route_offsets() const { return {route_off, route_off + N_ROUTE}; }
};

// What a backward pass needs beside the saved tensors: kept by the node until it is released.
struct Call : torch::CustomClassHolder {
    std::shared_ptr<Plan> plan;
    std::shared_ptr<Counter> counter;
    std::optional<Tensor> bias;
    std::vector<Tensor> weights, grads;      // w1, b1, w2, b2 of all experts and their gradient buffers
    bool accumulate = false;
    std::vector<int64_t> dummy_sizes;        // the marker parameter: its gradient is a tensor of zeros, never left out
    at::TensorOptions dummy_options;
    Tensor route;                            // the routing: a result for the caller as well
};

void check_tensor(const Tensor &t, const char *name) {
    TORCH_CHECK(t.is_cuda() && t.is_contiguous(), "mole_amd: ", name, " must be a contiguous tensor on the GPU (there is no CPU path)");
}

void check_input(const Plan &p, const Tensor &x, const Tensor &wg) {
    check_tensor(x, "x");
    check_tensor(wg, "the gate's weight");
    TORCH_CHECK(x.dim() == 2 && x.size(0) == p.head.S && x.size(1) == p.head.M && x.scalar_type() == p.dtype &&
                    wg.dim() == 2 && wg.size(0) == p.head.E && wg.size(1) == p.head.M && wg.scalar_type() == at::kFloat,
                "mole_amd: the layer's input or gate does not have the planned shape or type");
}
void check_saved(const Tensor &t, at::ScalarType dtype, int64_t numel, const char *name) {
    check_tensor(t, name);
    TORCH_CHECK(t.scalar_type() == dtype && t.numel() == numel, "mole_amd: ", name, " came back in another shape or type than they were saved in");
}

mole_layer arguments(const Call &c, const Tensor &x, const Tensor &wg, void *scores, char *act, char *ws, int64_t ws_bytes) {
    const Plan &p = *c.plan;
    char *route = (char *)c.route.data_ptr();
    mole_layer L = p.head;
    L.x = x.data_ptr();
    L.wg = wg.data_ptr<float>();
    L.logit_bias = c.bias.has_value() ? c.bias->data_ptr<float>() : nullptr;
    L.w1 = c.weights[0].data_ptr(); L.b1 = c.weights[1].data_ptr(); L.w2 = c.weights[2].data_ptr(); L.b2 = c.weights[3].data_ptr();
    L.scores = (float *)scores;
    L.gates = (float *)(route + p.route_off[Plan::GATES]);
    L.idx = (int32_t *)(route + p.route_off[Plan::IDX]);
    L.loc = (int32_t *)(route + p.route_off[Plan::LOC]);
    L.row = (int32_t *)(route + p.route_off[Plan::ROW]);
    L.counts = (int32_t *)(route + p.route_off[Plan::COUNTS]);
    L.kept_rows = (int32_t *)(route + p.route_off[Plan::KEPT]);
    L.offsets = (int32_t *)(route + p.route_off[Plan::OFFSETS]);
    L.capacity = (int32_t *)(route + p.route_off[Plan::CAPACITY]);
    L.xd = act + p.act_off[Plan::XD]; L.h = act + p.act_off[Plan::H]; L.a = act + p.act_off[Plan::A]; L.out = act + p.act_off[Plan::OUT];
    L.workspace = ws;
    L.workspace_bytes = (size_t)ws_bytes;
    return L;
}

void *current_stream(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// y, the scores and intermediates the backward reads (recorded passes), and the loss term, a tensor of its own: callers keep it, and part of a
// larger buffer would keep all of that.  c.route is set.
struct Outputs {
    Tensor y, scores, act, l_aux;
};
Outputs run_forward(Call &c, const Tensor &x, const Tensor &wg, bool forward_only) {
    const Plan &p = *c.plan;
    check_input(p, x, wg);
    const auto bytes = x.options().dtype(at::kByte);
    c.route = at::empty({p.route_bytes}, bytes);
    // (act in the layer's own type: hooks on saved tensors may convert it and back)
    const int64_t es = x.element_size();
    const int64_t only_scores = p.act_off[Plan::H] + up256(p.ws_fwd), only_bytes = only_scores + (int64_t)p.head.S * p.head.E * 4;
    Tensor act = at::empty({(forward_only ? only_bytes : p.act_bytes) / es}, x.options()), y = at::empty({p.head.S, p.head.M}, x.options());
    const auto f32 = x.options().dtype(at::kFloat);
    Tensor scores, l_aux = at::empty({}, f32), ws;
    if (!forward_only) {
        scores = at::empty({p.head.S, p.head.E}, f32);
        ws = at::empty({p.ws_fwd}, bytes);       // (released on return, for later work of this stream)
    }
    char *a = (char *)act.data_ptr();
    mole_layer L = arguments(c, x, wg, forward_only ? a + only_scores : scores.data_ptr(), a,
                             forward_only ? a + p.act_off[Plan::H] : (char *)ws.data_ptr(), p.ws_fwd);
    L.l_aux = l_aux.data_ptr<float>();
    if (forward_only) {
        L.forward_only = 2;
        L.h = nullptr;
    }
    check(mole_layer_fwd(&L, y.data_ptr(), current_stream(x)), "mole_layer_fwd");
    return {y, scores, act, l_aux};
}

struct LayerFn : torch::autograd::Function<LayerFn> {
    // dummy: an empty parameter that makes autograd record the node although x need not require a gradient
    static variable_list forward(AutogradContext *ctx, const Tensor &x, const Tensor &wg, const Tensor &dummy, c10::intrusive_ptr<Call> c) {
        c->dummy_sizes = dummy.sizes().vec();
        c->dummy_options = dummy.options();
        ctx->set_materialize_grads(false);
        auto [y, scores, act, l_aux] = run_forward(*c, x, wg, false);
        ctx->save_for_backward({x, wg, scores, act});
        ctx->saved_data["call"] = c10::IValue::make_capsule(std::move(c));
        return {y, l_aux};
    }

    static variable_list backward(AutogradContext *ctx, variable_list g) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &x = saved[0], &scores = saved[2], &act = saved[3], wg = saved[1].to(at::kFloat).contiguous();
        auto c = c10::static_intrusive_pointer_cast<Call>(ctx->saved_data["call"].toCapsule());
        const Plan &p = *c->plan;
        // (what hooks on saved tensors hand back need not be what was saved)
        check_input(p, x, wg);
        check_saved(scores, at::kFloat, (int64_t)p.head.S * p.head.E, "the scores");
        check_saved(act, p.dtype, p.act_bytes / x.element_size(), "the intermediates");
        Tensor dy = g[0].defined() ? g[0].contiguous() : at::zeros_like(x);      // (undefined: only l_aux was used)
        Tensor d_aux = g[1].defined() ? g[1].to(at::kFloat).contiguous() : Tensor();
        TORCH_CHECK(dy.scalar_type() == p.dtype && dy.numel() == x.numel(), "mole_amd: the output's gradient has another shape or type");
        Tensor tmp = at::empty({p.grad_bytes}, x.options().dtype(at::kByte));
        Tensor dx = at::empty({p.head.S, p.head.M}, x.options()), dwg = at::empty({p.head.E, p.head.M}, wg.options());
        char *t = (char *)tmp.data_ptr();
        mole_layer L = arguments(*c, x, wg, scores.data_ptr(), (char *)act.data_ptr(), t + p.grad_off[Plan::GRAD_WS], p.ws_bwd);
        mole_layer_grads G{};
        G.accumulate = c->accumulate;
        G.gelu_bwd = p.gelu_bwd;
        G.dy = dy.data_ptr();
        G.d_l_aux = d_aux.defined() ? d_aux.data_ptr<float>() : nullptr;
        G.dlogits = (float *)(t + p.grad_off[Plan::DLOGITS]);
        G.d_o = t + p.grad_off[Plan::D_O]; G.t = t + p.grad_off[Plan::T]; G.gxd = t + p.grad_off[Plan::GXD];
        G.g_w1 = c->grads[0].data_ptr(); G.g_b1 = c->grads[1].data_ptr(); G.g_w2 = c->grads[2].data_ptr(); G.g_b2 = c->grads[3].data_ptr();
        G.dx = dx.data_ptr();
        G.dwg = dwg.data_ptr<float>();
        check(mole_layer_bwd(&L, &G, current_stream(x)), "mole_layer_bwd");
        c->counter->value += 1;
        return {dx, dwg, at::zeros(c->dummy_sizes, c->dummy_options), Tensor()};
    }
};

// (y, l_aux, route, l_aux without its graph)
std::tuple<Tensor, Tensor, Tensor, Tensor> layer(const Tensor &x, const Tensor &wg, const Tensor &dummy, std::optional<Tensor> bias,
                                                 std::vector<Tensor> weights, std::vector<Tensor> grads, std::shared_ptr<Plan> plan,
                                                 bool accumulate, std::shared_ptr<Counter> counter) {
    TORCH_CHECK(weights.size() == 4 && grads.size() == 4, "mole_amd: four parameter and four gradient tensors");
    // (a trace would record the allocations and none of the kernels: its replays would return memory nothing has written)
    TORCH_CHECK(!at::tracer::impl::is_dispatch_enabled(), "mole_amd: the layer cannot be traced by torch.jit.trace");
    auto c = c10::make_intrusive<Call>();
    c->plan = std::move(plan);
    c->counter = std::move(counter);
    c->bias = std::move(bias);
    c->weights = std::move(weights);
    c->grads = std::move(grads);
    c->accumulate = accumulate;
    // (no_grad leaves forward-mode derivatives on: an input that carries a tangent goes through the node, which refuses it)
    if (!at::GradMode::is_enabled() && !x._fw_grad(0).defined() && !wg._fw_grad(0).defined()) {
        auto r = run_forward(*c, x, wg, true);
        return {r.y, r.l_aux, c->route, r.l_aux};
    }
    auto out = LayerFn::apply(x, wg, dummy, c);
    return {out[0], out[1], c->route, out[1].detach()};
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    py::class_<Counter, std::shared_ptr<Counter>>(m, "Counter")
        .def(py::init<int64_t>())
        .def_property("value", [](const Counter &c) { return c.value.load(); }, [](Counter &c, int64_t v) { c.value = v; });
    py::class_<Plan, std::shared_ptr<Plan>>(m, "Plan")
        .def(py::init<int, int64_t, int64_t, int64_t, int64_t, int64_t, double, int, bool, int>())
        .def("route_offsets", &Plan::route_offsets)
        .def_property_readonly("rows", [](const Plan &p) { return p.head.rows; });
    m.def("layer", &layer, py::call_guard<py::gil_scoped_release>());
}
