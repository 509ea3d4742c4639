// The host path of the attention module, the transformer block and the stage merge: what the Python modules of this
// package call for tensors on the GPU.  One autograd node per module call; allocation of results and scratch by PyTorch's
// caching allocator, everything else launches of libsswin3d.so on the current stream.
//
// A module call is a dozen launches of a few microseconds each on the small stages, so the host decides their speed: from
// Python (one autograd node, ctypes call and context manager per operator) a block's forward took about 250 us of host time,
// its launches 80.
#include <torch/extension.h>

#include <ATen/Context.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <hip/hip_runtime.h>

#include <array>
#include <atomic>
#include <mutex>
#include <optional>
#include <string>
#include <vector>

#include "../../include/sswin3d.h"

namespace {

using at::Tensor;
using c10::ScalarType;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

// ------------------------------------------------------------------------------------------
// launches
// ------------------------------------------------------------------------------------------
void* current_stream(const Tensor& t) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream(); }

int code_of(ScalarType t) {
    switch (t) {
        case at::kFloat: return SSWIN_F32;
        case at::kHalf: return SSWIN_F16;
        case at::kBFloat16: return SSWIN_BF16;
        default: TORCH_CHECK(false, "unsupported value dtype ", t);
    }
}

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* f32(const Tensor& t) { return t.defined() ? t.data_ptr<float>() : nullptr; }
int32_t* i32(const Tensor& t) { return t.defined() ? t.data_ptr<int32_t>() : nullptr; }

// A benchmark's recorder: called with (name, before) around every timed launch, with the GIL held.
PyObject* g_recorder = nullptr;
struct Timed {
    const char* name;
    explicit Timed(const char* n) : name(g_recorder ? n : nullptr) { if (name) tell(true); }
    ~Timed() { if (name) tell(false); }
    void tell(bool before) const {
        py::gil_scoped_acquire gil;
        if (g_recorder) py::reinterpret_borrow<py::object>(g_recorder)(name, before);
    }
};
#define RUN_NAMED(name, call)                                 \
    do {                                                      \
        int rc_;                                              \
        {                                                     \
            Timed timed_(name);                               \
            rc_ = call;                                       \
        }                                                     \
        TORCH_CHECK(rc_ == 0, sswin_last_error());            \
    } while (0)
#define RUN(call) RUN_NAMED(#call, call)

Tensor bytes(size_t n, const Tensor& like) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte)); }

// ------------------------------------------------------------------------------------------
// token plans
// ------------------------------------------------------------------------------------------
std::mutex g_pool_mutex;
std::vector<Tensor> g_pinned;            // pinned totals of finished plans, reused: allocating one costs tens of microseconds

Tensor take_pinned() {
    {
        std::lock_guard<std::mutex> lock(g_pool_mutex);
        if (!g_pinned.empty()) {
            Tensor t = std::move(g_pinned.back());
            g_pinned.pop_back();
            return t;
        }
    }
    return at::zeros({9}, at::TensorOptions().dtype(at::kLong).pinned_memory(true));
}
void give_pinned(Tensor&& t) {
    std::lock_guard<std::mutex> lock(g_pool_mutex);
    if (g_pinned.size() < 64) g_pinned.push_back(std::move(t));
}

struct SharedEvent {
    hipEvent_t event = nullptr;
    SharedEvent() { TORCH_CHECK(hipEventCreateWithFlags(&event, hipEventDisableTiming) == hipSuccess, "hipEventCreate failed"); }
    ~SharedEvent() { if (event) (void)hipEventDestroy(event); }
};

struct Plan : torch::CustomClassHolder {
    Tensor indices, tokens, plan, tasks, ws, totals;
    int64_t N = 0, n = 0, B = 0, g_cap = 0;
    int H = 0;
    bool order_only = false;
    std::shared_ptr<SharedEvent> event;
    // allocated; its kernels are in the stream; its totals are decoded; its totals failed their check, which every later use
    // reports again (a plan stays in its view's cache, and the tables of a failed one are not filled)
    enum State { FRESH, QUEUED, DONE, FAILED };
    std::atomic<int> state{FRESH};
    std::mutex mutex;                        // of the step from QUEUED to DONE or FAILED
    std::string failure;
    int64_t G = 0, windows = 0, A = 0, c_max = 0, buckets[4] = {0, 0, 0, 0}, oversize = 0;

    Plan(const Tensor& ind, int64_t batch, int64_t positions, int64_t heads, bool with_tasks, bool order) {
        TORCH_CHECK(ind.is_cuda(), "TokenPlan runs on the GPU only; there is no CPU fallback");
        TORCH_CHECK(ind.scalar_type() == at::kInt && ind.dim() == 2 && ind.size(1) == 2, "TokenPlan: indices must be int32 [N, 2]");
        c10::hip::HIPGuardMasqueradingAsCUDA guard(ind.device());
        indices = ind.contiguous();
        N = indices.size(0), n = positions, B = batch, H = (int)heads, order_only = order;
        g_cap = std::max<int64_t>(1, std::min(N, B) * H);
        const auto opt = indices.options();
        // order_only: the plan of a stride-2 merge, whose consumers read the voxel of every rank and nothing else
        tokens = at::empty({(order ? 1 : 5) * std::max<int64_t>(N, 1)}, opt);
        plan = at::empty({5 * g_cap}, opt);
        // group descriptors of the window-resident kernels and behind them the token records
        if (with_tasks) tasks = at::empty({(int64_t)sswin_token_plan_task_ints(N, g_cap, H)}, opt);
        ws = at::empty({(int64_t)sswin_token_plan_workspace_bytes(N, (int)B, (int)n)}, opt.dtype(at::kByte));
        totals = take_pinned();
    }
    ~Plan() override {
        if (event) (void)hipEventSynchronize(event->event);              // the kernels still write into totals
    }

    // Any number of threads may ask: the first one waits and decodes, the others wait for it.  The lock is taken without the GIL
    // only, so that a thread that holds the lock can never wait for one that holds the GIL.
    void finish() {
        if (state.load(std::memory_order_acquire) != DONE) {
            if (PyGILState_Check()) {
                py::gil_scoped_release nogil;
                complete();
            } else {
                complete();
            }
        }
    }
    void complete() {
        std::lock_guard<std::mutex> lock(mutex);
        TORCH_CHECK(state != FRESH, "token plan: its kernels were not launched");
        if (state == QUEUED) {
            TORCH_CHECK(hipEventSynchronize(event->event) == hipSuccess, "token plan: the stream failed");
            decode();
        }
        TORCH_CHECK(state == DONE, failure);
    }
    void decode() {
        int64_t* v = totals.data_ptr<int64_t>();
        const int rc = N > 0 ? sswin_token_plan_totals(v, H, g_cap) : 0;
        if (rc == 0) {
            G = v[0], windows = v[1], A = v[2], c_max = v[3], oversize = v[8];
            for (int b = 0; b < 4; ++b) buckets[b] = v[4 + b];
        } else {
            failure = sswin_last_error();
        }
        event.reset();
        give_pinned(std::move(totals));
        ws = Tensor();
        indices = Tensor();
        state.store(rc == 0 ? DONE : FAILED, std::memory_order_release);
    }
    const Plan& decoded() const {
        const int now = state.load(std::memory_order_acquire);
        TORCH_CHECK(now == DONE, now == FAILED ? failure : "token plan: the totals are there after finish()");
        return *this;
    }
};
using PlanPtr = c10::intrusive_ptr<Plan>;

// Launch allocated plans, four per library call; they share one event.  Where a call fails, the plans of the calls before it
// are in the stream and can be used, and no plan gives up the memory its kernels may still write before the event.
void enqueue_plans(const std::vector<PlanPtr>& plans) {
    if (plans.empty()) return;
    const Tensor& like = plans[0]->indices;
    for (const PlanPtr& p : plans) {
        TORCH_CHECK(p->state == Plan::FRESH, "TokenPlan: launched already");
        TORCH_CHECK(p->indices.device() == like.device(), "TokenPlan.batch: all index sets must live on one device");
    }
    c10::hip::HIPGuardMasqueradingAsCUDA guard(like.device());
    void* s = current_stream(like);
    auto event = std::make_shared<SharedEvent>();
    auto record = [&](size_t queued, size_t failed, const char* why) {       // [0, queued) launched, [queued, failed) perhaps in part
        const bool ok = hipEventRecord(event->event, static_cast<hipStream_t>(s)) == hipSuccess;
        if (!ok) (void)hipStreamSynchronize(static_cast<hipStream_t>(s));
        for (size_t i = 0; i < failed; ++i) {
            Plan& p = *plans[i];
            if (ok) p.event = event;
            if (!ok || i >= queued) p.failure = ok ? why : "hipEventRecord failed";
            p.state = ok && i < queued ? Plan::QUEUED : Plan::FAILED;
        }
        TORCH_CHECK(ok || queued < failed, "hipEventRecord failed");
    };
    for (size_t k = 0; k < plans.size(); k += 4) {
        sswin_token_plan_desc d[4];
        const int m = (int)std::min<size_t>(4, plans.size() - k);
        for (int i = 0; i < m; ++i) {
            Plan& p = *plans[k + i];
            d[i] = sswin_token_plan_desc{};
            d[i].indices = i32(p.indices), d[i].N = p.N, d[i].B = (int32_t)p.B, d[i].n = (int32_t)p.n, d[i].H = p.H;
            d[i].flags = (p.order_only ? SSWIN_PLAN_ORDER_ONLY : 0) | SSWIN_PLAN_TOTALS_DIRECT;
            d[i].tokens = i32(p.tokens), d[i].plan = i32(p.plan), d[i].g_cap = p.g_cap, d[i].tasks = i32(p.tasks);
            d[i].totals_out = p.totals.data_ptr<int64_t>(), d[i].ws = p.ws.data_ptr(), d[i].ws_bytes = (size_t)p.ws.numel();
        }
        try {
            RUN(sswin_token_plan_batch(d, m, s));
        } catch (...) {
            record(k, k + m, "token plan: its launch failed");
            throw;
        }
    }
    record(plans.size(), plans.size(), "");
}

// (batch, d, h, w) -> (window slot, position) of the padded grid rolled by -shift
Tensor window_indices(const Tensor& ind, int64_t batch, const std::vector<int64_t>& dims, const std::vector<int64_t>& window,
                      const std::vector<int64_t>& shift) {
    c10::hip::HIPGuardMasqueradingAsCUDA guard(ind.device());
    const Tensor x = ind.contiguous();
    Tensor out = at::empty({x.size(0), 2}, x.options());
    int32_t d[3], w[3], sh[3];
    for (int i = 0; i < 3; ++i) d[i] = (int32_t)dims.at(i), w[i] = (int32_t)window.at(i), sh[i] = (int32_t)shift.at(i);
    RUN(sswin_window_indices(i32(x), x.size(0), (int)batch, d, w, sh, i32(out), current_stream(x)));
    return out;
}

// ------------------------------------------------------------------------------------------
// dense layers
// ------------------------------------------------------------------------------------------
// rocBLAS handles the tall shapes that are left to a library better than hipBLASLt's heuristics
struct RocBlas {
    at::BlasBackend before = at::globalContext().blasPreferredBackend();
    RocBlas() { if (before != at::BlasBackend::Cublas) at::globalContext().setBlasPreferredBackend(at::BlasBackend::Cublas); }
    ~RocBlas() { if (before != at::BlasBackend::Cublas) at::globalContext().setBlasPreferredBackend(before); }
};

bool aligned(const Tensor& t) { return !t.defined() || (uintptr_t)t.data_ptr() % 16 == 0; }
Tensor ready(const Tensor& t) {
    if (!t.defined()) return t;
    Tensor c = t.contiguous();
    return aligned(c) ? c : c.clone();
}

bool dense_takes(const Tensor& x, const Tensor& w, int64_t P, int64_t K) {
    return sswin_dense_supported(code_of(x.scalar_type()), (int)P, (int)K) && w.scalar_type() == x.scalar_type();
}
// 16-bit layers with long reductions over many rows: the library's tiles are ahead (1364 rows 768 -> 2304: 11 us against 18,
// 8119 rows 768 -> 3072: 47 and 57; 8119 rows 384 -> 1152: 23 and 19)
bool library_ahead(const Tensor& x, int64_t P, int64_t K) {
    return x.scalar_type() != at::kFloat && K >= 768 && P >= 192 && x.size(0) >= 1024;
}

// parameters in the type of the products; fp32 ones under mixed precision are converted together by one launch
template <size_t COUNT> std::array<Tensor, COUNT> in_type(const std::array<Tensor, COUNT>& params, ScalarType type) {
    static_assert(COUNT <= SSWIN_CAST_PARTS, "parts of one launch");
    std::array<Tensor, COUNT> out;
    const void* src[COUNT];
    int64_t sizes[COUNT], total = 0;
    int which[COUNT], n = 0;
    for (size_t i = 0; i < COUNT; ++i) {
        const Tensor& p = params[i];
        if (!p.defined()) continue;
        if (p.scalar_type() == type || p.scalar_type() != at::kFloat || p.numel() % 8 != 0 || p.numel() == 0) {
            out[i] = ready(p.to(type));
            continue;
        }
        out[i] = ready(p);
        src[n] = out[i].data_ptr();
        sizes[n] = p.numel();
        total += sizes[n];
        which[n++] = (int)i;
    }
    if (n == 0) return out;
    const Tensor& first = out[which[0]];
    const Tensor all = at::empty({total}, first.options().dtype(type));
    RUN(sswin_cast_parts(code_of(type), src, sizes, n, ptr(all), current_stream(first)));
    int64_t at = 0;
    for (int i = 0; i < n; ++i) {
        Tensor& t = out[which[i]];
        t = all.narrow(0, at, sizes[i]).view(t.sizes());
        at += sizes[i];
    }
    return out;
}

// the kernels take pointers: a parameter or plan left on another device has to stop here
void same_device(const Tensor& x, std::initializer_list<const Tensor*> others) {
    for (const Tensor* t : others)
        TORCH_CHECK(!t->defined() || t->device() == x.device(), "all tensors of a call have to be on the same device: found ", x.device(), " and ", t->device());
}

// x [N, K], w [P, K] -> last step of x w^T + b
Tensor dense(const Tensor& x, const Tensor& w_in, const Tensor& b_in, int epilogue = SSWIN_DENSE_PLAIN, const Tensor& extra = Tensor(),
             Tensor* slope = nullptr, std::optional<ScalarType> out_type = std::nullopt) {
    TORCH_CHECK(w_in.dim() == 2 && w_in.size(1) == x.size(1) && (!b_in.defined() || (b_in.dim() == 1 && b_in.size(0) == w_in.size(0))),
                "a dense layer of weight ", w_in.sizes(), " on rows of ", x.size(1), " values");
    const int64_t N = x.size(0), K = x.size(1), P = w_in.size(0);
    TORCH_CHECK(epilogue != SSWIN_DENSE_RESIDUAL || (extra.dim() == 2 && extra.size(0) == N && extra.size(1) == P), "a dense layer of ", P,
                " columns added to rows of ", extra.sizes());
    const ScalarType out = out_type.value_or(x.scalar_type());
    const Tensor w = ready(w_in), b = ready(b_in);
    if (dense_takes(x, w, P, K) && (!b.defined() || b.scalar_type() == x.scalar_type()) && !(epilogue == SSWIN_DENSE_PLAIN && library_ahead(x, P, K))) {
        Tensor y = at::empty({N, P}, x.options().dtype(out));
        if (slope) *slope = at::empty({N, P}, x.options().dtype(out));
        const size_t nb = sswin_dense_forward_workspace_bytes(code_of(x.scalar_type()), N, (int)K, (int)P);
        const Tensor ws = nb ? bytes(nb, x) : Tensor();
        RUN(sswin_dense_forward(code_of(x.scalar_type()), code_of(out), 0, epilogue, ptr(x), N, (int)K, ptr(w), ptr(b), (int)P,
                                ptr(extra), ptr(y), slope ? ptr(*slope) : nullptr, ptr(ws), nb, current_stream(x)));
        return y;
    }
    RocBlas backend;
    const Tensor wt = w.to(x.scalar_type());
    Tensor y = at::linear(x, wt, b.defined() ? OptTensor(b.to(x.scalar_type())) : std::nullopt);
    if (epilogue == SSWIN_DENSE_GELU) {
        if (slope) *slope = at::gelu_backward(at::ones_like(y), y);
        y = at::gelu(y);
    } else if (epilogue == SSWIN_DENSE_RESIDUAL) {
        y = at::add(extra, y);
    }
    return y.to(out);
}

// dy [N, P], w [P, K] -> (dy w) * extra
Tensor dense_dx(const Tensor& dy, const Tensor& w_in, int epilogue = SSWIN_DENSE_PLAIN, const Tensor& extra = Tensor()) {
    const Tensor w = ready(w_in);
    const int64_t N = dy.size(0), P = dy.size(1), K = w.size(1);
    if (dense_takes(dy, w, K, P) && !(epilogue == SSWIN_DENSE_PLAIN && library_ahead(dy, K, P))) {
        Tensor dx = at::empty({N, K}, dy.options());
        const size_t nb = sswin_dense_forward_workspace_bytes(code_of(dy.scalar_type()), N, (int)P, (int)K);
        const Tensor ws = nb ? bytes(nb, dy) : Tensor();
        RUN(sswin_dense_forward(code_of(dy.scalar_type()), code_of(dy.scalar_type()), 1, epilogue, ptr(dy), N, (int)P, ptr(w), nullptr,
                                (int)K, ptr(extra), ptr(dx), nullptr, ptr(ws), nb, current_stream(dy)));
        return dx;
    }
    RocBlas backend;
    Tensor dx = at::mm(dy, w.to(dy.scalar_type()));
    return epilogue == SSWIN_DENSE_SCALE ? dx.mul_(extra) : dx;
}

// dy [N, P], x [N, K] -> dy^T x and the column sums of dy, in `out`
std::pair<Tensor, Tensor> dense_dw(const Tensor& dy, const Tensor& x, bool want_bias, ScalarType out) {
    const int64_t N = dy.size(0), P = dy.size(1), K = x.size(1);
    const auto opt = x.options().dtype(out);
    void* s = current_stream(x);
    if (N > 0 && out == at::kFloat && x.scalar_type() == at::kFloat && K <= 96 && N > 1024) {
        const size_t nb = sswin_tall_linear_weight_grad_workspace_bytes(N, (int)P, (int)K);
        if (nb) {                                                        // up to 96 input channels: one pass over both operands
            Tensor dw = at::empty({P, K}, opt), db = want_bias ? at::empty({P}, opt) : Tensor(), ws = bytes(nb, x);
            RUN(sswin_tall_linear_weight_grad(f32(dy), f32(x), N, (int)P, (int)K, f32(dw), f32(db), ptr(ws), nb, s));
            return {dw, db};
        }
    }
    if (N > 0 && sswin_dense_supported(code_of(x.scalar_type()), (int)P, (int)K)) {
        Tensor dw = at::empty({P, K}, opt), db = want_bias ? at::empty({P}, opt) : Tensor();
        const size_t nb = sswin_dense_weight_grad_workspace_bytes(code_of(x.scalar_type()), N, (int)P, (int)K);
        Tensor ws = bytes(nb, x);
        RUN(sswin_dense_weight_grad(code_of(x.scalar_type()), code_of(out), ptr(dy), ptr(x), N, (int)P, (int)K, ptr(dw), ptr(db), ptr(ws), nb, s));
        return {dw, db};
    }
    RocBlas backend;
    return {at::mm(dy.t(), x).to(out), want_bias ? dy.sum(0).to(out) : Tensor()};
}

struct DenseGrads {
    Tensor dx, dw, db;
};
// all gradients of a layer: dy [N, P], x [N, K], w [P, K]; which of them are asked for
DenseGrads dense_backward(const Tensor& dy, const Tensor& x, const Tensor& w_in, bool want_dx, bool want_weight, bool want_bias, ScalarType out,
                          int epilogue = SSWIN_DENSE_PLAIN, const Tensor& extra = Tensor()) {
    DenseGrads g;
    const int64_t N = x.size(0), P = dy.size(1), K = x.size(1);
    const int dt = code_of(x.scalar_type());
    if (want_dx && (want_weight || want_bias) && dy.scalar_type() == x.scalar_type() && w_in.scalar_type() == x.scalar_type() &&
        sswin_dense_backward_small_supported(dt, N, (int)P, (int)K) && !(epilogue == SSWIN_DENSE_PLAIN && library_ahead(dy, K, P))) {
        const Tensor w = ready(w_in);
        const auto opt = x.options().dtype(out);
        g.dx = at::empty({N, K}, dy.options());
        g.dw = at::empty({P, K}, opt);
        if (want_bias) g.db = at::empty({P}, opt);
        RUN(sswin_dense_backward_small(dt, code_of(out), epilogue, ptr(dy), ptr(x), ptr(w), N, (int)P, (int)K, ptr(extra), ptr(g.dx), ptr(g.dw), ptr(g.db),
                                       current_stream(x)));
        return g;
    }
    if (want_weight || want_bias) std::tie(g.dw, g.db) = dense_dw(dy, x, want_bias, out);
    if (want_dx) g.dx = dense_dx(dy, w_in, epilogue, extra);
    return g;
}

// both layers of the feed-forward part as one launch, where that is ahead: x [N, D], w1 [hidden, D], w2 [D, hidden]
bool mlp_takes(const Tensor& x, const Tensor& w1, const Tensor& w2) {
    return w1.dim() == 2 && w2.dim() == 2 && w1.size(1) == x.size(1) && w2.size(0) == x.size(1) && w2.size(1) == w1.size(0) &&
           w1.scalar_type() == x.scalar_type() && w2.scalar_type() == x.scalar_type() &&
           sswin_mlp_preferred(code_of(x.scalar_type()), x.size(0), (int)x.size(1), (int)w1.size(0));
}
Tensor mlp_workspace(const Tensor& x, const Tensor& w1, bool backward, size_t& nb) {
    nb = sswin_mlp_workspace_bytes(code_of(x.scalar_type()), (int)x.size(1), (int)w1.size(0), backward);
    return nb ? bytes(nb, x) : Tensor();
}
Tensor feed_forward(const Tensor& x, const Tensor& w1_in, const Tensor& b1_in, const Tensor& w2_in, const Tensor& b2_in, const Tensor& residual, Tensor* act,
                    Tensor* slope) {
    auto bias_of = [&](const Tensor& b, int64_t n) { return !b.defined() || (b.dim() == 1 && b.size(0) == n && b.scalar_type() == x.scalar_type()); };
    const int64_t N = x.size(0), D = x.size(1);
    if (mlp_takes(x, w1_in, w2_in) && bias_of(b1_in, w1_in.size(0)) && bias_of(b2_in, D) && residual.dim() == 2 && residual.sizes() == x.sizes()) {
        const Tensor w1 = ready(w1_in), b1 = ready(b1_in), w2 = ready(w2_in), b2 = ready(b2_in);
        const int64_t hidden = w1.size(0);
        Tensor y = at::empty(x.sizes(), residual.options());
        if (act) *act = at::empty({N, hidden}, x.options()), *slope = at::empty({N, hidden}, x.options());
        size_t nb;
        const Tensor ws = mlp_workspace(x, w1, false, nb);
        RUN(sswin_mlp_forward(code_of(x.scalar_type()), code_of(residual.scalar_type()), ptr(x), N, (int)D, (int)hidden, ptr(w1), ptr(b1), ptr(w2), ptr(b2),
                              ptr(residual), ptr(y), act ? ptr(*act) : nullptr, act ? ptr(*slope) : nullptr, ptr(ws), nb, current_stream(x)));
        return y;
    }
    const Tensor g = dense(x, w1_in, b1_in, SSWIN_DENSE_GELU, Tensor(), slope);
    if (act) *act = g;
    return dense(g, w2_in, b2_in, SSWIN_DENSE_RESIDUAL, residual, nullptr, residual.scalar_type());
}
// dy [N, D] -> du [N, hidden] = (dy w2) slope and dx = du w1
std::pair<Tensor, Tensor> feed_forward_dx(const Tensor& dy, const Tensor& w1_in, const Tensor& w2_in, const Tensor& slope) {
    const Tensor w1 = ready(w1_in), w2 = ready(w2_in);
    const int64_t N = dy.size(0), D = dy.size(1), hidden = w1.size(0);
    Tensor du = at::empty({N, hidden}, dy.options()), dx = at::empty({N, D}, dy.options());
    size_t nb;
    const Tensor ws = mlp_workspace(dy, w1, true, nb);
    RUN(sswin_mlp_backward(code_of(dy.scalar_type()), ptr(dy), N, (int)D, (int)hidden, ptr(w1), ptr(w2), ptr(slope), ptr(du), ptr(dx), ptr(ws), nb,
                           current_stream(dy)));
    return {du, dx};
}

// ------------------------------------------------------------------------------------------
// row normalisation
// ------------------------------------------------------------------------------------------
Tensor norm_forward(const Tensor& x, const Tensor& gamma_in, const Tensor& beta_in, double eps, ScalarType out, Tensor* stats) {
    TORCH_CHECK(x.dim() == 2 && gamma_in.dim() == 1 && gamma_in.size(0) == x.size(1) && beta_in.sizes() == gamma_in.sizes() &&
                    gamma_in.scalar_type() == x.scalar_type() && beta_in.scalar_type() == x.scalar_type(),
                "a norm with a gain of ", gamma_in.sizes(), " ", gamma_in.scalar_type(), " and an offset of ", beta_in.sizes(), " ", beta_in.scalar_type(),
                " on rows of ", x.sizes(), " ", x.scalar_type());
    const Tensor gamma = ready(gamma_in), beta = ready(beta_in);
    Tensor y = at::empty(x.sizes(), x.options().dtype(out));
    if (stats) *stats = at::empty({2, x.size(0)}, x.options().dtype(at::kFloat));
    RUN(sswin_layer_norm_forward(code_of(x.scalar_type()), code_of(out), ptr(x), x.size(0), (int)x.size(1), ptr(gamma), ptr(beta), (float)eps, ptr(y),
                                 stats ? f32(*stats) : nullptr, current_stream(x)));
    return y;
}

// copy: dx in dy's type as well
Tensor norm_backward(const Tensor& dy, const Tensor& x, const Tensor& stats, const Tensor& gamma_in, const Tensor& dres, Tensor& dgamma, Tensor& dbeta,
                     Tensor* copy = nullptr) {
    const Tensor gamma = ready(gamma_in);
    Tensor dx = at::empty_like(x);
    dgamma = at::empty_like(gamma);
    dbeta = at::empty_like(gamma);
    const size_t nb = sswin_layer_norm_backward_workspace_bytes(code_of(x.scalar_type()), x.size(0), (int)x.size(1));
    Tensor ws = bytes(nb, x);
    if (copy) *copy = dy.scalar_type() == x.scalar_type() ? dx : at::empty(x.sizes(), dy.options());
    RUN(sswin_layer_norm_backward_copy(code_of(x.scalar_type()), code_of(dy.scalar_type()), ptr(dy), ptr(x), f32(stats), x.size(0), (int)x.size(1),
                                       ptr(gamma), ptr(dres), ptr(dx), copy && !copy->is_same(dx) ? ptr(*copy) : nullptr, ptr(dgamma), ptr(dbeta), ptr(ws),
                                       nb, current_stream(x)));
    return dx;
}

// ------------------------------------------------------------------------------------------
// attention on a projected qkv [N, 3 H hd]
// ------------------------------------------------------------------------------------------
struct Attention : torch::CustomClassHolder {
    PlanPtr plan;
    Tensor mask;            // int8 [nW, n] or undefined
    Tensor code;            // int32 position codes of the bias table, or undefined: the bias is [H, n, n]
    int offset0 = 0, n = 0, H = 0;
    double scale = 1.0;
    bool resident = false;  // the window-resident kernels (heads of 32, windows of at most 128 positions)
    bool flash = false;     // the kernels for heads of 16 or 32 and windows of any size
    enum { BY_SIZE, WINDOWS, CHUNKS } family = BY_SIZE;   // which of them: a wavefront a window and head, or chunks of 32 tokens

    int regions() const { return mask.defined() ? (int)mask.size(0) : 0; }
};
using AttentionPtr = c10::intrusive_ptr<Attention>;

struct AttentionSaved {
    Tensor bias32, aux;     // bias or table; log-sum-exp of every attention row, or P
    Tensor words;           // flash, int32.  A wavefront a window and head: token words [N], the list of the windows and the forward's largest |V|;
                            // chunks: token words [N], window offsets [N], and the order of the work where there is one
};

// What the kernels that take a window and head a wavefront add to the token words; 0: the chunks' kernels run
int64_t flash_list_ints(const Attention& a, int dt, int64_t N, int hd, int rows) {
    const int64_t windows = a.plan->G / a.H;
    if (a.family == Attention::CHUNKS || (a.family == Attention::BY_SIZE && !sswin_flash_window_faster(N, windows, a.plan->A / a.H))) return 0;
    const int64_t ints = (int64_t)sswin_flash_window_list_ints(dt, N, a.H, hd, a.n, rows, windows);
    TORCH_CHECK(ints || a.family != Attention::WINDOWS, "attention: no shape for a wavefront a window and head");
    return ints;
}

Tensor attention_forward(Attention& a, const Tensor& qkv, const Tensor& bias, AttentionSaved& saved) {
    Plan& tp = *a.plan;
    tp.finish();
    TORCH_CHECK(qkv.dim() == 2 && qkv.size(0) == tp.N && qkv.size(1) % (3 * a.H) == 0 && tp.H == a.H && tp.n == a.n, "attention: qkv of ", qkv.sizes(),
                " for a plan of ", tp.N, " tokens in windows of ", tp.n, " and ", tp.H, " heads");
    TORCH_CHECK(!tp.order_only && (!a.resident || tp.tasks.defined()), "attention: the plan was made without what the attention reads");
    same_device(qkv, {&bias, &a.mask, &a.code, &tp.tokens});
    TORCH_CHECK(!a.code.defined() || (a.code.numel() == a.n && a.code.scalar_type() == at::kInt && a.code.is_contiguous()), "attention: position codes of ",
                a.code.sizes());
    TORCH_CHECK(a.code.defined() ? bias.dim() == 2 && bias.size(1) == a.H : bias.dim() == 3 && bias.size(0) == a.H && bias.size(1) == a.n && bias.size(2) == a.n,
                "attention: bias of ", bias.sizes());
    TORCH_CHECK(!a.mask.defined() || (a.mask.dim() == 2 && a.mask.size(0) > 0 && a.mask.size(1) == a.n), "attention: mask of ", a.mask.sizes());
    if (a.flash && !(a.scale > 0 && sswin_flash_supported(code_of(qkv.scalar_type()), qkv.size(0), a.H, (int)(qkv.size(1) / 3 / a.H), (int)bias.size(0))))
        a.flash = false;                                                 // more tokens than the kernels address: the products
    TORCH_CHECK(!a.resident || tp.oversize == 0, "window-resident attention: ", tp.oversize, " groups hold more than 128 tokens");
    const int64_t N = qkv.size(0), D = qkv.size(1) / 3;
    const int hd = (int)(D / a.H), dt = code_of(qkv.scalar_type());
    void* s = current_stream(qkv);
    const auto fopt = qkv.options().dtype(at::kFloat);
    if (a.flash) {
        const Tensor table32 = saved.bias32 = bias.to(at::kFloat).contiguous();
        const int64_t listed = flash_list_ints(a, dt, N, hd, (int)table32.size(0));
        if (listed) {                                                    // a wavefront a window and head
            saved.words = at::empty({N + listed}, tp.tokens.options());
            saved.aux = at::empty({a.H, N}, fopt);
            Tensor o = at::empty({N, D}, qkv.options());
            int32_t* const list = i32(saved.words) + N;
            RUN_NAMED("sswin_flash_tokens", sswin_flash_window_tokens(i32(tp.plan), tp.g_cap, tp.G, i32(tp.tokens), N, a.H, a.n, i32(a.code),
                                                                      a.mask.defined() ? a.mask.data_ptr<int8_t>() : nullptr, a.regions(), i32(saved.words), list, s));
            RUN_NAMED("sswin_flash_forward", sswin_flash_window_forward(dt, i32(tp.plan), tp.g_cap, tp.G, i32(tp.tokens), i32(saved.words), list, N, a.H, hd, a.n,
                                                                        ptr(qkv), (float)a.scale, f32(table32), (int)table32.size(0), a.offset0, ptr(o),
                                                                        f32(saved.aux), s));
            return o;
        }
        const int64_t ordered = (int64_t)sswin_flash_order_ints(N, a.H);
        saved.words = at::empty({2 * N + ordered}, tp.tokens.options());
        int32_t* const order = ordered ? i32(saved.words) + 2 * N : nullptr;
        saved.aux = at::empty({a.H, N}, fopt);
        Tensor o = at::empty({N, D}, qkv.options());
        RUN_NAMED("sswin_flash_tokens", sswin_flash_tokens_ordered(i32(tp.plan), tp.g_cap, tp.G, i32(tp.tokens), N, a.H, a.n, i32(a.code),
                                                                   a.mask.defined() ? a.mask.data_ptr<int8_t>() : nullptr, a.regions(), i32(saved.words),
                                                                   i32(saved.words) + N, order, s));
        RUN_NAMED("sswin_flash_forward", sswin_flash_forward_ordered(dt, i32(tp.tokens), i32(saved.words), order, N, a.H, hd, a.n, ptr(qkv), (float)a.scale,
                                                                     f32(table32), (int)table32.size(0), a.offset0, ptr(o), f32(saved.aux), s));
        return o;
    }
    if (a.code.defined()) {
        const ScalarType kind = bias.scalar_type();
        const Tensor table = (kind == at::kHalf || kind == at::kBFloat16 ? bias : bias.to(at::kFloat)).contiguous();
        if (a.resident) {                                                // as [query, key] and turned
            saved.bias32 = at::empty({2, a.H, a.n, a.n}, fopt);
            RUN(sswin_bias_pair_from_typed_table(code_of(table.scalar_type()), ptr(table), (int)table.size(0), a.H, i32(a.code), a.offset0, a.n,
                                                 f32(saved.bias32), s));
        } else {
            saved.bias32 = at::empty({a.H, a.n, a.n}, fopt);
            RUN(sswin_bias_from_typed_table(code_of(table.scalar_type()), ptr(table), (int)table.size(0), a.H, i32(a.code), a.offset0, a.n,
                                            f32(saved.bias32), s));
        }
    } else {
        saved.bias32 = bias.to(at::kFloat).contiguous();
    }
    Tensor out = at::empty({N, D}, qkv.options());
    const int8_t* mask = a.mask.defined() ? a.mask.data_ptr<int8_t>() : nullptr;
    if (a.resident) {
        saved.aux = at::empty({std::max<int64_t>(a.H * N, 1)}, fopt);
        const auto run = a.code.defined() ? sswin_window_attention_forward_pair : sswin_window_attention_forward;
        RUN_NAMED("sswin_window_attention_forward", run(dt, i32(tp.tasks), tp.g_cap, tp.buckets, i32(tp.tokens), N, a.H, hd, ptr(qkv), 3 * D, 0, ptr(qkv),
                                                        3 * D, (int)D, ptr(qkv), 3 * D, (int)(2 * D), (float)a.scale, f32(saved.bias32), a.n, mask,
                                                        a.regions(), ptr(out), D, 0, f32(saved.aux), s));
        return out;
    }
    Tensor p = saved.aux = at::empty({tp.A}, fopt);
    RUN(sswin_fused_tokens_to_sq(dt, 1, i32(tp.plan), tp.g_cap, tp.G, i32(tp.tokens), tp.N, tp.H, hd, ptr(qkv), 3 * D, 0, ptr(qkv), 3 * D, (int)D,
                                 (float)a.scale, f32(saved.bias32), a.n, mask, a.regions(), f32(p), nullptr, s));
    RUN(sswin_group_softmax(0, i32(tp.plan), tp.g_cap, tp.G, tp.N, tp.H, (int)tp.c_max, f32(p), nullptr, f32(p), s));
    RUN(sswin_fused_sq_to_tokens(dt, 0, i32(tp.plan), tp.g_cap, tp.G, i32(tp.tokens), tp.N, tp.H, hd, f32(p), ptr(qkv), 3 * D, (int)(2 * D), ptr(out), D, 0,
                                 1.f, s));
    return out;
}

// gradient of the [H, n, n] bias, or of the [rows, H] table where positions are coded, from dS, one [c x c] block per group
Tensor bias_gradient(Plan& tp, int H, int n, const Tensor& code, int offset0, const Tensor& d_s, at::IntArrayRef sizes, ScalarType type) {
    void* s = current_stream(d_s);
    Tensor out;
    if (!code.defined()) {
        out = at::zeros(sizes, d_s.options());
        const size_t nb = sswin_fused_bias_grad_workspace_bytes(tp.G, H, n);
        Tensor ws = bytes(nb, d_s);
        RUN(sswin_fused_bias_grad(i32(tp.plan), tp.g_cap, tp.G, i32(tp.tokens), tp.N, H, n, f32(d_s), f32(out), ptr(ws), nb, s));
        return out.to(type);
    }
    const int rows = (int)sizes[0];
    out = at::empty(sizes, d_s.options());
    const size_t nb = sswin_bias_table_grad_workspace_bytes(tp.G, H, rows);
    Tensor ws = bytes(nb, d_s);
    if (tp.tasks.defined() && n <= 128 && tp.buckets[0] + tp.buckets[1] + tp.buckets[2] + tp.buckets[3] == tp.G)
        // every group has a task descriptor: the batches of dS are dealt evenly from the descriptor lists
        RUN(sswin_bias_table_grad_tasks(i32(tp.tasks), tp.g_cap, tp.buckets, tp.G, i32(tp.tokens), tp.N, H, n, i32(code), offset0, rows, f32(d_s),
                                        f32(out), ptr(ws), nb, s));
    else
        RUN(sswin_bias_table_grad(i32(tp.plan), tp.g_cap, tp.G, i32(tp.tokens), tp.N, H, n, i32(code), offset0, rows, f32(d_s), f32(out), ptr(ws), nb, s));
    return out.to(type);
}
Tensor bias_gradient(const Attention& a, const Tensor& d_s, const Tensor& bias) {
    return bias_gradient(*a.plan, a.H, a.n, a.code, a.offset0, d_s, bias.sizes(), bias.scalar_type());
}

Tensor attention_backward(const Attention& a, const Tensor& qkv, const Tensor& bias, const AttentionSaved& saved, const Tensor& out, const Tensor& d_out,
                          bool want_bias, Tensor& d_bias) {
    Plan& tp = *a.plan;
    const int64_t N = qkv.size(0), D = qkv.size(1) / 3;
    const int hd = (int)(D / a.H), dt = code_of(qkv.scalar_type());
    void* s = current_stream(qkv);
    Tensor d_qkv = at::empty_like(qkv);
    const auto fopt = qkv.options().dtype(at::kFloat);
    if (a.flash && flash_list_ints(a, dt, N, hd, (int)saved.bias32.size(0))) {
        const int rows = (int)saved.bias32.size(0);
        Tensor d_table = want_bias ? at::empty({rows, a.H}, fopt) : Tensor();
        const size_t nb = sswin_flash_window_backward_workspace_bytes(N, a.H, rows, tp.G / a.H);
        Tensor ws = bytes(nb, qkv);
        RUN_NAMED("sswin_flash_backward", sswin_flash_window_backward(dt, i32(tp.plan), tp.g_cap, tp.G, i32(tp.tokens), i32(saved.words), i32(saved.words) + N, N, a.H,
                                                                      hd, a.n, ptr(qkv), (float)a.scale, f32(saved.bias32), rows, a.offset0, ptr(out),
                                                                      f32(saved.aux), ptr(d_out), ptr(d_qkv), f32(d_table), ptr(ws), nb, s));
        if (want_bias) d_bias = d_table.to(bias.scalar_type());
        return d_qkv;
    }
    if (a.flash) {
        Tensor d_s = want_bias ? at::empty({std::max<int64_t>(tp.A, 1)}, fopt) : Tensor(), delta = at::empty({a.H, N}, fopt);
        RUN_NAMED("sswin_flash_backward", sswin_flash_backward_ordered(dt, i32(tp.tokens), i32(saved.words), i32(saved.words) + N,
                                                                       saved.words.numel() > 2 * N ? i32(saved.words) + 2 * N : nullptr, N, a.H, hd, a.n, ptr(qkv),
                                                                       (float)a.scale, f32(saved.bias32), (int)saved.bias32.size(0), a.offset0, ptr(out),
                                                                       f32(saved.aux), ptr(d_out), ptr(d_qkv), f32(delta), f32(d_s), s));
        if (want_bias) d_bias = bias_gradient(a, d_s, bias);
        return d_qkv;
    }
    if (a.resident) {
        const int8_t* mask = a.mask.defined() ? a.mask.data_ptr<int8_t>() : nullptr;
        Tensor d_s = want_bias ? at::empty({std::max<int64_t>(tp.A, 1)}, fopt) : Tensor();
        const bool pair = a.code.defined();                              // as the forward stored it
        TORCH_CHECK(saved.bias32.numel() == (pair ? 2 : 1) * (int64_t)a.H * a.n * a.n, "attention: a saved bias of ", saved.bias32.sizes());
        const auto run = pair ? sswin_window_attention_backward_pair : sswin_window_attention_backward;
        RUN_NAMED("sswin_window_attention_backward", run(dt, i32(tp.tasks), tp.g_cap, tp.buckets, i32(tp.tokens), N, a.H, hd, ptr(qkv), 3 * D, 0, ptr(qkv),
                                                         3 * D, (int)D, ptr(qkv), 3 * D, (int)(2 * D), (float)a.scale, f32(saved.bias32), a.n, mask,
                                                         a.regions(), ptr(out), D, 0, ptr(d_out), D, 0, f32(saved.aux), ptr(d_qkv), 3 * D, 0, ptr(d_qkv),
                                                         3 * D, (int)D, ptr(d_qkv), 3 * D, (int)(2 * D), f32(d_s), 3, s));
        if (want_bias) d_bias = bias_gradient(a, d_s, bias);
        return d_qkv;
    }
    const Tensor& p = saved.aux;
    Tensor d_s = at::empty({tp.A}, fopt);
    // dS = P (dO V^T - dO . O): the softmax backward is the epilogue of the product ; dV = P^T dO
    RUN(sswin_fused_score_grad(dt, i32(tp.plan), tp.g_cap, tp.G, i32(tp.tokens), tp.N, tp.H, hd, (int)tp.c_max, ptr(d_out), D, 0, ptr(qkv), 3 * D,
                               (int)(2 * D), ptr(out), D, 0, f32(p), f32(d_s), s));
    auto to_tokens = [&](int kmajor, const Tensor& sq, const Tensor& b, int64_t stride, int col, int o_col, float scale) {
        RUN(sswin_fused_sq_to_tokens(dt, kmajor, i32(tp.plan), tp.g_cap, tp.G, i32(tp.tokens), tp.N, tp.H, hd, f32(sq), ptr(b), stride, col, ptr(d_qkv), 3 * D,
                                     o_col, scale, s));
    };
    to_tokens(1, p, d_out, D, 0, (int)(2 * D), 1.f);
    // dQ = scale * dS K ; dK = scale * dS^T Q
    to_tokens(0, d_s, qkv, 3 * D, (int)D, 0, (float)a.scale);
    to_tokens(1, d_s, qkv, 3 * D, 0, (int)D, (float)a.scale);
    if (want_bias) d_bias = bias_gradient(a, d_s, bias);
    return d_qkv;
}

// ------------------------------------------------------------------------------------------
// autograd nodes
// ------------------------------------------------------------------------------------------
// gradients formed by kernels carry no graph of their own: differentiating them again is an error, not a zero
variable_list once(variable_list grads) {
    if (!at::GradMode::is_enabled()) return grads;
    variable_list marked;
    for (Tensor& g : grads) marked.push_back(g.defined() ? g.detach().set_requires_grad(true) : g);
    auto node = std::make_shared<torch::autograd::DelayedError>("trying to differentiate twice a function that was marked with @once_differentiable",
                                                                 (int64_t)marked.size());
    return (*node)(std::move(marked));
}

struct NoAutocast {
    c10::impl::ExcludeDispatchKeyGuard guard{c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA)};
};

template <typename T> c10::IValue capsule(const c10::intrusive_ptr<T>& p) { return c10::IValue::make_capsule(p); }
template <typename T> c10::intrusive_ptr<T> opened(const c10::IValue& v) { return c10::static_intrusive_pointer_cast<T>(v.toCapsule()); }

Tensor or_undefined(const OptTensor& t) { return t ? *t : Tensor(); }
bool asks(const Tensor& t) { return t.defined() && t.requires_grad(); }

// Whether a call has to be an autograd node.  A forward-mode tangent counts with gradients switched off as well: the node
// refuses it, the bare computation would drop it.
bool wants_node(const Tensor& t) { return t.defined() && ((at::GradMode::is_enabled() && t.requires_grad()) || t._fw_grad(0).defined()); }
bool wants_node(std::initializer_list<const Tensor*> ts) {
    for (const Tensor* t : ts)
        if (wants_node(*t)) return true;
    return false;
}

// attention alone: qkv [N, 3, H, hd] -> [N, H hd]
struct AttentionNode : torch::autograd::Function<AttentionNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& bias, AttentionPtr a) {
        NoAutocast off;
        const Tensor x = ready(qkv);
        const Tensor flat = x.view({x.size(0), -1});
        AttentionSaved saved;
        Tensor out = attention_forward(*a, flat, bias, saved);
        if (ctx) {
            ctx->save_for_backward({flat, bias, saved.bias32, saved.aux, out, saved.words});
            ctx->saved_data["a"] = capsule(a);
            ctx->saved_data["shape"] = qkv.sizes();
            ctx->saved_data["bias"] = bias.requires_grad();
        }
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        NoAutocast off;
        const auto v = ctx->get_saved_variables();
        const auto a = opened<Attention>(ctx->saved_data["a"]);
        c10::hip::HIPGuardMasqueradingAsCUDA guard(v[0].device());
        Tensor d_bias;
        const Tensor d_out = ready(grads[0].to(v[0].scalar_type()));
        Tensor d = attention_backward(*a, v[0], v[1], AttentionSaved{v[2], v[3], v[5]}, v[4], d_out, ctx->saved_data["bias"].toBool(), d_bias);
        return once({d.view(ctx->saved_data["shape"].toIntVector()), d_bias, Tensor()});
    }
};

// the attention module: proj(attention(qkv(x)))
struct ModuleNode : torch::autograd::Function<ModuleNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& qkv_w, const OptTensor& qkv_bias, const Tensor& bias,
                          const Tensor& proj_w, const OptTensor& proj_bias, AttentionPtr a, ScalarType type) {
        NoAutocast off;
        const Tensor qkv_b = or_undefined(qkv_bias), proj_b = or_undefined(proj_bias);
        same_device(x_in, {&qkv_w, &qkv_b, &proj_w, &proj_b});
        const Tensor x = ready(x_in.to(type));
        const auto w = in_type<4>({qkv_w, qkv_b, proj_w, proj_b}, type);
        const Tensor qkv = dense(x, w[0], w[1]);
        AttentionSaved saved;
        Tensor o = attention_forward(*a, qkv, bias, saved);
        Tensor y = dense(o, w[2], w[3]);
        if (ctx) {
            ctx->save_for_backward({x, w[0], bias, w[2], qkv, saved.bias32, saved.aux, o, saved.words});
            ctx->saved_data["a"] = capsule(a);
            ctx->saved_data["how"] = std::vector<int64_t>{(int64_t)x_in.scalar_type(), x_in.requires_grad(), qkv_w.requires_grad(), asks(qkv_b),
                                                          bias.requires_grad(), proj_w.requires_grad(), asks(proj_b), (int64_t)qkv_w.scalar_type(),
                                                          (int64_t)proj_w.scalar_type()};
        }
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        NoAutocast off;
        const auto v = ctx->get_saved_variables();
        const auto a = opened<Attention>(ctx->saved_data["a"]);
        const auto how = ctx->saved_data["how"].toIntVector();
        const Tensor &x = v[0], &qkv_w = v[1], &bias = v[2], &proj_w = v[3], &qkv = v[4], &o = v[7];
        c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
        const Tensor dy = ready(grads[0].to(x.scalar_type()));
        Tensor d_bias;
        const DenseGrads d_proj = dense_backward(dy, o, proj_w, true, how[5], how[6], (ScalarType)how[8]);
        const Tensor d_qkv = attention_backward(*a, qkv, bias, AttentionSaved{v[5], v[6], v[8]}, o, d_proj.dx, how[4], d_bias);
        const DenseGrads d_in = dense_backward(d_qkv, x, qkv_w, how[1], how[2], how[3], (ScalarType)how[7]);
        const Tensor dx = how[1] ? d_in.dx.to((ScalarType)how[0]) : Tensor();
        return once({dx, d_in.dw, d_in.db, d_bias, d_proj.dw, d_proj.db, Tensor(), Tensor()});
    }
};

// the transformer block: h = x + proj(attention(qkv(norm1(x)))), y = h + linear2(gelu(linear1(norm2(h))))
struct BlockNode : torch::autograd::Function<BlockNode> {
    enum { X, G1, B1, QKVW, QKVB, TABLE, PROJW, PROJB, G2, B2, W1, C1, W2, C2, PARAMS };
    // given: the tensors that are there; which: the enumerator of each (biases may be missing)
    static Tensor forward(AutogradContext* ctx, at::TensorList given, std::vector<int64_t> which, AttentionPtr a, double eps1, double eps2,
                          ScalarType type) {
        NoAutocast off;
        Tensor p[PARAMS];
        for (size_t i = 0; i < which.size(); ++i) {
            p[which[i]] = given[i];
            same_device(p[X], {&p[which[i]]});
        }
        const Tensor x = ready(p[X]);
        const ScalarType stream_type = x.scalar_type();                  // of the residual stream
        const ScalarType params_type = p[QKVW].scalar_type();
        Tensor stats1, stats2, slope;
        const auto w = in_type<8>({p[QKVW], p[QKVB], p[PROJW], p[PROJB], p[W1], p[C1], p[W2], p[C2]}, type);
        const Tensor x1 = norm_forward(x, p[G1], p[B1], eps1, type, ctx ? &stats1 : nullptr);
        const Tensor qkv = dense(x1, w[0], w[1]);
        AttentionSaved saved;
        const Tensor o = attention_forward(*a, qkv, p[TABLE], saved);
        const Tensor h = dense(o, w[2], w[3], SSWIN_DENSE_RESIDUAL, x, nullptr, stream_type);
        const Tensor x2 = norm_forward(h, p[G2], p[B2], eps2, type, ctx ? &stats2 : nullptr);
        Tensor g;
        Tensor y = feed_forward(x2, w[4], w[5], w[6], w[7], h, ctx ? &g : nullptr, ctx ? &slope : nullptr);
        if (ctx) {
            ctx->save_for_backward({x, p[G1], w[0], p[TABLE], w[2], p[G2], w[4], w[6], stats1, x1, qkv, saved.bias32, saved.aux, o, h, stats2, x2, g,
                                    slope, saved.words});
            ctx->saved_data["a"] = capsule(a);
            ctx->saved_data["which"] = which;
            std::vector<int64_t> asked;
            for (const Tensor& t : p) asked.push_back(asks(t));
            ctx->saved_data["asked"] = asked;
            ctx->saved_data["params"] = (int64_t)params_type;
        }
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        NoAutocast off;
        const auto v = ctx->get_saved_variables();
        const auto a = opened<Attention>(ctx->saved_data["a"]);
        const auto which = ctx->saved_data["which"].toIntVector(), ask = ctx->saved_data["asked"].toIntVector();
        const Tensor &x = v[0], &g1 = v[1], &qkvw = v[2], &table = v[3], &projw = v[4], &g2 = v[5], &w1 = v[6], &w2 = v[7], &stats1 = v[8], &x1 = v[9],
                     &qkv = v[10], &o = v[13], &h = v[14], &stats2 = v[15], &x2 = v[16], &g = v[17], &slope = v[18];
        c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
        const ScalarType type = x1.scalar_type(), wt = (ScalarType)ctx->saved_data["params"].toInt();
        const Tensor dy = ready(grads[0]);
        const Tensor dyt = dy.to(type);
        Tensor out[PARAMS];
        auto through = [&](int w, const Tensor& d, const Tensor& in, const Tensor& weight, int epilogue = SSWIN_DENSE_PLAIN, const Tensor& extra = Tensor()) {
            DenseGrads r = dense_backward(d, in, weight, true, ask[w], ask[w + 1], wt, epilogue, extra);
            out[w] = r.dw, out[w + 1] = r.db;
            return r.dx;
        };
        Tensor d_x2;
        if (mlp_takes(x2, w1, w2)) {
            const auto [du, dx] = feed_forward_dx(dyt, w1, w2, slope);
            if (ask[W2] || ask[C2]) std::tie(out[W2], out[C2]) = dense_dw(dyt, g, ask[C2], wt);
            if (ask[W1] || ask[C1]) std::tie(out[W1], out[C1]) = dense_dw(du, x2, ask[C1], wt);
            d_x2 = dx;
        } else {
            d_x2 = through(W1, through(W2, dyt, g, w2, SSWIN_DENSE_SCALE, slope), x2, w1);
        }
        Tensor dht;                                                      // dh in the layers' type
        const Tensor dh = norm_backward(d_x2, h, stats2, g2, dy, out[G2], out[B2], &dht);
        const Tensor d_o = through(PROJW, dht, o, projw);
        const Tensor d_qkv = attention_backward(*a, qkv, table, AttentionSaved{v[11], v[12], v[19]}, o, d_o, ask[TABLE], out[TABLE]);
        out[X] = norm_backward(through(QKVW, d_qkv, x1, qkvw), x, stats1, g1, dh, out[G1], out[B1]);
        variable_list result;
        for (int64_t w : which) result.push_back(ask[w] ? out[w] : Tensor());
        result.resize(which.size() + 5);                                 // the arguments that are no tensors
        return once(std::move(result));
    }
};

// stride-2 merge: mean of the children's rows, norm, Linear
struct MergeNode : torch::autograd::Function<MergeNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& gamma, const Tensor& beta, const Tensor& w, PlanPtr plan, double eps,
                          ScalarType type) {
        NoAutocast off;
        plan->finish();
        TORCH_CHECK(x_in.dim() == 2 && x_in.size(0) == plan->N, "merge: rows of ", x_in.sizes(), " for a plan of ", plan->N, " voxels");
        same_device(x_in, {&gamma, &beta, &w, &plan->tokens});
        const Tensor x = ready(x_in);
        const int64_t M = plan->windows, D = x.size(1);
        Tensor pooled = at::empty({M, D}, x.options()), stats;
        RUN(sswin_pool_windows(code_of(x.scalar_type()), 0, 1, i32(plan->plan), plan->g_cap, M, i32(plan->tokens), plan->N, ptr(x), D, (int)D, ptr(pooled), D,
                               current_stream(x)));
        const Tensor x1 = norm_forward(pooled, gamma, beta, eps, type, ctx ? &stats : nullptr);
        const auto wt = in_type<1>({w}, type);
        Tensor y = dense(x1, wt[0], Tensor());
        if (ctx) {
            ctx->save_for_backward({gamma, wt[0], pooled, stats, x1});
            ctx->saved_data["params"] = (int64_t)w.scalar_type();
            ctx->saved_data["p"] = capsule(plan);
        }
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        NoAutocast off;
        const auto v = ctx->get_saved_variables();
        const auto plan = opened<Plan>(ctx->saved_data["p"]);
        const Tensor &gamma = v[0], &w = v[1], &pooled = v[2], &stats = v[3], &x1 = v[4];
        c10::hip::HIPGuardMasqueradingAsCUDA guard(pooled.device());
        const Tensor dy = ready(grads[0].to(x1.scalar_type()));
        Tensor dg, db;
        const DenseGrads d = dense_backward(dy, x1, w, true, true, false, (ScalarType)ctx->saved_data["params"].toInt());
        const Tensor d_pool = norm_backward(d.dx, pooled, stats, gamma, Tensor(), dg, db);
        const int64_t D = pooled.size(1);
        Tensor dx = at::empty({plan->N, D}, pooled.options());
        RUN(sswin_pool_windows(code_of(dx.scalar_type()), 1, 1, i32(plan->plan), plan->g_cap, plan->windows, i32(plan->tokens), plan->N, ptr(d_pool), D, (int)D,
                               ptr(dx), D, current_stream(dx)));
        return once({dx, dg, db, d.dw, Tensor(), Tensor(), Tensor()});
    }
};

// ------------------------------------------------------------------------------------------
// Python entry points
// ------------------------------------------------------------------------------------------
// path: "resident", "flash" or "products" (the attention matrix in memory); "flash_windows" and "flash_chunks" are the two families of flash kernels
// whatever the sizes
AttentionPtr make_attention(const PlanPtr& plan, const OptTensor& mask, const OptTensor& code, int64_t offset0, int64_t n, int64_t heads, double scale,
                            const std::string& path) {
    auto a = c10::make_intrusive<Attention>();
    a->plan = plan;
    if (mask) a->mask = mask->to(at::kChar).contiguous();
    if (code) a->code = *code;
    a->offset0 = (int)offset0, a->n = (int)n, a->H = (int)heads, a->scale = scale;
    a->resident = path == "resident", a->flash = path.rfind("flash", 0) == 0;
    a->family = path == "flash_windows" ? Attention::WINDOWS : path == "flash_chunks" ? Attention::CHUNKS : Attention::BY_SIZE;
    TORCH_CHECK(a->resident || path == "flash" || a->family != Attention::BY_SIZE || path == "products", "attention path ", path);
    TORCH_CHECK(!a->flash || code, "the flash path takes its bias from a relative position table");
    return a;
}

Tensor attention(const Tensor& qkv, const Tensor& bias, const PlanPtr& plan, const OptTensor& mask, const OptTensor& code, int64_t offset0, int64_t n,
                 double scale, const std::string& path) {
    c10::hip::HIPGuardMasqueradingAsCUDA guard(qkv.device());
    auto a = make_attention(plan, mask, code, offset0, n, qkv.size(2), scale, path);
    if (!wants_node({&qkv, &bias})) return AttentionNode::forward(nullptr, qkv, bias, a);
    return AttentionNode::apply(qkv, bias, a);
}

Tensor attention_module(const Tensor& x, const Tensor& qkv_w, const OptTensor& qkv_b, const Tensor& bias, const Tensor& proj_w, const OptTensor& proj_b,
                        const PlanPtr& plan, const OptTensor& mask, const OptTensor& code, int64_t offset0, int64_t n, int64_t heads, double scale,
                        const std::string& path, ScalarType type) {
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    auto a = make_attention(plan, mask, code, offset0, n, heads, scale, path);
    const Tensor qb = or_undefined(qkv_b), pb = or_undefined(proj_b);
    if (!wants_node({&x, &qkv_w, &qb, &bias, &proj_w, &pb})) return ModuleNode::forward(nullptr, x, qkv_w, qkv_b, bias, proj_w, proj_b, a, type);
    return ModuleNode::apply(x, qkv_w, qkv_b, bias, proj_w, proj_b, a, type);
}

Tensor block(std::vector<OptTensor> params, const PlanPtr& plan, const OptTensor& mask, const Tensor& code, int64_t offset0, int64_t n, int64_t heads,
             double scale, const std::string& path, double eps1, double eps2, ScalarType type) {
    TORCH_CHECK(params.size() == BlockNode::PARAMS, "block: ", (int)BlockNode::PARAMS, " tensors expected");
    variable_list given;
    std::vector<int64_t> which;
    bool node = false;
    for (size_t i = 0; i < params.size(); ++i)
        if (params[i] && params[i]->defined()) {
            node = node || wants_node(*params[i]);
            given.push_back(*params[i]);
            which.push_back((int64_t)i);
        }
    c10::hip::HIPGuardMasqueradingAsCUDA guard(given.at(0).device());
    auto a = make_attention(plan, mask, code, offset0, n, heads, scale, path);
    if (!node) return BlockNode::forward(nullptr, given, which, a, eps1, eps2, type);
    return BlockNode::apply(at::TensorList(given), which, a, eps1, eps2, type);
}

Tensor merge(const Tensor& x, const Tensor& gamma, const Tensor& beta, const Tensor& w, const PlanPtr& plan, double eps, ScalarType type) {
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    if (!wants_node({&x, &gamma, &beta, &w})) return MergeNode::forward(nullptr, x, gamma, beta, w, plan, eps, type);
    return MergeNode::apply(x, gamma, beta, w, plan, eps, type);
}

// the bias gradient alone: dS of a plan's groups, as the operators' product lays it out
Tensor plan_bias_gradient(const PlanPtr& plan, const Tensor& d_s, const OptTensor& code, int64_t offset0, const std::vector<int64_t>& sizes, ScalarType type) {
    plan->finish();
    c10::hip::HIPGuardMasqueradingAsCUDA guard(d_s.device());
    const Tensor c = or_undefined(code);
    TORCH_CHECK(!plan->order_only && d_s.scalar_type() == at::kFloat && d_s.is_contiguous() && d_s.numel() >= plan->A, "bias gradient: dS of ", d_s.sizes(),
                " for a plan of ", plan->A, " scores");
    TORCH_CHECK(c.defined() ? sizes.size() == 2 && sizes[1] == plan->H && c.numel() == plan->n && c.scalar_type() == at::kInt && c.is_contiguous()
                            : sizes == std::vector<int64_t>({plan->H, plan->n, plan->n}),
                "bias gradient: a bias of ", sizes, " for ", plan->H, " heads and windows of ", plan->n);
    same_device(d_s, {&c, &plan->tokens});
    return bias_gradient(*plan, plan->H, (int)plan->n, c, (int)offset0, d_s, sizes, type);
}

Tensor window_coords(const PlanPtr& plan, const std::vector<int64_t>& dims, const std::vector<int64_t>& window) {
    plan->finish();
    c10::hip::HIPGuardMasqueradingAsCUDA guard(plan->plan.device());
    Tensor out = at::empty({plan->windows, 4}, plan->plan.options());
    int32_t d[3], w[3];
    for (int i = 0; i < 3; ++i) d[i] = (int32_t)dims.at(i), w[i] = (int32_t)window.at(i);
    RUN(sswin_window_coords(i32(plan->plan), plan->g_cap, plan->windows, d, w, i32(out), current_stream(out)));
    return out;
}

bool norm_supported(const Tensor& x) {
    return x.dim() == 2 && x.size(0) > 0 && (x.scalar_type() == at::kFloat || x.scalar_type() == at::kHalf || x.scalar_type() == at::kBFloat16) &&
           sswin_layer_norm_supported(code_of(x.scalar_type()), (int)x.size(1));
}

void set_recorder(py::object r) {
    PyObject* old = g_recorder;
    g_recorder = r.is_none() ? nullptr : r.release().ptr();
    Py_XDECREF(old);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    py::class_<Plan, PlanPtr>(m, "Plan")
        .def(py::init<const Tensor&, int64_t, int64_t, int64_t, bool, bool>())
        .def("_finish", &Plan::finish)
        .def_readonly("tokens", &Plan::tokens)
        .def_readonly("plan", &Plan::plan)
        .def_property_readonly("tasks", [](const Plan& p) { return p.tasks.defined() ? OptTensor(p.tasks) : std::nullopt; })
        .def_property_readonly("device", [](const Plan& p) { return p.tokens.device(); })
        .def_readonly("N", &Plan::N)
        .def_readonly("H", &Plan::H)
        .def_readonly("n", &Plan::n)
        .def_readonly("B", &Plan::B)
        .def_readonly("g_cap", &Plan::g_cap)
        .def_readonly("order_only", &Plan::order_only)
        .def_property_readonly("G", [](const Plan& p) { return p.decoded().G; })
        .def_property_readonly("windows", [](const Plan& p) { return p.decoded().windows; })
        .def_property_readonly("A", [](const Plan& p) { return p.decoded().A; })
        .def_property_readonly("c_max", [](const Plan& p) { return p.decoded().c_max; })
        .def_property_readonly("oversize_groups", [](const Plan& p) { return p.decoded().oversize; })
        .def_property_readonly("buckets", [](const Plan& p) { return std::vector<int64_t>(p.decoded().buckets, p.buckets + 4); });
    m.def("enqueue_plans", &enqueue_plans);
    m.def("window_indices", &window_indices);
    m.def("window_coords", &window_coords);
    m.def("bias_gradient", &plan_bias_gradient);
    m.def("attention", &attention);
    m.def("attention_module", &attention_module);
    m.def("block", &block);
    m.def("merge", &merge);
    m.def("norm_supported", &norm_supported);
    m.def("set_recorder", &set_recorder);
}
