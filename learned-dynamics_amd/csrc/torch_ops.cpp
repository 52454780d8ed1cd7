// Host side of the linear maps and of the PaiNN layers in C++: what ops.py and painn.py call per forward pass.  A call
// checks its operands, allocates outputs, looks packed weights up and enqueues kernels of libmanagan_hip.so on torch's
// current stream: about 3 us per launch, where the same steps through ctypes took about 12, which is what a network of
// node-sized launches was bound by.  No arithmetic happens here.
#include "torch_common.hpp"

#include <algorithm>
#include <atomic>
#include <climits>
#include <limits>
#include <map>
#include <mutex>
#include <tuple>
#include <unordered_map>

using namespace mgt;
namespace py = pybind11;

namespace {

enum { kActNone = 0, kActSilu = 1, kActLeaky = 2 };
enum { kModeFp32 = 0, kModeBf16x3 = 1, kModeF16x2 = 2 };

std::atomic<int64_t> g_epoch{0};        // of invalidate_weight_caches

// ------------------------------------------------------------------ tensors derived from weights, kept per version
// An entry belongs to a tensor OBJECT (a weak reference keeps the address from being reused) and its version counter;
// a view (the transposed weight of an input-gradient product is a fresh view of the parameter) is kept under the tensor
// it views.  It goes when that tensor does: a Python weak reference to it says when.  Inference tensors have no version
// counter: nothing is kept for them.  (Callers hold the GIL.)
void watch_owner(const at::Tensor& owner);       // entries of this tensor are forgotten when it goes

template <typename Value>
class WeightCache {
public:
    using Key = std::tuple<const void*, int, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t>;
    struct Slot {
        c10::weak_intrusive_ptr<c10::TensorImpl> owner;
        uint32_t version;
        const void* data;
        int64_t epoch;
        Value value;
    };

    // whether an entry for the current version is there (always true for tensors nothing is kept for)
    bool has(const at::Tensor& W, int kind, int64_t extra) {
        const at::Tensor owner = W.is_view() ? at::Tensor(W._base()) : W;
        if (owner.is_inference()) return true;
        c10::TensorImpl* impl = owner.unsafeGetTensorImpl();
        std::lock_guard<std::mutex> lock(mutex_);
        auto it = slots_.find(Key{impl, kind, extra, W.storage_offset(), W.size(0), W.size(-1), W.stride(0), W.stride(-1)});
        return it != slots_.end() && it->second.version == impl->version_counter().current_version() &&
               it->second.data == owner.data_ptr() && it->second.epoch == g_epoch.load();
    }

    template <typename Make>
    Value get(const at::Tensor& W, int kind, int64_t extra, Make&& make) {
        const at::Tensor owner = W.is_view() ? at::Tensor(W._base()) : W;
        if (owner.is_inference()) return make();
        c10::TensorImpl* impl = owner.unsafeGetTensorImpl();
        const Key key{impl, kind, extra, W.storage_offset(), W.size(0), W.size(-1), W.stride(0), W.stride(-1)};
        const uint32_t version = impl->version_counter().current_version();
        const void* data = owner.data_ptr();
        const int64_t epoch = g_epoch.load();
        {
            std::lock_guard<std::mutex> lock(mutex_);
            auto it = slots_.find(key);
            if (it != slots_.end() && it->second.version == version && it->second.data == data && it->second.epoch == epoch)
                return it->second.value;
        }
        Value v = make();
        watch_owner(owner);
        Slot slot{c10::weak_intrusive_ptr<c10::TensorImpl>(owner.getIntrusivePtr()), version, data, epoch, v};
        std::lock_guard<std::mutex> lock(mutex_);
        auto it = slots_.find(key);
        if (it == slots_.end()) slots_.emplace(key, std::move(slot));
        else std::swap(it->second, slot);                     // (the old value goes with `slot`, after the lock)
        return v;
    }

    void forget(const void* impl) {
        std::vector<Slot> gone;                               // (destroyed after the lock: what they free may call back)
        std::lock_guard<std::mutex> lock(mutex_);
        for (auto it = slots_.lower_bound(Key{impl, INT_MIN, INT64_MIN, INT64_MIN, INT64_MIN, INT64_MIN, INT64_MIN, INT64_MIN});
             it != slots_.end() && std::get<0>(it->first) == impl; it = slots_.erase(it))
            gone.push_back(std::move(it->second));
    }

private:
    std::mutex mutex_;
    std::map<Key, Slot> slots_;
};

template <typename Value>
WeightCache<Value>& cache() {
    static WeightCache<Value>* c = new WeightCache<Value>;     // never destroyed: the allocator may be gone by then
    return *c;
}

// Python weak references to the tensors that have entries, with one callback for all of them (the GIL guards the maps)
struct Owners {
    py::object callback;
    std::unordered_map<const void*, py::object> refs;         // tensor -> weak reference
    std::unordered_map<PyObject*, const void*> tensors;       // weak reference -> tensor
};
Owners& owners() {
    static Owners* o = new Owners;                             // never destroyed: tensors may outlive the interpreter's modules
    return *o;
}
void owner_gone(py::object ref) {
    Owners& o = owners();
    auto it = o.tensors.find(ref.ptr());
    if (it == o.tensors.end()) return;
    const void* impl = it->second;
    o.tensors.erase(it);
    o.refs.erase(impl);
    cache<at::Tensor>().forget(impl);
    cache<float>().forget(impl);
}
void watch_owner(const at::Tensor& owner) {
    Owners& o = owners();
    const void* impl = owner.unsafeGetTensorImpl();
    if (o.refs.count(impl)) return;
    if (!o.callback) o.callback = py::cpp_function(&owner_gone);
    py::object obj = py::cast(owner);
    PyObject* ref = PyWeakref_NewRef(obj.ptr(), o.callback.ptr());
    if (!ref) throw py::error_already_set();
    o.tensors.emplace(ref, impl);
    o.refs.emplace(impl, py::reinterpret_steal<py::object>(ref));
}

at::Tensor bytes_like(const at::Tensor& t, size_t n) {
    return at::empty({(int64_t)n}, t.options().dtype(at::kByte).requires_grad(false));
}
at::Tensor floats(const at::Tensor& like, at::IntArrayRef shape) {
    return at::empty(shape, like.options().requires_grad(false));
}

// fp16 hi / lo planes + inverse row scales of W, its reduction dimension zero-padded to k_pad
at::Tensor packed_f16x2(const at::Tensor& W, int64_t k_pad) {
    return cache<at::Tensor>().get(W, 2, k_pad, [&] {
        size_t n = 0;
        check(mg_linear_f16x2_packed_weight_bytes((int)k_pad, (int)W.size(0), &n));
        at::Tensor p = bytes_like(W, n);
        check(mg_linear_f16x2_pack_weight_padded(fp(W), W.stride(0), W.stride(1), (int)W.size(1), (int)W.size(0), (int)k_pad,
                                                 p.data_ptr(), stream_of(W)));
        return p;
    });
}
at::Tensor packed_bf16x3(const at::Tensor& W) {
    return cache<at::Tensor>().get(W, 1, 0, [&] {
        size_t n = 0;
        check(mg_linear_packed_weight_bytes((int)W.size(1), (int)W.size(0), &n));
        at::Tensor p = bytes_like(W, n);
        check(mg_linear_pack_weight(fp(W), W.stride(0), W.stride(1), (int)W.size(1), (int)W.size(0), p.data_ptr(), stream_of(W)));
        return p;
    });
}
at::Tensor packed_weight(const at::Tensor& W, bool f16) {
    TORCH_CHECK(W.is_cuda() && W.scalar_type() == at::kFloat && W.dim() == 2, "W must be a float32 CUDA matrix");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(W.device());
    if (!f16) return packed_bf16x3(W);
    TORCH_CHECK(W.size(1) % 8 == 0, "packed_weight_f16x2: dim_in must be a multiple of 8");
    return packed_f16x2(W, (W.size(1) + 31) / 32 * 32);
}

// (max_o sum_i |W[o, i]|, max_o |bias[o]|): |act(x W^T + bias)| <= |x|max * first + second for |act(z)| <= |z|; read back
// once per version of the parameters, both with one copy, other Python threads running meanwhile.  Infinite where a parameter
// is NaN: no bound, and the next layer goes in fp32
std::pair<float, float> norms_of(const at::Tensor& W, const OptTensor& bias) {
    auto read = [](std::vector<at::Tensor> t) {
        const at::Tensor stacked = at::stack(t);
        py::gil_scoped_release release;
        const at::Tensor host = stacked.cpu();
        std::pair<float, float> v{host.data_ptr<float>()[0], host.numel() > 1 ? host.data_ptr<float>()[1] : 0.f};
        return v;
    };
    c10::InferenceMode off(false);
    at::NoGradGuard no_grad;
    auto of_weight = [&] { return W.detach().abs().sum(1).amax(); };
    auto of_bias = [&] { return bias->detach().abs().amax(); };
    auto bound = [](float v) {                                // (a product with a row maximum must not round below the true one)
        return v == v ? v * (1.0f + 1e-6f) : std::numeric_limits<float>::infinity();
    };
    auto& kept = cache<float>();
    if (bias.has_value() && !kept.has(W, 3, 0) && !kept.has(*bias, 4, 0)) {
        const auto both = read({of_weight(), of_bias()});
        return {kept.get(W, 3, 0, [&] { return bound(both.first); }), kept.get(*bias, 4, 0, [&] { return bound(both.second); })};
    }
    const float weight = kept.get(W, 3, 0, [&] { return bound(read({of_weight()}).first); });
    return {weight, bias.has_value() ? kept.get(*bias, 4, 0, [&] { return bound(read({of_bias()}).first); }) : 0.f};
}

// ------------------------------------------------------------------ linear maps
// upper bounds of the row maxima of |x|: mul * base + add, base (rows / rows_per, parts) or (1, parts)
struct Bound {
    OptTensor base;
    float mul = 1.f, add = 0.f;
    int64_t rows_per = 1;
};

// the bound behind a layer with these norms (infinite factors stay numbers: 0 * inf would be none)
Bound through(const Bound& b, const std::pair<float, float>& norms) {
    auto product = [](float x, float y) { return x == 0.f || y == 0.f ? 0.f : x * y; };
    return Bound{b.base, product(b.mul, norms.first), product(b.add, norms.first) + norms.second, b.rows_per};
}

bool f16x2_takes(int64_t rows, int64_t dim_in, int64_t dim_out, const at::Tensor& x) {
    return dim_in % 32 == 0 && dim_in >= 64 && dim_out >= 8 && rows >= 1 && aligned16(x);
}

at::Tensor row_absmax(const at::Tensor& x) {
    check_input(x, "x");
    TORCH_CHECK(x.dim() == 2, "x must have two dims");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    at::Tensor out = floats(x, {x.size(0), 1});
    check(mg_row_absmax(fp(x), x.size(0), (int)x.size(1), fp(out), stream_of(x)));
    return out;
}

int64_t rowmax_parts(int64_t rows, int64_t dim_in, int64_t dim_out, bool sequential) {
    return sequential ? mg_tensor_linear_f16x2_rowmax_parts_sequential(rows, (int)dim_in, (int)dim_out)
                      : mg_tensor_linear_f16x2_rowmax_parts(rows, (int)dim_in, (int)dim_out);
}

// x (rows, k) plain rows; y preallocated; packed: W's planes where the caller holds them; without a base in b the rows' maxima are found on the
// way, and returned
OptTensor run_f16x2(const at::Tensor& W, int64_t k, const float* x, int64_t rows, const Bound& b, const OptTensor& bias, int act,
               bool accumulate, int out_comps, at::Tensor& y, at::Tensor* ymax, bool sequential, int64_t bias_rows = -1,
               const OptTensor& packed = OptTensor(), int64_t x_stride = -1, int64_t max_column = 0) {
    const at::Tensor planes = packed.has_value() ? *packed : packed_f16x2(W, k);
    const bool bounded = b.base.has_value();
    TORCH_CHECK(bounded || (x_stride < 0 && b.mul == 1.f && b.add == 0.f && b.rows_per == 1), "row maxima are found of contiguous rows");
    at::Tensor base = bounded ? *b.base : floats(y, {rows, 1});
    mg_f16x2_linear a{};
    a.packed_W = planes.data_ptr();
    a.x = x;
    if (bounded) {
        a.x_rowmax = fp(base) + max_column;                    // (x_stride: a column of `base` for each block of columns of x)
        a.x_rowmax_parts = x_stride < 0 ? (int)base.size(1) : 1;
        a.x_rowmax_stride = base.size(0) > 1 || rows == b.rows_per ? base.size(1) : 0;
        a.x_rows_per_bound = b.rows_per;
        a.bound_mul = b.mul;
        a.bound_add = b.add;
    }
    a.rows = rows;
    a.dim_in = (int)k;
    a.dim_out = (int)W.size(0);
    a.bias = fp(bias);
    a.bias_rows = bias_rows < 0 ? rows : bias_rows;
    a.act = act;
    a.accumulate = accumulate;
    a.out_comps = out_comps;
    a.sequential = sequential;
    a.y = fp(y);
    a.y_rowmax = ymax ? fp(*ymax) : nullptr;
    if (bounded) check(mg_tensor_linear_f16x2_run_strided(&a, x_stride < 0 ? k : x_stride, stream_of(y)));
    else check(mg_tensor_linear_f16x2_run_unbounded(&a, fp(base), stream_of(y)));
    return base;
}

void check_bound(const at::Tensor& b, int64_t rows, int64_t rows_per) {
    check_input(b, "x_rowmax");
    TORCH_CHECK(b.dim() == 2 && (b.size(0) == 1 || b.size(0) * rows_per == rows),
                "x_rowmax must be (rows / rows_per_bound, parts) or (1, parts)");
}

// y = act(x W^T + bias) for plain rows through the two-piece fp16 split
std::tuple<at::Tensor, OptTensor> linear_f16x2(const at::Tensor& W, const at::Tensor& x, const OptTensor& x_rowmax, double mul,
                                               double add, const OptTensor& bias, int act, const OptTensor& out,
                                               bool accumulate, int out_comps, bool want_rowmax, int64_t rows_per,
                                               bool sequential) {
    check_input(x, "x");
    TORCH_CHECK(x.dim() == 2 && W.dim() == 2 && x.size(1) == W.size(1), "expected x (rows, dim_in) and W (dim_out, dim_in)");
    const int64_t rows = x.size(0), dim_in = W.size(1), dim_out = W.size(0);
    Bound b{x_rowmax.has_value() ? x_rowmax : OptTensor(row_absmax(x)), (float)mul, (float)add, rows_per};
    check_bound(*b.base, rows, rows_per);
    if (bias.has_value()) {
        check_input(*bias, "bias");
        TORCH_CHECK(bias->numel() == dim_out, "bias size mismatch");
    }
    TORCH_CHECK(rows % out_comps == 0, "rows must be a multiple of out_comps");
    TORCH_CHECK(!want_rowmax || out_comps == 1, "row maxima are only produced for out_comps == 1");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    at::Tensor y;
    if (out.has_value()) {
        check_input(*out, "out");
        TORCH_CHECK(out->numel() == rows * dim_out, "out has wrong size");
        y = *out;
    } else if (out_comps == 1) {
        y = floats(x, {rows, dim_out});
    } else {
        y = floats(x, {rows / out_comps, dim_out, out_comps});
    }
    at::Tensor ymax;
    if (want_rowmax) ymax = floats(x, {rows, rowmax_parts(rows, dim_in, dim_out, sequential)});
    run_f16x2(W, dim_in, fp(x), rows, b, bias, act, accumulate, out_comps, y, want_rowmax ? &ymax : nullptr, sequential);
    return {y, want_rowmax ? OptTensor(ymax) : OptTensor()};
}

// x (rows, dim, comps) -> one plain row per (row, comp), channels zero-padded to `pad`, and the row maxima
std::pair<at::Tensor, at::Tensor> components_to_rows(const at::Tensor& x, int64_t rows, int64_t dim, int T, int64_t pad) {
    at::Tensor x2 = floats(x, {rows * T, pad}), m = floats(x, {rows * T, 1});
    check(mg_components_to_rows(fp(x), rows, (int)dim, T, (int)pad, fp(x2), fp(m), stream_of(x)));
    return {x2, m};
}

bool power_of_two(int64_t v) { return v > 0 && (v & (v - 1)) == 0; }

// Whether a tensor linear of R = rows x components goes through plain component rows and the split-fp16 kernels.
// Channels: from 32 its error against float64 is no larger than that of fp32 products summed in k order (2-norm, 32 channels
// 0.95e-7 against 1.03e-7, 64 1.0e-7 against 1.45e-7, 128 1.0e-7 against 2.0e-7); with fewer the rounding of the pieces outweighs
// the shorter sum (16 channels 0.88e-7 against 0.74e-7, 24 0.91e-7 against 0.89e-7), and they stay in fp32 below 32 768.
// R: the generic kernel is the slower one at every R that was measured, with the transposition counted (64 -> 64: 17.3 against
// 7.1 us at 960, 18.0 against 12.1 at 15 360; 256 -> 256: 32.5 against 8.9 and 47 against 30; three components), down to 96 (16.8
// against 6.8).  The line at 960 is no crossover: calls below it have kept fp32 arithmetic in k order.
// With `sequential` the line is 32 768 for every width: below it an element's order of summation does not depend on R.
constexpr int64_t kComponentRows = 960, kComponentRowsF32 = 32768, kComponentChannels = 32;
bool component_rows_take(int64_t R, int64_t dim_in, int64_t dim_out, bool sequential) {
    if (dim_out < 64) return false;
    if (sequential) return R >= kComponentRowsF32;
    return dim_in > 8 && R >= (dim_in >= kComponentChannels ? kComponentRows : kComponentRowsF32);
}

std::tuple<at::Tensor, OptTensor> linear_fwd(int64_t inds, const at::Tensor& W, const at::Tensor& x, const OptTensor& bias,
                                             int act, const OptTensor& out, bool accumulate, int x_layout, int y_layout,
                                             const OptTensor& row_bound, double mul, double add, int64_t rows_per,
                                             bool want_rowmax, const OptTensor& x2_given, const OptTensor& x2max_given,
                                             bool sequential) {
    TORCH_CHECK(W.is_cuda(), "W must be a CUDA tensor");
    check_input(x, "x");
    TORCH_CHECK(W.scalar_type() == at::kFloat, "W must be float32");
    TORCH_CHECK(W.dim() == 2, "expected W to be a matrix (2 dims)");
    TORCH_CHECK(inds >= 0 && inds <= 2,
                "tensor_linear currently only supports a number of indices up to 2. go edit the code to add more (easy with "
                "copy/paste).");
    const int64_t dim_out = W.size(0), dim_in = W.size(1);
    const int T = inds == 0 ? 1 : inds == 1 ? 3 : 9;
    int64_t batch_dims;
    if (x_layout == 0) {
        batch_dims = x.dim() - (1 + inds);
        TORCH_CHECK(batch_dims >= 0, "x has too few dims");
        TORCH_CHECK(x.size(batch_dims) == dim_in, "channel dim size mismatch for x");
        for (int64_t i = batch_dims + 1; i <= batch_dims + inds; i++)
            TORCH_CHECK(x.size(i) == 3, "expected tensor index dim to be 3d for input x");
    } else {
        batch_dims = x.dim() - 2;
        TORCH_CHECK(batch_dims >= 0 && x.size(-1) == dim_in && x.size(-2) == T,
                    "component-major x must have shape (..., 3^inds, dim_in)");
    }
    std::vector<int64_t> y_shape(x.sizes().begin(), x.sizes().begin() + batch_dims);
    int64_t rows = 1;
    for (int64_t d : y_shape) rows *= d;
    if (y_layout == 0) {
        y_shape.push_back(dim_out);
        for (int64_t k = 0; k < inds; k++) y_shape.push_back(3);
    } else {
        y_shape.push_back(T);
        y_shape.push_back(dim_out);
    }
    if (bias.has_value()) {
        check_input(*bias, "bias");
        TORCH_CHECK(bias->numel() == dim_out, "bias size mismatch");
    }
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    at::Tensor y;
    if (out.has_value()) {
        check_input(*out, "out");
        TORCH_CHECK(out->sizes() == at::IntArrayRef(y_shape), "out has wrong shape");
        y = *out;
    } else {
        y = floats(x, y_shape);
    }
    const int mode = mg_get_linear_mode();
    const bool plain_rows = inds == 0 || x_layout == 1;
    const int64_t R = rows * T;
    const int out_comps = inds == 0 || y_layout == 1 ? 1 : T;
    at::Tensor ymax;
    const bool emit = want_rowmax && out_comps == 1 && !accumulate;
    auto rowmax_buffer = [&](int64_t k) {
        if (emit) ymax = floats(x, {R, rowmax_parts(R, k, dim_out, sequential)});
        return emit ? &ymax : nullptr;
    };
    const int64_t k_pad = (dim_in + 31) / 32 * 32;
    if (mode == kModeF16x2 && inds > 0 && x_layout == 0 && component_rows_take(R, dim_in, dim_out, sequential) &&
        !row_bound.has_value() &&
        (y_layout == 1 || !(want_rowmax || accumulate || bias.has_value() || act != kActNone))) {
        // (row, chan, comp) -> (row, comp, chan) rows, then the plain-row matrix path: its component-major output is
        // written at the full store rate, and with the reference's output layout its component epilogue still beats the
        // generic kernel (61 against 104 us for 16384 x 128 x 3 -> 384)
        at::Tensor x2, x2max;
        if (x2_given.has_value() && x2_given->dim() == 2 && x2_given->size(0) == R && x2_given->size(1) == k_pad) {
            x2 = *x2_given;
            x2max = *x2max_given;
        } else if (k_pad <= 256 && power_of_two(k_pad)) {
            std::tie(x2, x2max) = components_to_rows(x, rows, dim_in, T, k_pad);
        } else {
            at::Tensor xt = x.reshape({rows, dim_in, T}).transpose(1, 2);
            xt = k_pad != dim_in ? at::constant_pad_nd(xt, {0, k_pad - dim_in}) : xt.contiguous();
            x2 = xt.reshape({R, k_pad});
            x2max = row_absmax(x2);
        }
        run_f16x2(W, k_pad, fp(x2), R, Bound{x2max}, bias, act, accumulate, out_comps, y, rowmax_buffer(k_pad), sequential);
    } else if (plain_rows && mode == kModeF16x2 && f16x2_takes(R, dim_in, dim_out, x) && (!sequential || R >= 256)) {
        Bound b;
        if (row_bound.has_value()) {
            b = Bound{row_bound, (float)mul, (float)add, rows_per};
            TORCH_CHECK(row_bound->dim() == 2 && (row_bound->size(0) * rows_per == R || row_bound->size(0) == 1),
                        "row_bound must be (rows / rows_per_bound, parts)");
        } else {
            // A pass of its own.  On the way it would be one launch less (256 x 64 -> 64: 3.9 us of the GPU and 5.9 of the host, 6.3 and
            // 8.7 with the pass).  But the binding's fp32 linear, which promises less host time than this operator, is a kernel of
            // 10.4 us there: 4.4 us a call while launches may queue up, 5.6 in processes where they wait for the GPU before that,
            // where this operator then takes 5.3.  Chains and the linears of rows inside the layers find theirs on the way.
            b = Bound{row_absmax(x.reshape({R, dim_in}))};
        }
        run_f16x2(W, dim_in, fp(x), R, b, bias, act, accumulate, out_comps, y, rowmax_buffer(dim_in), sequential);
    } else if (mode == kModeBf16x3 && plain_rows && dim_in % 32 == 0 && dim_in >= 64 && dim_out >= 64 && R >= 1024 &&
               aligned16(x)) {
        check(mg_tensor_linear_packed(packed_bf16x3(W).data_ptr(), fp(x), R, (int)dim_in, (int)dim_out, fp(bias), act,
                                      accumulate, out_comps, fp(y), stream_of(x)));
    } else {
        check(mg_tensor_linear_layout((int)inds, fp(W), W.stride(0), W.stride(1), fp(x), rows, (int)dim_in, (int)dim_out,
                                      fp(bias), act, accumulate, x_layout, y_layout, fp(y), stream_of(x)));
    }
    return {y, ymax.defined() ? OptTensor(ymax) : OptTensor()};
}

// Weight gradients with one dimension of at most 16 from where the split-fp16 products take them (below, fp32 products in the order
// of the rows): fp32, the wide operand read once, at half their time or less (figures at the kernel).
bool narrow_wgrad_takes(int64_t inds, int64_t rows, const at::Tensor& dy, const at::Tensor& x, int64_t dim_in, int64_t dim_out) {
    return mg_get_linear_mode() == kModeF16x2 && rows * (inds == 0 ? 1 : inds == 1 ? 3 : 9) >= 4096 &&
           mg_tensor_linear_wgrad_narrow_supported((int)inds, rows, (int)dim_in, (int)dim_out) && aligned16(dim_in < dim_out ? dy : x);
}
void narrow_wgrad(int64_t inds, int64_t rows, const at::Tensor& dy, const at::Tensor& x, int64_t dim_in, int64_t dim_out, at::Tensor& dW,
                  float* db = nullptr) {
    size_t n = 0;
    check(mg_tensor_linear_wgrad_narrow_workspace_bytes(rows, (int)dim_in, (int)dim_out, &n));
    at::Tensor ws = bytes_like(x, n);
    check(mg_tensor_linear_wgrad_narrow((int)inds, fp(dy), fp(x), rows, (int)dim_in, (int)dim_out, ws.data_ptr(), fp(dW), db,
                                        stream_of(x)));
}

// dW (and with want_bias db): see ops.tensor_linear_wgrad
std::tuple<at::Tensor, OptTensor> linear_wgrad(int64_t inds, const at::Tensor& dy, const at::Tensor& x,
                                               const OptTensor& dy_bound, const OptTensor& x_bound, bool want_bias) {
    check_input(dy, "dy");
    check_input(x, "x");
    TORCH_CHECK(!want_bias || inds == 0, "the bias gradient is defined for plain rows only");
    const int64_t batch_dims = x.dim() - (1 + inds);
    const int64_t dim_in = x.size(batch_dims), dim_out = dy.size(batch_dims);
    int64_t rows = 1;
    for (int64_t i = 0; i < batch_dims; i++) rows *= x.size(i);
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    const int T = inds == 0 ? 1 : inds == 1 ? 3 : 9;
    const int mode = mg_get_linear_mode();
    at::Tensor dW = floats(x, {dim_out, dim_in});
    auto workspace = [&](int64_t n_rows, int64_t n_in, int64_t n_out) {
        size_t n = 0;
        check(mg_tensor_linear_wgrad_workspace_bytes(n_rows, (int)n_in, (int)n_out, &n));
        return bytes_like(x, n);
    };
    OptTensor db;
    if (narrow_wgrad_takes(inds, rows, dy, x, dim_in, dim_out)) {
        at::Tensor bias_grad;
        if (want_bias) bias_grad = floats(x, {dim_out});
        narrow_wgrad(inds, rows, dy, x, dim_in, dim_out, dW, want_bias ? fp(bias_grad) : nullptr);
        if (want_bias) db = bias_grad;
    } else if (inds == 0 && mode == kModeF16x2 && aligned16(x) && aligned16(dy) &&
        mg_tensor_linear_wgrad_f16x2_supported(rows, (int)dim_in, (int)dim_out)) {
        if (dy_bound.has_value()) check_input(*dy_bound, "dy_bound");
        if (x_bound.has_value()) check_input(*x_bound, "x_bound");
        at::Tensor bias_grad;
        if (want_bias) bias_grad = floats(x, {dim_out});
        at::Tensor ws = workspace(rows, dim_in, dim_out);
        check(mg_tensor_linear_wgrad_f16x2(fp(dy), fp(x), fp(dy_bound), dy_bound.has_value() ? dy_bound->numel() : 0, fp(x_bound),
                                           x_bound.has_value() ? x_bound->numel() : 0, rows, (int)dim_in, (int)dim_out,
                                           ws.data_ptr(), fp(dW), want_bias ? fp(bias_grad) : nullptr, stream_of(x)));
        if (want_bias) db = bias_grad;
    } else if (inds > 0 && mode == kModeF16x2 && rows * T >= 4096 && std::max(dim_in, dim_out) <= 256) {
        // (row, chan, comp) -> one plain row per (row, comp), channels zero-padded to a power of two: the sum over rows
        // and components is then the plain-row weight gradient, on the matrix cores; the transposition also yields the
        // row maxima the kernel scales by
        auto pad_of = [](int64_t d) {
            int64_t p = 32;
            while (p < d) p *= 2;
            return p;
        };
        const int64_t o_pad = pad_of(dim_out), i_pad = pad_of(dim_in);
        auto [dy2, dy2max] = components_to_rows(dy, rows, dim_out, T, o_pad);
        auto [x2, x2max] = components_to_rows(x, rows, dim_in, T, i_pad);
        at::Tensor ws = workspace(rows * T, i_pad, o_pad);
        at::Tensor padded = o_pad == dim_out && i_pad == dim_in ? dW : floats(x, {o_pad, i_pad});
        check(mg_tensor_linear_wgrad_f16x2(fp(dy2), fp(x2), fp(dy2max), rows * T, fp(x2max), rows * T, rows * T, (int)i_pad,
                                           (int)o_pad, ws.data_ptr(), fp(padded), nullptr, stream_of(x)));
        if (o_pad != dim_out || i_pad != dim_in) dW = padded.slice(0, 0, dim_out).slice(1, 0, dim_in).contiguous();
    } else {
        at::Tensor ws = workspace(rows, dim_in, dim_out);
        check(mg_tensor_linear_wgrad((int)inds, fp(dy), fp(x), rows, (int)dim_in, (int)dim_out, ws.data_ptr(), fp(dW),
                                     stream_of(x)));
        if (want_bias) db = dy.reshape({-1, dim_out}).sum(0);
    }
    return {dW, db};
}

at::Tensor silu_order(const at::Tensor& z, int order, const OptTensor& mul) {
    check_input(z, "z");
    if (mul.has_value()) {
        check_input(*mul, "mul");
        TORCH_CHECK(mul->sizes() == z.sizes(), "mul must have the shape of z");
    }
    TORCH_CHECK(order >= 0 && order <= 4, "silu_order: order must be in 0..4");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(z.device());
    at::Tensor out = floats(z, z.sizes());
    check(mg_silu_order(fp(z), fp(mul), z.numel(), order, fp(out), stream_of(z)));
    return out;
}

// ------------------------------------------------------------------ MLPs (inference)
using Tensors = std::vector<at::Tensor>;

const std::vector<int> kSiluMlp{kActSilu, kActSilu, kActNone};

bool aligned_all(const Tensors& t) { return std::all_of(t.begin(), t.end(), [](const at::Tensor& v) { return aligned16(v); }); }

// Whether the three layers of an MLP on x (rows, k) go through one kernel (k: W[0]'s columns after zero padding).
// A workgroup reads all three weights whatever the number of rows, about 30 us of a kernel at 128 -> 512 -> 512 -> 512 and 10 us
// at 128 -> 128: for wide layers of few rows the three launches that split the reduction of each over the chip are faster, as long
// as their workgroups of 32 rows x 64 columns are one round of it (us, one kernel / three launches: 128 -> 512 29.9 / 18.9 at 337
// rows, 29.3 / 25.2 at 1024, 29.3 / 31.9 at 1100, 33.7 / 61.8 at 4096, 69 / 98 at 16 336; 256 -> 448 27.9 / 23.6 at 1100, 27.9 / 32.2 at
// 1280; 256 -> 384 22.2 / 21.3 at 1100, 22.3 / 31.0 at 1408; 512 -> 384 25.6 / 23.4 and 25.5 / 33.6).  From 288 to 352 columns
// neither is ahead before 1024 rows, and one kernel is beyond (256 -> 320 19.2 / 19.0 at 1024, 19.2 / 20.3 at 1280).  Narrower
// layers take one kernel (64 -> 256 12.6 / 14.2 at 64 rows, 26 / 53 at 16 384; 128 -> 128 9.9 / 14.2 at 64).  Distance from float64
// at 128 -> 512: 2.3e-7 against 2.2..2.5e-7 with split reductions, 2.75e-7 against 4.1e-7 at 16 336 rows.
constexpr int64_t kMlpWide = 256;
bool mlp_in_three(int64_t rows, int64_t dim) {
    if (dim >= 384) return (rows + 31) / 32 * ((dim + 63) / 64) <= 256;
    return dim > kMlpWide && rows < 1024;
}
bool packs_f16x2(const at::Tensor& W) { return W.size(1) % 32 == 0 && W.size(1) >= 64 && W.size(0) >= 8; }

bool mlp_takes_rows(int64_t rows, int64_t k, int64_t dim) {
    return mg_get_linear_mode() == kModeF16x2 && rows >= 1 && !mlp_in_three(rows, dim) && k >= 64 && dim >= 64 &&
           mg_mlp_f16x2_supported((int)k, (int)dim);
}
bool mlp_takes(int64_t rows, int64_t k, const Tensors& W, const at::Tensor& x) {
    const int64_t dim = W[0].size(0);
    if (!mlp_takes_rows(rows, k, dim)) return false;
    for (size_t l = 0; l < 3; l++)
        if (W[l].size(0) != dim || (l > 0 && W[l].size(1) != dim)) return false;
    return aligned16(x);
}

// planes: kept alive by the caller until the launch is queued
mg_mlp_f16x2 mlp_args(const at::Tensor& x, const Tensors& W, const Tensors& b, at::Tensor& y, Tensors& planes) {
    mg_mlp_f16x2 a{};
    for (int l = 0; l < 3; l++) {
        planes.push_back(packed_f16x2(W[l], l == 0 ? x.size(1) : W[l].size(1)));
        a.packed_W[l] = planes.back().data_ptr();
        a.bias[l] = fp(b[l]);
    }
    a.x = fp(x);
    a.rows = x.size(0);
    a.dim_in = (int)x.size(1);
    a.dim = (int)W[0].size(0);
    a.y = fp(y);
    return a;
}
at::Tensor mlp_fused(const at::Tensor& x, const Tensors& W, const Tensors& b) {
    at::Tensor y = floats(x, {x.size(0), W[2].size(0)});
    Tensors planes;
    const mg_mlp_f16x2 a = mlp_args(x, W, b, y, planes);
    check(mg_mlp_f16x2_forward(&a, stream_of(x)));
    return y;
}

// a chain of linears with fused bias and activation; the row bounds the split-fp16 layers scale by travel as
// mul * base + add through the layers' norms, so that only the first layer ever looks at the data for them
at::Tensor chain(at::Tensor h, const Tensors& W, const Tensors& b, const std::vector<int>& act, Bound bound) {
    if (act == kSiluMlp && mlp_takes(h.size(0), h.size(1), W, h) && aligned_all(b)) return mlp_fused(h, W, b);
    for (size_t k = 0; k < W.size(); k++) {
        const int64_t rows = h.size(0), dim_in = W[k].size(1), dim_out = W[k].size(0);
        at::Tensor y = floats(h, {rows, dim_out});
        const OptTensor bias(b[k]);
        if (rows == 0) {
            h = y;
            continue;
        }
        if (mg_get_linear_mode() == kModeF16x2 && f16x2_takes(rows, dim_in, dim_out, h)) {
            if (!bound.base.has_value()) bound = Bound{};
            bound.base = run_f16x2(W[k], dim_in, fp(h), rows, bound, bias, act[k], false, 1, y, nullptr, false);
        } else {
            y = std::get<0>(linear_fwd(0, W[k], h, bias, act[k], OptTensor(y), false, 0, 0, OptTensor(), 1, 0, 1, false,
                                       OptTensor(), OptTensor(), false));
        }
        if (bound.base.has_value() && k + 1 < W.size()) bound = through(bound, norms_of(W[k], bias));
        h = y;
    }
    return h;
}

void check_chain(const at::Tensor& x, const Tensors& W, const Tensors& b, const std::vector<int>& act) {
    check_input(x, "x");
    TORCH_CHECK(x.dim() == 2 && W.size() == b.size() && W.size() == act.size() && !W.empty(), "linear_chain: bad arguments");
    int64_t dim = x.size(1);
    for (size_t k = 0; k < W.size(); k++) {
        TORCH_CHECK(W[k].is_cuda() && W[k].scalar_type() == at::kFloat && W[k].dim() == 2 && W[k].size(1) == dim,
                    "linear_chain: weights must be float32 CUDA matrices that follow each other");
        check_input(b[k], "bias");
        TORCH_CHECK(b[k].numel() == W[k].size(0), "bias size mismatch");
        dim = W[k].size(0);
    }
}

at::Tensor linear_chain(const at::Tensor& x, const Tensors& W, const Tensors& b, const std::vector<int>& act,
                        const OptTensor& bound, double mul, double add) {
    check_chain(x, W, b, act);
    if (bound.has_value()) check_bound(*bound, x.size(0), 1);
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    return chain(x, W, b, act, Bound{bound, (float)mul, (float)add});
}

// ------------------------------------------------------------------ PaiNN layers (inference)
// Update.forward: x_a (batch, nodes, n), x_v (batch, nodes, n, 3); W_lrv (3n, n) the stacked l, r, v maps
std::tuple<at::Tensor, at::Tensor> painn_update(const at::Tensor& x_a, const at::Tensor& x_v, const at::Tensor& W_lrv,
                                                const Tensors& W, const Tensors& b, int groups, const at::Tensor& gamma,
                                                const at::Tensor& beta, double eps, bool residual) {
    check_input(x_a, "x_a");
    check_input(x_v, "x_v");
    TORCH_CHECK(x_a.dim() == 3 && x_v.dim() == 4 && x_v.size(3) == 3 && x_v.size(2) == x_a.size(2) &&
                    x_v.size(0) == x_a.size(0) && x_v.size(1) == x_a.size(1),
                "x_a must have shape (batch, nodes, n) and x_v (batch, nodes, n, 3)");
    const int64_t B = x_a.size(0), N = x_a.size(1), n = x_a.size(2), rows = B * N;
    TORCH_CHECK(W_lrv.size(0) == 3 * n && W_lrv.size(1) == n, "W_lrv must have shape (3n, n)");
    check_input(gamma, "gamma");
    check_input(beta, "beta");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x_a.device());
    at::Tensor ip = floats(x_a, {rows, n}), cat = floats(x_a, {rows, 2 * n}), lrv, cat_max;
    if (n <= 256) cat_max = floats(x_a, {rows, 1});
    const mg_stream_t st = stream_of(x_a);
    // Where the maps, in fp16 pieces, are faster than their linear and what follows it (figures at the kernel).  Of up to 128 channels
    // that is from one node on, where that linear would be fp32: 2.7 and 2.5e-7 of float64 at 128, 3.6 and 3.2e-7 with it
    const bool maps = mg_get_linear_mode() == kModeF16x2 && rows >= (n <= 128 ? 1 : n <= 224 ? 1280 : 2304) && packs_f16x2(W_lrv) &&
                      mg_painn_update_maps_supported((int)n) && aligned16(x_v) && aligned16(x_a);
    if (maps) {
        lrv = floats(x_a, {rows, 3, n});
        const at::Tensor planes = packed_f16x2(W_lrv, n);
        check(mg_painn_update_maps(fp(x_v), fp(x_a), rows, (int)n, planes.data_ptr(), fp(ip), fp(cat), fp(cat_max), fp(lrv), st));
    } else {
        // component-major (rows, 3, 3n): the GEMM stores whole rows, the two kernels below read with unit stride
        lrv = std::get<0>(linear_fwd(1, W_lrv, x_v.reshape({rows, n, 3}), OptTensor(), kActNone, OptTensor(), false, 0, 1, OptTensor(),
                                     1, 0, 1, false, OptTensor(), OptTensor(), false));
        check(mg_painn_update_pre(fp(lrv), 1, fp(x_a), rows, (int)n, fp(ip), fp(cat), n <= 256 ? fp(cat_max) : nullptr, st));
    }
    check_chain(cat, W, b, kSiluMlp);
    at::Tensor y = chain(cat, W, b, kSiluMlp, Bound{n <= 256 ? OptTensor(cat_max) : OptTensor()});          // (rows, 3n)
    at::Tensor out_a = floats(x_a, x_a.sizes()), out_v = floats(x_v, x_v.sizes());
    size_t scratch_bytes = 0;
    check(mg_group_norm_scratch_bytes((int)B, groups, &scratch_bytes));
    at::Tensor scratch = bytes_like(x_a, std::max<size_t>(scratch_bytes, 8));
    check(mg_painn_update_post(fp(lrv), maps ? 2 : 1, fp(ip), fp(y), (int)B, (int)N, (int)n, groups, (float)eps, fp(gamma), fp(beta),
                               residual ? fp(x_a) : nullptr, residual ? fp(x_v) : nullptr, scratch.data_ptr(), fp(out_a), fp(out_v), st));
    return {out_a, out_v};
}

// TensGroupNorm.forward of x (batch, nodes, chan, ..) and the sums that its adjoint reads again
std::tuple<at::Tensor, at::Tensor> tens_norm_fwd(const at::Tensor& x, const at::Tensor& gamma, int groups, double eps) {
    check_input(x, "x");
    check_input(gamma, "gamma");
    TORCH_CHECK(x.dim() >= 3 && x.dim() <= 5 && gamma.numel() == x.size(2), "x must have shape (batch, nodes, chan, (3,)^inds)");
    const int64_t B = x.size(0), N = x.size(1), C = x.size(2), T = C * N * B ? x.numel() / (B * N * C) : 1;
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    size_t n = 0;
    check(mg_group_norm_scratch_bytes((int)B, groups, &n));
    at::Tensor scratch = bytes_like(x, std::max<size_t>(n, 8)), y = floats(x, x.sizes());
    check(mg_group_norm(0, fp(x), C, nullptr, 0, (int)B, (int)N, (int)C, groups, (int)T, (float)eps, fp(gamma), nullptr, nullptr, 0, nullptr,
                        scratch.data_ptr(), fp(y), stream_of(x)));
    return {y, scratch};
}
// TensGroupNorm.forward of several x (batch, nodes, chan, ..) over the same nodes, with res[k] added: two launches
Tensors tens_norms(const Tensors& x, const Tensors& gamma, const std::vector<OptTensor>& res, const std::vector<int64_t>& groups,
                   const std::vector<double>& eps) {
    const size_t count = x.size();
    TORCH_CHECK(count >= 1 && count <= MG_TENS_NORMS && gamma.size() == count && res.size() == count && groups.size() == count && eps.size() == count,
                "tens_norms: up to ", MG_TENS_NORMS, " norms");
    const int64_t B = x[0].size(0), N = x[0].dim() >= 3 ? x[0].size(1) : -1;
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x[0].device());
    mg_tens_norm norms[MG_TENS_NORMS];
    Tensors out;
    size_t bytes = 0;
    for (size_t k = 0; k < count; k++) {
        check_input(x[k], "x");
        check_input(gamma[k], "gamma");
        TORCH_CHECK(x[k].dim() >= 3 && x[k].dim() <= 5 && x[k].size(0) == B && x[k].size(1) == N && gamma[k].numel() == x[k].size(2),
                    "x must have shape (batch, nodes, chan, (3,)^inds)");
        if (res[k].has_value()) {
            check_input(*res[k], "res");
            TORCH_CHECK(res[k]->sizes() == x[k].sizes(), "res has wrong shape");
        }
        out.push_back(floats(x[k], x[k].sizes()));
        int64_t comps = 1;
        for (int64_t d = 3; d < x[k].dim(); d++) comps *= x[k].size(d);
        norms[k] = {fp(x[k]), fp(gamma[k]), res[k].has_value() ? fp(*res[k]) : nullptr, fp(out[k]), (int)x[k].size(2), (int)comps,
                    (int)groups[k], (float)eps[k]};
        size_t n = 0;
        check(mg_group_norm_scratch_bytes((int)B, (int)groups[k], &n));
        bytes += n;
    }
    at::Tensor scratch = bytes_like(x[0], std::max<size_t>(bytes, 8));
    check(mg_tens_group_norms(norms, (int)count, (int)B, (int)N, scratch.data_ptr(), stream_of(x[0])));
    return out;
}
std::tuple<at::Tensor, at::Tensor> tens_norm_bwd(const at::Tensor& dy, const at::Tensor& x, const at::Tensor& gamma, const at::Tensor& scratch,
                                                 int groups, double eps) {
    check_input(dy, "dy");
    check_input(x, "x");
    check_input(gamma, "gamma");
    TORCH_CHECK(x.dim() >= 3 && x.dim() <= 5 && dy.sizes() == x.sizes() && gamma.numel() == x.size(2) && x.numel() > 0, "tens_norm_bwd: sizes");
    const int64_t B = x.size(0), N = x.size(1), C = x.size(2), T = x.numel() / (B * N * C);
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    size_t n = 0, kept = 0;
    check(mg_tensor_norm_grad_workspace_bytes_of((int)B, (int)N, (int)C, groups, (int)T, &n));
    check(mg_group_norm_scratch_bytes((int)B, groups, &kept));
    TORCH_CHECK(scratch.is_cuda() && scratch.is_contiguous() && (size_t)scratch.nbytes() >= kept, "tens_norm_bwd: the sums of the forward pass");
    at::Tensor ws = bytes_like(x, n), dx = floats(x, x.sizes()), dgamma = floats(x, gamma.sizes());
    check(mg_tensor_norm_grad(fp(dy), fp(x), (int)B, (int)N, (int)C, groups, (int)T, (float)eps, fp(gamma), scratch.data_ptr(), ws.data_ptr(),
                              fp(dx), fp(dgamma), stream_of(x)));
    return {dx, dgamma};
}

struct MessageArgs {
    const at::Tensor &row_ptr, &dst, &r_ij, &x_a, &x_v;
    int64_t B, N, n, rows, E;
};
MessageArgs message_args(const at::Tensor& row_ptr, const at::Tensor& dst, const at::Tensor& r_ij, const at::Tensor& x_a,
                         const at::Tensor& x_v) {
    check_input(row_ptr, "row_ptr", at::kInt);
    check_input(dst, "dst", at::kInt);
    check_input(r_ij, "r_ij");
    check_input(x_a, "x_a");
    check_input(x_v, "x_v");
    TORCH_CHECK(x_a.dim() == 3 && x_v.dim() == 4 && x_v.size(3) == 3 && x_v.size(2) == x_a.size(2) &&
                    x_v.size(0) == x_a.size(0) && x_v.size(1) == x_a.size(1),
                "x_a must have shape (batch, nodes, n) and x_v (batch, nodes, n, 3)");
    MessageArgs m{row_ptr, dst, r_ij, x_a, x_v, x_a.size(0), x_a.size(1), x_a.size(2), x_a.size(0) * x_a.size(1), dst.numel()};
    TORCH_CHECK(row_ptr.numel() == m.rows + 1, "row_ptr must have nodes+1 entries");
    TORCH_CHECK(r_ij.dim() == 2 && r_ij.size(0) == m.E && r_ij.size(1) == 3, "r_ij must have shape (edges, 3)");
    return m;
}

// The filter MLP on the encodings enc (rows, k) of a grid, all at most 1 in magnitude; where k exceeds the first layer's
// input the encodings end in zero columns and the weight is padded likewise (a reduction the matrix path takes).
at::Tensor filter_grid(const at::Tensor& enc, const at::Tensor& unit, const Tensors& W, const Tensors& b) {
    check_input(enc, "enc");
    check_input(unit, "unit");
    const int64_t k = enc.size(1), rows = enc.size(0);
    if (k == W[0].size(1)) {
        check_chain(enc, W, b, kSiluMlp);
        return chain(enc, W, b, kSiluMlp, Bound{OptTensor(unit)});
    }
    TORCH_CHECK(k > W[0].size(1) && k % 32 == 0 && mg_get_linear_mode() == kModeF16x2 && aligned16(enc),
                "filter_grid: encodings of a wrong width");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(enc.device());
    if (mlp_takes(rows, k, W, enc) && aligned_all(b)) return mlp_fused(enc, W, b);
    at::Tensor h = floats(enc, {rows, W[0].size(0)});
    const OptTensor b0(b[0]);
    run_f16x2(W[0], k, fp(enc), rows, Bound{OptTensor(unit)}, b0, kActSilu, false, 1, h, nullptr, false);
    const auto [l1, bmax] = norms_of(W[0], b0);
    check_chain(h, {W[1], W[2]}, {b[1], b[2]}, {kActSilu, kActNone});
    return chain(h, {W[1], W[2]}, {b[1], b[2]}, {kActSilu, kActNone}, Bound{OptTensor(unit), l1, bmax});
}

// Several of them, in one launch where their layers have one width that the MLP kernel takes for as many rows as they have together
Tensors filter_grids(const Tensors& enc, const Tensors& unit, const std::vector<Tensors>& W, const std::vector<Tensors>& b) {
    const size_t jobs = enc.size();
    TORCH_CHECK(unit.size() == jobs && W.size() == jobs && b.size() == jobs, "filter_grids: as many encodings, weights and biases");
    int64_t rows = 0;
    bool together = jobs > 1;
    for (size_t k = 0; k < jobs; k++) {
        TORCH_CHECK(W[k].size() == 3 && b[k].size() == 3, "filter_grids: three layers expected");
        if (enc[k].dim() == 2) rows += enc[k].size(0);
    }
    for (size_t k = 0; k < jobs && together; k++)
        together = enc[k].dim() == 2 && enc[k].size(0) > 0 && enc[k].size(1) >= W[k][0].size(1) && enc[k].device() == enc[0].device() &&
                   W[k][0].size(0) == W[0][0].size(0) && mlp_takes(rows, enc[k].size(1), W[k], enc[k]) && aligned_all(b[k]);
    Tensors y;
    if (!together) {
        for (size_t k = 0; k < jobs; k++) y.push_back(filter_grid(enc[k], unit[k], W[k], b[k]));
        return y;
    }
    c10::hip::HIPGuardMasqueradingAsCUDA guard(enc[0].device());
    Tensors planes;
    std::vector<mg_mlp_f16x2> args;
    for (size_t k = 0; k < jobs; k++) {
        check_input(enc[k], "enc");
        for (int l = 0; l < 3; l++) {
            TORCH_CHECK(W[k][l].is_cuda() && W[k][l].scalar_type() == at::kFloat && W[k][l].dim() == 2, "filter_grids: weights must be float32 CUDA matrices");
            check_input(b[k][l], "bias");
            TORCH_CHECK(b[k][l].numel() == W[k][l].size(0), "bias size mismatch");
        }
        y.push_back(floats(enc[k], {enc[k].size(0), W[k][2].size(0)}));
        args.push_back(mlp_args(enc[k], W[k], b[k], y[k], planes));
    }
    std::vector<const mg_mlp_f16x2*> at;
    for (const mg_mlp_f16x2& a : args) at.push_back(&a);
    check(mg_mlp_f16x2_forward_many(at.data(), (int)jobs, stream_of(enc[0])));
    return y;
}

// Message.forward with the filter interpolated from its grid, which is evaluated here: enc (rows, k) the grid's
// encodings, k the first layer's reduction dimension after zero padding.  sliced: the grid in LDS, the last layer of
// mlp_actv given with its rows slice by slice.
std::tuple<at::Tensor, at::Tensor> painn_message_grid(const at::Tensor& row_ptr, const at::Tensor& dst, const at::Tensor& r_ij,
                                                      const OptTensor& order, const at::Tensor& x_a, const at::Tensor& x_v,
                                                      const Tensors& W_actv, const Tensors& b_actv, const OptTensor& enc,
                                                      const OptTensor& unit, const Tensors& W_dist, const Tensors& b_dist,
                                                      const OptTensor& table_given, double period, double epsilon, bool sliced,
                                                      bool residual) {
    const MessageArgs m = message_args(row_ptr, dst, r_ij, x_a, x_v);
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x_a.device());
    const at::Tensor flat_a = x_a.reshape({m.rows, m.n});
    check_chain(flat_a, W_actv, b_actv, kSiluMlp);
    const at::Tensor actv = chain(flat_a, W_actv, b_actv, kSiluMlp, Bound{});
    TORCH_CHECK(actv.size(1) == 4 * m.n, "actv must have shape (nodes, 4n)");
    at::Tensor table;
    if (table_given.has_value()) {
        check_input(*table_given, "table");
        table = *table_given;
    } else {
        table = filter_grid(*enc, *unit, W_dist, b_dist);
    }
    TORCH_CHECK(table.dim() == 2 && table.size(1) == 4 * m.n, "table must have shape (rows, 4n)");
    if (order.has_value()) {
        check_input(*order, "node_order", at::kInt);
        TORCH_CHECK(order->numel() == m.rows, "node_order must have one entry per node");
    }
    const int* ord = order.has_value() ? order->data_ptr<int>() : nullptr;
    at::Tensor out_a = floats(x_a, x_a.sizes()), out_v = floats(x_v, x_v.sizes());
    const mg_stream_t st = stream_of(x_a);
    const float *res_a = residual ? fp(x_a) : nullptr, *res_v = residual ? fp(x_v) : nullptr;
    if (sliced) {
        at::Tensor rec = floats(x_a, {m.E, 8});
        check(mg_painn_edge_records(fp(r_ij), m.E, (int)table.size(0), (float)period, (float)epsilon, fp(rec), st));
        check(mg_painn_table_message_sliced(row_ptr.data_ptr<int>(), dst.data_ptr<int>(), ord, m.rows, m.E, fp(rec), fp(table),
                                            (int)table.size(0), fp(actv), fp(x_v), (int)m.n, res_a, res_v, fp(out_a), fp(out_v),
                                            st));
    } else {
        check(mg_painn_table_message(row_ptr.data_ptr<int>(), dst.data_ptr<int>(), ord, m.rows, m.E, fp(r_ij), fp(table),
                                     (int)table.size(0), (float)period, fp(actv), fp(x_v), (int)m.n, (float)epsilon, res_a,
                                     res_v, fp(out_a), fp(out_v), st));
    }
    return {out_a, out_v};
}

// Message.forward with the filter MLP on every edge and the filter stored, unless the caller has it as `filters` (few edges: the kernels that fold its layers into
// the edge kernel are made for tiles of 256 edges)
std::tuple<at::Tensor, at::Tensor> painn_message_edges(const at::Tensor& row_ptr, const at::Tensor& dst, const at::Tensor& r_ij,
                                                       const at::Tensor& x_a, const at::Tensor& x_v, const Tensors& W_actv,
                                                       const Tensors& b_actv, const at::Tensor& unit, const Tensors& W_dist,
                                                       const Tensors& b_dist, double rmax, double epsilon, bool residual,
                                                       const OptTensor& filters) {
    const MessageArgs m = message_args(row_ptr, dst, r_ij, x_a, x_v);
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x_a.device());
    const at::Tensor flat_a = x_a.reshape({m.rows, m.n});
    check_chain(flat_a, W_actv, b_actv, kSiluMlp);
    const at::Tensor actv = chain(flat_a, W_actv, b_actv, kSiluMlp, Bound{});
    TORCH_CHECK(actv.size(1) == 4 * m.n, "weights must end in 4n rows");
    const mg_stream_t st = stream_of(x_a);
    at::Tensor filt;
    if (filters.has_value()) {
        check_input(*filters, "filters");
        TORCH_CHECK(filters->dim() == 2 && filters->size(0) == m.E && filters->size(1) == 4 * m.n, "filters must have shape (edges, 4n)");
        filt = *filters;
    }
    TORCH_CHECK(filt.defined() || (W_dist.size() == 3 && W_dist[2].size(0) == 4 * m.n), "weights must end in 4n rows");
    const int64_t n_rbf = filt.defined() ? 0 : W_dist[0].size(1), hidden = filt.defined() ? 0 : W_dist[0].size(0), g = hidden / 4;
    if (filt.defined()) {
    } else if (n_rbf <= 32 && hidden % 4 == 0 && g >= 1 && g <= 256 && 256 % g == 0) {
        at::Tensor h = floats(x_a, {m.E, hidden});
        check(mg_painn_radial_linear(fp(r_ij), m.E, (int)n_rbf, (float)rmax, fp(W_dist[0]), W_dist[0].stride(0),
                                     W_dist[0].stride(1), fp(b_dist[0]), (int)hidden, kActSilu, fp(h), st));
        const auto [l1, bmax] = norms_of(W_dist[0], OptTensor(b_dist[0]));
        filt = chain(h, {W_dist[1], W_dist[2]}, {b_dist[1], b_dist[2]}, {kActSilu, kActNone}, Bound{OptTensor(unit), l1, bmax});
    } else {
        at::Tensor enc = floats(x_a, {m.E, n_rbf});
        check(mg_painn_radial_encode(fp(r_ij), m.E, (int)n_rbf, (float)rmax, fp(enc), st));
        check_chain(enc, W_dist, b_dist, kSiluMlp);
        filt = chain(enc, W_dist, b_dist, kSiluMlp, Bound{OptTensor(unit)});
    }
    at::Tensor out_a = floats(x_a, x_a.sizes()), out_v = floats(x_v, x_v.sizes());
    check(mg_painn_message(row_ptr.data_ptr<int>(), dst.data_ptr<int>(), nullptr, m.rows, m.E, fp(r_ij), fp(filt), fp(actv),
                           fp(x_v), (int)m.n, (float)epsilon, residual ? fp(x_a) : nullptr, residual ? fp(x_v) : nullptr,
                           fp(out_a), fp(out_v), st));
    return {out_a, out_v};
}

// ------------------------------------------------------------------ PaiNN layers under differentiation
// A value and its forward-mode tangent travel as one array of 2 R rows (values first): one launch per linear map, weight
// gradient and activation for both.  The halves are handed out as two tensors on one storage, and taken back as one array
// where they still lie one behind the other.
at::Tensor on_storage(const at::Tensor& of, int64_t offset, at::IntArrayRef shape) {
    std::vector<int64_t> strides(shape.size());
    int64_t step = 1;
    for (size_t k = shape.size(); k-- > 0;) {
        strides[k] = step;
        step *= shape[k];
    }
    // (not a view: the halves are written once, before they are handed out, and have version counters of their own)
    return at::empty({0}, of.options().requires_grad(false)).set_(of.storage(), of.storage_offset() + offset, shape, strides);
}
OptTensor second_half(const at::Tensor& y, at::IntArrayRef shape, bool dual) {
    return dual ? OptTensor(on_storage(y, y.numel() / 2, shape)) : OptTensor();
}
at::Tensor stacked(const at::Tensor& p, const OptTensor& t, int64_t cols) {
    check_input(p, "x");
    const int64_t rows = cols ? p.numel() / cols : 0;
    if (!t.has_value()) return p.reshape({rows, cols});
    check_input(*t, "tangent of x");
    TORCH_CHECK(t->numel() == p.numel(), "a tangent must have the shape of its value");
    if (t->storage().data() == p.storage().data() && t->storage_offset() == p.storage_offset() + p.numel())
        return on_storage(p, 0, {2 * rows, cols});
    return at::cat({p.reshape({rows, cols}), t->reshape({rows, cols})});
}

// Packed planes of several weights that the next kernels read, those that are missing in one launch.  `passing`: weights that
// do not outlive this pass; their planes are returned and not kept.
std::vector<OptTensor> pack_ahead(const Tensors& weights, const Tensors& passing = {}) {
    std::vector<OptTensor> out(passing.size());
    if (mg_get_linear_mode() != kModeF16x2) return out;
    Tensors missing, planes;
    for (const at::Tensor& W : weights)
        if (packs_f16x2(W) && !cache<at::Tensor>().has(W, 2, W.size(1))) missing.push_back(W);
    const size_t kept = missing.size();
    for (const at::Tensor& W : passing)
        if (packs_f16x2(W)) missing.push_back(W);
    if (missing.size() < 2 && kept == missing.size()) return out;
    std::vector<mg_f16x2_weight> jobs;
    for (const at::Tensor& W : missing) {
        size_t bytes = 0;
        check(mg_linear_f16x2_packed_weight_bytes((int)W.size(1), (int)W.size(0), &bytes));
        planes.push_back(bytes_like(W, bytes));
        jobs.push_back({fp(W), (long)W.stride(0), (long)W.stride(1), (int)W.size(1), (int)W.size(0), (int)W.size(1),
                        planes.back().data_ptr()});
    }
    check(mg_linear_f16x2_pack_weights(jobs.data(), (int)jobs.size(), stream_of(missing[0])));
    for (size_t k = 0; k < kept; k++) {
        const at::Tensor p = planes[k];
        cache<at::Tensor>().get(missing[k], 2, missing[k].size(1), [&] { return p; });
    }
    for (size_t k = 0, at = kept; k < passing.size(); k++)
        if (packs_f16x2(passing[k])) out[k] = planes[at++];
    return out;
}

// sum_k W_k x_k for x = [x_1 | x_2 | ..] (R, G C), one plain row per (row, component) of tensors of T components: the arithmetic of
// tensor linears one by one (linear_fwd), each x_k with row maxima, and each weight with scales, of its own.  Also
// the row maxima (R, G) of |x_k| where they were needed.
std::tuple<at::Tensor, OptTensor> row_linears_fwd(const at::Tensor& x, const Tensors& W, int64_t T, bool sequential) {
    check_input(x, "x");
    TORCH_CHECK(!W.empty() && (T == 1 || T == 3 || T == 9) && x.dim() == 2, "row_linears: operands");
    const int64_t R = x.size(0), G = (int64_t)W.size(), O = W[0].size(0), C = W[0].size(1);
    for (const at::Tensor& w : W)
        TORCH_CHECK(w.is_cuda() && w.scalar_type() == at::kFloat && w.dim() == 2 && w.size(0) == O && w.size(1) == C && x.size(1) == G * C,
                    "row_linears: weights (dim_out, chan), x (rows, weights chan)");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    at::Tensor y = floats(x, {R, O});
    const bool split = mg_get_linear_mode() == kModeF16x2 && f16x2_takes(R, C, O, x) &&
                       (T == 1 ? !sequential || R >= 256 : component_rows_take(R, C, O, sequential));
    OptTensor x_max;
    if (split) {
        pack_ahead(W);
        x_max = row_absmax(x.view({R * G, C})).view({R, G});
    }
    std::vector<const float*> weights;
    for (const at::Tensor& w : W)
        if (w.stride(1) == 1 && w.stride(0) == W[0].stride(0) && w.stride(0) % 4 == 0 && aligned16(w)) weights.push_back(fp(w));
    if (!split && G <= 8 && C % 32 == 0 && aligned16(x) && (int64_t)weights.size() == G) {
        at::Tensor m = floats(x, {R, G});
        check(mg_tensor_linear_products(weights.data(), W[0].stride(0), (int)G, fp(x), R, (int)C, (int)O, fp(y), fp(m), stream_of(x)));
        return {y, m};
    }
    for (int64_t k = 0; k < G; k++) {
        if (split)
            run_f16x2(W[k], C, fp(x) + k * C, R, Bound{x_max}, OptTensor(), kActNone, k > 0, 1, y, nullptr, sequential, -1, OptTensor(),
                      G * C, k);
        else
            check(mg_tensor_linear_rows(fp(W[k]), W[k].stride(0), W[k].stride(1), fp(x) + k * C, G * C, R, (int)C, (int)O, k > 0, fp(y),
                                        stream_of(x)));
    }
    return {y, x_max};
}

// Its gradients for x and the weights, (dim_out, chan) each
std::tuple<OptTensor, Tensors> row_linears_bwd(const at::Tensor& dy, const at::Tensor& x, const Tensors& W, OptTensor x_max, int64_t T,
                                               bool want_x, bool want_W) {
    check_input(dy, "dy");
    check_input(x, "x");
    const int64_t R = x.size(0), G = (int64_t)W.size(), O = W[0].size(0), C = W[0].size(1);
    TORCH_CHECK(dy.dim() == 2 && dy.size(0) == R && dy.size(1) == O && x.size(1) == G * C, "row_linears: gradient sizes");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    const bool f16x2 = mg_get_linear_mode() == kModeF16x2;
    const bool split_x = f16x2 && f16x2_takes(R, O, G * C, dy) && (T == 1 || component_rows_take(R, O, C, false));
    const bool split_W = f16x2 && aligned16(x) && aligned16(dy) && (T == 1 || std::max(C, O) <= 256) &&
                         mg_tensor_linear_wgrad_f16x2_supported(R, (int)C, (int)O);
    const bool narrow = narrow_wgrad_takes(0, R, dy, x, G * C, O);
    OptTensor dx, dy_max;
    if ((want_x && split_x) || (want_W && split_W && !narrow)) dy_max = row_absmax(dy);
    if (want_x) {
        // (one linear: the columns' scales are those of the transposed weights' rows, one for each channel of each x_k)
        const at::Tensor Wt = (G == 1 ? W[0] : at::cat(W, 1)).t();
        dx = floats(x, x.sizes());
        if (split_x) run_f16x2(Wt, O, fp(dy), R, Bound{dy_max}, OptTensor(), kActNone, false, 1, *dx, nullptr, false, -1,
                               G == 1 ? OptTensor() : pack_ahead({}, {Wt})[0]);
        else check(mg_tensor_linear_rows(fp(Wt), Wt.stride(0), Wt.stride(1), fp(dy), O, R, (int)O, (int)(G * C), 0, fp(*dx), stream_of(x)));
    }
    Tensors dW;
    if (want_W) {
        at::Tensor all = floats(x, {O, G * C});
        size_t n = 0;
        if (!narrow) check(mg_tensor_linear_wgrad_workspace_bytes(R, (int)(G * C), (int)O, &n));
        at::Tensor ws = bytes_like(x, n);
        if (narrow) {
            narrow_wgrad(0, R, dy, x, G * C, O, all);
        } else if (split_W) {
            if (!x_max.has_value()) x_max = row_absmax(x.view({R * G, C}));
            check(mg_tensor_linear_wgrad_f16x2_groups(fp(dy), fp(x), fp(dy_max), R, fp(x_max), (int)G, R, (int)(G * C), (int)O,
                                                      ws.data_ptr(), fp(all), stream_of(x)));
        } else {
            check(mg_tensor_linear_wgrad(0, fp(dy), fp(x), R, (int)(G * C), (int)O, ws.data_ptr(), fp(all), stream_of(x)));
        }
        for (int64_t k = 0; k < G; k++) dW.push_back(all.narrow(1, k * C, C));
    }
    return {dx, dW};
}

// y = x W^T, with the bias added to the first bias_rows rows
at::Tensor rows_linear(const at::Tensor& W, const OptTensor& bias, const at::Tensor& x, int64_t bias_rows, Bound bound,
                       const OptTensor& packed = OptTensor()) {
    const int64_t rows = x.size(0), dim_in = W.size(1), dim_out = W.size(0);
    at::Tensor y = floats(x, {rows, dim_out});
    if (rows == 0) return y;
    if (mg_get_linear_mode() == kModeF16x2 && f16x2_takes(rows, dim_in, dim_out, x)) {
        if (!bound.base.has_value()) bound = Bound{};
        run_f16x2(W, dim_in, fp(x), rows, bound, bias, kActNone, false, 1, y, nullptr, false, bias_rows, packed);
        return y;
    }
    auto piece = [&](int64_t lo, int64_t hi, const OptTensor& b) {
        if (hi > lo)
            linear_fwd(0, W, x.narrow(0, lo, hi - lo), b, kActNone, OptTensor(y.narrow(0, lo, hi - lo)), false, 0, 0, OptTensor(), 1,
                       0, 1, false, OptTensor(), OptTensor(), false);
    };
    const int64_t cut = bias.has_value() ? std::min(bias_rows, rows) : rows;
    piece(0, cut, bias);
    piece(cut, rows, OptTensor());
    return y;
}

// dW over all rows and db over the first bias_rows
std::pair<at::Tensor, OptTensor> rows_wgrad(const at::Tensor& dy, const at::Tensor& x, int64_t bias_rows, bool want_bias,
                                            const OptTensor& dy_bound, const OptTensor& x_bound) {
    const int64_t rows = x.size(0), dim_in = x.size(1), dim_out = dy.size(1);
    if (mg_get_linear_mode() == kModeF16x2 && aligned16(x) && aligned16(dy) &&
        mg_tensor_linear_wgrad_f16x2_supported(rows, (int)dim_in, (int)dim_out)) {
        at::Tensor dW = floats(x, {dim_out, dim_in}), db;
        if (want_bias) db = floats(x, {dim_out});
        size_t n = 0;
        check(mg_tensor_linear_wgrad_workspace_bytes(rows, (int)dim_in, (int)dim_out, &n));
        at::Tensor ws = bytes_like(x, n);
        check(mg_tensor_linear_wgrad_f16x2_rows(fp(dy), fp(x), fp(dy_bound), dy_bound.has_value() ? dy_bound->numel() : 0, fp(x_bound),
                                                x_bound.has_value() ? x_bound->numel() : 0, rows, bias_rows, (int)dim_in, (int)dim_out,
                                                ws.data_ptr(), fp(dW), want_bias ? fp(db) : nullptr, stream_of(x)));
        return {dW, want_bias ? OptTensor(db) : OptTensor()};
    }
    at::Tensor dW = std::get<0>(linear_wgrad(0, dy, x, dy_bound, x_bound, false));
    return {dW, want_bias ? OptTensor(dy.narrow(0, 0, bias_rows).sum(0)) : OptTensor()};
}

// rows_wgrad of several layers over the same rows
struct RowsGradient {
    at::Tensor dy, x;
    bool want_bias;
    OptTensor dy_bound, x_bound;
};
std::vector<std::pair<at::Tensor, OptTensor>> rows_wgrads(const std::vector<RowsGradient>& of, int64_t bias_rows) {
    std::vector<std::pair<at::Tensor, OptTensor>> out;
    bool merged = mg_get_linear_mode() == kModeF16x2;
    for (const RowsGradient& g : of)
        merged = merged && aligned16(g.x) && aligned16(g.dy) && g.x.size(0) == of[0].x.size(0) &&
                 mg_tensor_linear_wgrad_f16x2_supported(g.x.size(0), (int)g.x.size(1), (int)g.dy.size(1));
    if (!merged) {
        for (const RowsGradient& g : of) out.push_back(rows_wgrad(g.dy, g.x, bias_rows, g.want_bias, g.dy_bound, g.x_bound));
        return out;
    }
    std::vector<mg_wgrad_f16x2> jobs;
    for (const RowsGradient& g : of) {
        at::Tensor dW = floats(g.x, {g.dy.size(1), g.x.size(1)});
        OptTensor db;
        if (g.want_bias) db = floats(g.x, {g.dy.size(1)});
        jobs.push_back({fp(g.dy), fp(g.x), fp(g.dy_bound), g.dy_bound.has_value() ? g.dy_bound->numel() : 0, fp(g.x_bound),
                        g.x_bound.has_value() ? g.x_bound->numel() : 0, bias_rows, (int)g.x.size(1), (int)g.dy.size(1), fp(dW),
                        db.has_value() ? fp(*db) : nullptr});
        out.emplace_back(dW, db);
    }
    const int64_t rows = of[0].x.size(0);
    size_t n = 0;
    check(mg_tensor_linear_wgrad_f16x2_many_workspace_bytes(jobs.data(), (int)jobs.size(), rows, &n));
    at::Tensor ws = bytes_like(of[0].x, n);
    check(mg_tensor_linear_wgrad_f16x2_many(jobs.data(), (int)jobs.size(), rows, ws.data_ptr(), stream_of(of[0].x)));
    return out;
}

// Wide layers on values and tangents together: the one kernel has one accumulator for the large products there, 2.75e-7 from
// float64 where the split reductions of few rows are at 2.5e-7: it takes over where those end (4.1e-7 beyond).
bool mlp_dual_takes(int64_t rows, const Tensors& W, bool dual) {
    const int dim = (int)W[0].size(0);
    return !dual || dim <= kMlpWide || !mg_tensor_linear_f16x2_splits_k(rows, dim, dim);
}

// Linear, SiLU, Linear, SiLU, Linear on S = [x; x_t] (R or 2 R rows): y and what the adjoint reads again
std::pair<at::Tensor, std::vector<OptTensor>> mlp_rows_fwd(const at::Tensor& S, int64_t R, OptTensor bound, const Tensors& W,
                                                           const Tensors& b, bool train) {
    check_chain(S, W, b, kSiluMlp);
    const bool dual = S.size(0) != R;
    if (train) pack_ahead({W[0], W[1], W[2], W[0].t(), W[1].t(), W[2].t()});
    if (mlp_takes(S.size(0), S.size(1), W, S) && aligned_all(b) && mlp_dual_takes(S.size(0), W, dual)) {
        const int64_t rows = S.size(0), dim = W[0].size(0);
        mg_mlp_f16x2 a{};
        at::Tensor y = floats(S, {rows, dim});
        if (!bound.has_value()) {
            bound = floats(S, {rows, 1});
            a.x_rowmax = fp(*bound);
        }
        std::vector<OptTensor> saved{bound};
        Tensors planes;
        for (int l = 0; l < 3; l++) {
            planes.push_back(packed_f16x2(W[l], W[l].size(1)));
            a.packed_W[l] = planes[l].data_ptr();
            a.bias[l] = fp(b[l]);
            if (l == 2) break;
            at::Tensor z = floats(S, {rows, dim}), m = floats(S, {rows, 1}), h = floats(S, {rows, dim});
            a.z[l] = fp(z);
            a.h[l] = fp(h);
            a.h_rowmax[l] = fp(m);
            saved.insert(saved.end(), {OptTensor(z), OptTensor(m), OptTensor(h)});
        }
        a.x = fp(S);
        a.rows = R;
        a.dual = dual;
        a.dim_in = (int)S.size(1);
        a.dim = (int)dim;
        a.y = fp(y);
        check(mg_mlp_f16x2_forward(&a, stream_of(S)));
        return {y, saved};
    }
    if (!bound.has_value() && S.size(1) >= 64) bound = row_absmax(S);
    std::vector<OptTensor> saved{bound};
    at::Tensor h = S;
    Bound hb{bound};
    for (int l = 0; l < 2; l++) {
        at::Tensor z = rows_linear(W[l], OptTensor(b[l]), h, R, hb), m = floats(z, {z.size(0), 1});
        h = floats(z, z.sizes());
        check(mg_silu_rows_fwd(fp(z), R, (int)z.size(1), dual, fp(h), fp(m), stream_of(z)));
        hb = Bound{OptTensor(m)};
        saved.insert(saved.end(), {OptTensor(z), OptTensor(m), OptTensor(h)});
    }
    return {rows_linear(W[2], OptTensor(b[2]), h, R, hb), saved};
}

// gradients of the rows S (if wanted), then of the three weights and biases
std::tuple<OptTensor, Tensors> mlp_rows_bwd(at::Tensor g, OptTensor g_bound, const at::Tensor& S, int64_t R, const Tensors& W,
                                            const std::vector<OptTensor>& saved, bool want_x, bool want_params) {
    const bool dual = S.size(0) != R;
    Tensors params(6);
    OptTensor g_x;
    auto weight_grads = [&](int l, const at::Tensor& dz, const OptTensor& dz_bound) {
        if (!want_params) return;
        auto [dW, db] = rows_wgrad(dz, l == 0 ? S : *saved[3 * l], R, true, dz_bound, l == 0 ? saved[0] : saved[3 * l - 1]);
        params[2 * l] = dW;
        params[2 * l + 1] = *db;
    };
    const int64_t dim = W[0].size(0);
    if (saved[0].has_value() && g.size(1) == dim && aligned16(g) && mlp_takes(S.size(0), S.size(1), W, S) &&
        mlp_dual_takes(S.size(0), W, dual)) {
        const int64_t rows = S.size(0);
        mg_mlp_f16x2_grad a{};
        if (!g_bound.has_value()) {
            g_bound = floats(g, {rows, 1});
            a.dy_rowmax = fp(*g_bound);
        }
        at::Tensor dz[2], m[2];
        Tensors planes;
        for (int l = 0; l < 3; l++) {
            planes.push_back(packed_f16x2(W[l].t(), W[l].size(0)));
            a.packed_Wt[l] = planes[l].data_ptr();
            if (l == 2) break;
            dz[l] = floats(g, {rows, dim});
            m[l] = floats(g, {rows, 1});
            a.z[l] = fp(*saved[3 * l + 1]);
            a.dz[l] = fp(dz[l]);
            a.dz_rowmax[l] = fp(m[l]);
        }
        if (want_x) {
            g_x = floats(S, S.sizes());
            a.dx = fp(*g_x);
        }
        a.dy = fp(g);
        a.rows = R;
        a.dual = dual;
        a.dim_in = (int)S.size(1);
        a.dim = (int)dim;
        check(mg_mlp_f16x2_adjoint(&a, stream_of(g)));
        if (want_params) {
            const auto of = rows_wgrads({{dz[0], S, true, OptTensor(m[0]), saved[0]},
                                         {dz[1], *saved[3], true, OptTensor(m[1]), saved[2]},
                                         {g, *saved[6], true, g_bound, saved[5]}}, R);
            for (int l = 0; l < 3; l++) {
                params[2 * l] = of[l].first;
                params[2 * l + 1] = *of[l].second;
            }
        }
        return {g_x, params};
    }
    for (int l = 2; l >= 0; l--) {
        if (!g_bound.has_value()) g_bound = row_absmax(g);
        weight_grads(l, g, g_bound);
        if (l == 0) {
            if (want_x) g_x = rows_linear(W[0].t(), OptTensor(), g, 0, Bound{g_bound});
            break;
        }
        const at::Tensor dh = rows_linear(W[l].t(), OptTensor(), g, 0, Bound{g_bound});
        const at::Tensor& z = *saved[3 * l - 2];
        g = floats(z, z.sizes());
        at::Tensor m = floats(z, {z.size(0), 1});
        check(mg_silu_rows_bwd(fp(z), fp(dh), R, (int)z.size(1), dual, fp(g), fp(m), stream_of(z)));
        g_bound = m;
    }
    return {g_x, params};
}

std::vector<int64_t> with_last(const at::Tensor& x, int64_t last) {
    std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = last;
    return shape;
}

std::tuple<at::Tensor, OptTensor, std::vector<OptTensor>> mlp_silu_fwd(const at::Tensor& x, const OptTensor& x_t, const OptTensor& bound,
                                                                       const Tensors& W, const Tensors& b, bool train) {
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    const at::Tensor S = stacked(x, x_t, x.size(-1));
    auto [y, saved] = mlp_rows_fwd(S, x.numel() / x.size(-1), bound, W, b, train);
    const auto shape = with_last(x, y.size(1));
    return {on_storage(y, 0, shape), second_half(y, shape, x_t.has_value()), saved};
}

std::tuple<OptTensor, OptTensor, Tensors> mlp_silu_bwd(const at::Tensor& g, const OptTensor& g_t, const at::Tensor& x, const OptTensor& x_t,
                                                       const Tensors& W, const std::vector<OptTensor>& saved, bool want_x,
                                                       bool want_params) {
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    const bool dual = x_t.has_value();
    const at::Tensor S = stacked(x, x_t, x.size(-1)), G = stacked(g, g_t, g.size(-1));
    auto [g_x, params] = mlp_rows_bwd(G, OptTensor(), S, x.numel() / x.size(-1), W, saved, want_x, want_params);
    if (!want_x) return {OptTensor(), OptTensor(), params};
    return {on_storage(*g_x, 0, x.sizes()), second_half(*g_x, x.sizes(), dual), params};
}

// x W_d^T + the three layers with LeakyReLU(0.1) between them; W: the layers' weights, then W_d.  From the row count at which plain
// linears leave the fp32 kernel, for every size: the slope at zero should not depend on it.
bool mlp_leaky_takes(const at::Tensor& x, const Tensors& W, const Tensors& b) {
    if (mg_get_linear_mode() != kModeF16x2 || x.dim() != 2 || x.size(0) < 256 || W.size() != 4 || b.size() != 3) return false;
    for (const at::Tensor& t : W)
        if (!t.is_cuda() || t.scalar_type() != at::kFloat || t.dim() != 2 || !packs_f16x2(t)) return false;
    const int64_t K = W[0].size(1), O = W[0].size(0), N = W[2].size(0);
    if (x.size(1) != K || W[1].size(0) != O || W[1].size(1) != O || W[2].size(1) != O || W[3].size(0) != N || W[3].size(1) != K) return false;
    for (int l = 0; l < 3; l++)
        if (!b[l].is_cuda() || b[l].scalar_type() != at::kFloat || !b[l].is_contiguous() || b[l].numel() != W[l].size(0)) return false;
    return x.is_cuda() && x.scalar_type() == at::kFloat && x.is_contiguous() && aligned16(x) && aligned_all(b) &&
           mg_mlp_leaky_f16x2_supported((int)K, (int)O, (int)N);
}

// saved: row maxima of |x|, then h and its row maxima of either hidden layer
// residual: of x + y
std::tuple<at::Tensor, Tensors> mlp_leaky_fwd(const at::Tensor& x, const Tensors& W, const Tensors& b, bool residual) {
    TORCH_CHECK(mlp_leaky_takes(x, W, b), "mlp_leaky_fwd: sizes or types");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    pack_ahead({W[0], W[1], W[2], W[3], W[0].t(), W[1].t(), W[2].t(), W[3].t()});
    const int64_t rows = x.size(0), dim = W[0].size(0);
    mg_mlp_leaky_f16x2 a{};
    at::Tensor y = floats(x, {rows, W[2].size(0)});
    Tensors saved{floats(x, {rows, 1})}, planes;
    for (int l = 0; l < 3; l++) {
        planes.push_back(packed_f16x2(W[l], W[l].size(1)));
        a.packed_W[l] = planes[l].data_ptr();
        a.bias[l] = fp(b[l]);
        if (l == 2) break;
        saved.push_back(floats(x, {rows, dim}));
        a.h[l] = fp(saved.back());
        saved.push_back(floats(x, {rows, 1}));
        a.h_rowmax[l] = fp(saved.back());
    }
    a.x = fp(x);
    a.x_rowmax = fp(saved[0]);
    a.rows = rows;
    a.dim_in = (int)W[0].size(1);
    a.dim = (int)dim;
    a.dim_out = (int)W[2].size(0);
    a.y = fp(y);
    check((residual ? mg_mlp_leaky_f16x2_residual_forward : mg_mlp_leaky_f16x2_forward)(&a, stream_of(x)));
    run_f16x2(W[3], W[3].size(1), fp(x), rows, Bound{OptTensor(saved[0])}, OptTensor(), kActNone, true, 1, y, nullptr, true);
    return {y, saved};
}

std::tuple<OptTensor, Tensors> mlp_leaky_bwd(const at::Tensor& g, const at::Tensor& x, const Tensors& W, const Tensors& saved,
                                             bool want_x, bool want_params, bool residual) {
    check_input(g, "gradient");
    TORCH_CHECK(W.size() == 4 && saved.size() == 5 && g.dim() == 2 && g.size(0) == x.size(0) && g.size(1) == W[2].size(0) && aligned16(g),
                "mlp_leaky_bwd: sizes");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    const int64_t rows = x.size(0), dim = W[0].size(0);
    mg_mlp_leaky_f16x2_grad a{};
    at::Tensor dz[2], m[2], g_max = floats(x, {rows, 1});
    OptTensor g_x;
    Tensors planes;
    for (int l = 0; l < 3; l++) {
        planes.push_back(packed_f16x2(W[l].t(), W[l].size(0)));
        a.packed_Wt[l] = planes[l].data_ptr();
        if (l == 2) break;
        dz[l] = floats(x, {rows, dim});
        m[l] = floats(x, {rows, 1});
        a.h[l] = fp(saved[1 + 2 * l]);
        a.dz[l] = fp(dz[l]);
        a.dz_rowmax[l] = fp(m[l]);
    }
    a.dy = fp(g);
    a.dy_rowmax = fp(g_max);
    if (want_x) {
        g_x = floats(x, x.sizes());
        a.dx = fp(*g_x);
    }
    a.rows = rows;
    a.dim_in = (int)W[0].size(1);
    a.dim = (int)dim;
    a.dim_out = (int)W[2].size(0);
    check((residual ? mg_mlp_leaky_f16x2_residual_adjoint : mg_mlp_leaky_f16x2_adjoint)(&a, stream_of(x)));
    if (want_x) run_f16x2(W[3].t(), W[3].size(0), fp(g), rows, Bound{OptTensor(g_max)}, OptTensor(), kActNone, true, 1, *g_x, nullptr, false);
    Tensors params;
    if (want_params) {
        for (auto& [dW, db] : rows_wgrads({{dz[0], x, true, OptTensor(m[0]), OptTensor(saved[0])},
                                           {dz[1], saved[1], true, OptTensor(m[1]), OptTensor(saved[2])},
                                           {g, saved[3], true, OptTensor(g_max), OptTensor(saved[4])},
                                           {g, x, false, OptTensor(g_max), OptTensor(saved[0])}}, rows)) {
            params.push_back(dW);
            if (db.has_value()) params.push_back(*db);
        }
    }
    return {g_x, params};
}

// enc, enc_t, row bounds of both, dir, dir_t
std::tuple<at::Tensor, OptTensor, at::Tensor, at::Tensor, OptTensor> edge_encode_fwd(const at::Tensor& r, const OptTensor& r_t, int64_t n,
                                                                                     double rmax, double eps) {
    check_input(r, "r_ij");
    TORCH_CHECK(r.dim() == 2 && r.size(1) == 3, "r_ij must have shape (edges, 3)");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(r.device());
    const int64_t E = r.size(0), copies = r_t.has_value() ? 2 : 1;
    if (r_t.has_value()) check_input(*r_t, "tangent of r_ij");
    at::Tensor enc = floats(r, {copies * E, n}), bound = floats(r, {copies * E, 1}), dir = floats(r, {copies * E, 3});
    check(mg_painn_edge_encode_fwd(fp(r), fp(r_t), E, (int)n, (float)rmax, (float)eps, fp(enc), fp(bound), fp(dir),
                                   r_t.has_value() ? fp(dir) + 3 * E : nullptr, stream_of(r)));
    const bool dual = r_t.has_value();
    return {on_storage(enc, 0, {E, n}), second_half(enc, {E, n}, dual), bound, on_storage(dir, 0, {E, 3}), second_half(dir, {E, 3}, dual)};
}

std::tuple<at::Tensor, OptTensor> edge_encode_bwd(const at::Tensor& r, const OptTensor& r_t, int64_t n, double rmax, double eps,
                                                  const at::Tensor& g_enc, const OptTensor& g_enc_t, const at::Tensor& g_dir,
                                                  const OptTensor& g_dir_t) {
    c10::hip::HIPGuardMasqueradingAsCUDA guard(r.device());
    const bool dual = r_t.has_value();
    const at::Tensor G = stacked(g_enc, g_enc_t, n);
    check_input(g_dir, "g_dir");
    if (dual) check_input(*g_dir_t, "g_dir_t");
    at::Tensor g_r = floats(r, r.sizes()), g_rt;
    if (dual) g_rt = floats(r, r.sizes());
    check(mg_painn_edge_encode_bwd(fp(r), fp(r_t), r.size(0), (int)n, (float)rmax, (float)eps, fp(G), fp(g_dir), fp(g_dir_t), fp(g_r),
                                   dual ? fp(g_rt) : nullptr, stream_of(r)));
    return {g_r, dual ? OptTensor(g_rt) : OptTensor()};
}

// in: dist, dist_t, actv, actv_t, v, v_t, dir, dir_t (the odd ones may be missing)
mg_painn_combine_dual combine_in(const std::vector<OptTensor>& in) {
    TORCH_CHECK(in.size() == 8, "combine_dual: eight operands expected");
    for (int k = 0; k < 8; k++) {
        TORCH_CHECK(k % 2 == 1 || in[k].has_value(), "combine_dual: a value is missing");
        if (in[k].has_value()) check_input(*in[k], "operand of the message");
        TORCH_CHECK(k % 2 == 0 || !in[k].has_value() || in[k]->numel() == in[k - 1]->numel(), "a tangent must have the shape of its value");
    }
    const int64_t E = in[6]->size(0), rows = in[4]->size(0), n = in[4]->size(1);
    TORCH_CHECK(in[0]->dim() == 2 && in[0]->size(0) == E && in[0]->size(1) == 4 * n && in[6]->size(1) == 3 && in[2]->dim() == 2 &&
                    in[2]->size(0) == rows && in[2]->size(1) == 4 * n && in[4]->dim() == 3 && in[4]->size(2) == 3,
                "combine_dual: dist (edges, 4n), actv (nodes, 4n), v (nodes, n, 3) and dir (edges, 3) expected");
    return {fp(in[0]), fp(in[1]), fp(in[2]), fp(in[3]), fp(in[4]), fp(in[5]), fp(in[6]), fp(in[7]), E, rows, (int)n};
}

// The rows a, a_t, v, v_t (any may be missing) that a layer adds to its results
mg_painn_rows rows_in(const std::vector<OptTensor>& in, int64_t rows, int64_t n) {
    TORCH_CHECK(in.size() == 4, "four arrays of rows expected");
    for (int k = 0; k < 4; k++) {
        if (!in[k].has_value()) continue;
        check_input(*in[k], "rows to add");
        TORCH_CHECK(in[k]->numel() == rows * n * (k < 2 ? 1 : 3), "rows to add: wrong shape");
    }
    return {fp(in[0]), fp(in[1]), fp(in[2]), fp(in[3])};
}

// residual: nothing, or a, a_t, v, v_t.  Each result on storage of its own: a dual tensor copies a tangent that shares its value's.
Tensors combine_dual_fwd(const std::vector<OptTensor>& in, const at::Tensor& node, const at::Tensor& row_ptr, int64_t n_out,
                         const std::vector<OptTensor>& residual) {
    const mg_painn_combine_dual a = combine_in(in);
    check_input(node, "node", at::kInt);
    check_input(row_ptr, "row_ptr", at::kInt);
    TORCH_CHECK(node.numel() == a.E && row_ptr.numel() == n_out + 1, "combine_dual: index sizes");
    const at::Tensor& like = *in[0];
    c10::hip::HIPGuardMasqueradingAsCUDA guard(like.device());
    mg_painn_rows res{};
    if (!residual.empty()) res = rows_in(residual, n_out, a.n);
    Tensors out{floats(like, {n_out, a.n, 3}), floats(like, {n_out, a.n}), floats(like, {n_out, a.n, 3}), floats(like, {n_out, a.n})};
    check(mg_painn_combine_dual_add_fwd(&a, node.data_ptr<int>(), row_ptr.data_ptr<int>(), n_out, &res, fp(out[0]), fp(out[2]),
                                        fp(out[1]), fp(out[3]), stream_of(like)));
    return out;
}

std::vector<OptTensor> combine_dual_bwd(const std::vector<OptTensor>& in, const at::Tensor& row_ptr, const OptTensor& order,
                                        const Tensors& g, const at::Tensor& grad_row, int64_t n_grad_rows, const std::vector<bool>& want,
                                        bool residual) {
    const mg_painn_combine_dual a = combine_in(in);
    check_input(row_ptr, "row_ptr", at::kInt);
    check_input(grad_row, "grad_row", at::kInt);
    if (order.has_value()) check_input(*order, "order", at::kInt);
    TORCH_CHECK(row_ptr.numel() == a.n_rows + 1 && grad_row.numel() == a.E && (!order.has_value() || order->numel() == a.E) &&
                    g.size() == 4 && want.size() == 8,
                "combine_dual: index sizes");
    for (int k = 0; k < 4; k++) {
        check_input(g[k], "gradient of the message");
        TORCH_CHECK(g[k].numel() == n_grad_rows * a.n * (k % 2 == 0 ? 3 : 1), "combine_dual: gradient sizes");
    }
    const at::Tensor& like = *in[0];
    c10::hip::HIPGuardMasqueradingAsCUDA guard(like.device());
    std::vector<OptTensor> out(8);
    float* p[8];
    for (int k = 0; k < 8; k += 2) {             // a value's gradient and its tangent's, one behind the other
        p[k] = p[k + 1] = nullptr;
        const auto shape = in[k]->sizes();
        const bool first = want[k] || (k == 6 && want[7]), second = want[k + 1] && in[k + 1].has_value();
        if (!first && !second) continue;
        std::vector<int64_t> both(shape.begin(), shape.end());
        both[0] *= 2;
        at::Tensor buf = floats(like, both);
        if (first) out[k] = on_storage(buf, 0, shape);
        if (second) out[k + 1] = on_storage(buf, in[k]->numel(), shape);
        p[k] = first ? fp(buf) : nullptr;
        p[k + 1] = second ? fp(buf) + in[k]->numel() : nullptr;
    }
    const mg_painn_combine_dual_grad d{p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7]};
    // (v went past the message as well: its gradient is the sum's own plus that of the result it was added to)
    TORCH_CHECK(!residual || n_grad_rows == a.n_rows, "combine_dual: rows to add");
    const mg_painn_rows add{nullptr, nullptr, residual ? fp(g[0]) : nullptr, residual ? fp(g[2]) : nullptr};
    check(mg_painn_combine_dual_add_bwd(&a, row_ptr.data_ptr<int>(), order.has_value() ? order->data_ptr<int>() : nullptr, fp(g[0]),
                                        fp(g[2]), fp(g[1]), fp(g[3]), grad_row.data_ptr<int>(), n_grad_rows, &add, &d,
                                        stream_of(like)));
    return out;
}

// x_v (and its tangent) as one plain row per (row, component), and the row maxima
std::pair<at::Tensor, at::Tensor> vector_rows(const at::Tensor& x_v, const OptTensor& x_vt, int64_t R, int64_t n) {
    const int64_t copies = x_vt.has_value() ? 2 : 1;
    if (n >= 32 && n <= 256 && power_of_two(n)) {
        at::Tensor x2 = floats(x_v, {copies * R * 3, n}), m = floats(x_v, {copies * R * 3, 1});
        check(mg_components_to_rows(fp(x_v), R, (int)n, 3, (int)n, fp(x2), fp(m), stream_of(x_v)));
        if (x_vt.has_value())
            check(mg_components_to_rows(fp(*x_vt), R, (int)n, 3, (int)n, fp(x2) + R * 3 * n, fp(m) + R * 3, stream_of(x_v)));
        return {x2, m};
    }
    at::Tensor x2 = stacked(x_v, x_vt, n * 3).reshape({copies * R, n, 3}).transpose(1, 2).contiguous().reshape({copies * R * 3, n});
    return {x2, row_absmax(x2)};
}

// Update.forward with its adjoint's operands: x_a (batch, nodes, n), x_v (batch, nodes, n, 3), weights {l, r, v}
std::tuple<Tensors, std::vector<OptTensor>> painn_update_train_fwd(const at::Tensor& x_a, const OptTensor& x_at, const at::Tensor& x_v,
                                                                   const OptTensor& x_vt, const Tensors& lrv_W, const Tensors& W,
                                                                   const Tensors& b, int groups, const at::Tensor& gamma,
                                                                   const at::Tensor& beta, double eps, bool residual) {
    check_input(x_a, "x_a");
    check_input(x_v, "x_v");
    check_input(gamma, "gamma");
    check_input(beta, "beta");
    const int64_t B = x_a.size(0), N = x_a.size(1), n = x_a.size(2), R = B * N;
    TORCH_CHECK(x_v.numel() == 3 * x_a.numel() && gamma.numel() == n && beta.numel() == n, "painn_update: operand sizes");
    const bool dual = x_vt.has_value();
    for (const OptTensor& t : {x_at, x_vt})
        if (t.has_value()) check_input(*t, "tangent");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x_a.device());
    const int64_t copies = dual ? 2 : 1;
    const at::Tensor W_lrv = at::cat(lrv_W);
    const auto lrv_planes = pack_ahead({W[0], W[1], W[2], W[0].t(), W[1].t(), W[2].t()}, {W_lrv, W_lrv.t()});
    auto [x2, x2max] = vector_rows(x_v, x_vt, R, n);
    const at::Tensor lrv = rows_linear(W_lrv, OptTensor(), x2, 0, Bound{OptTensor(x2max)}, lrv_planes[0]);
    at::Tensor ip = floats(x_a, {copies * R, n}), cat = floats(x_a, {copies * R, 2 * n}), cat_max = floats(x_a, {copies * R, 1});
    const mg_stream_t st = stream_of(x_a);
    check(mg_painn_update_pre_fwd(fp(lrv), fp(x_a), fp(x_at), R, (int)n, dual, fp(ip), fp(cat), fp(cat_max), st));
    auto [y, mlp_saved] = mlp_rows_fwd(cat, R, OptTensor(cat_max), W, b, false);
    TORCH_CHECK(y.size(1) == 3 * n, "the update's MLP must end in 3n columns");
    long fwd = 0, bwd = 0;
    check(mg_painn_update_scratch_floats((int)B, (int)N, (int)n, groups, &fwd, &bwd));
    at::Tensor scratch = floats(x_a, {std::max<int64_t>(fwd, 1)}), stats = floats(x_a, {B * groups, 4});
    Tensors out;                                 // (each on storage of its own, as combine_dual_fwd's)
    for (int k = 0; k < copies; k++) {
        out.push_back(floats(x_a, x_a.sizes()));
        out.push_back(floats(x_v, x_v.sizes()));
    }
    mg_painn_rows res{};
    if (residual) res = rows_in({OptTensor(x_a), x_at, OptTensor(x_v), x_vt}, R, n);
    check(mg_painn_update_post_add_fwd(fp(lrv), fp(ip), fp(y), fp(gamma), fp(beta), (int)B, (int)N, (int)n, groups, (float)eps, dual,
                                       fp(scratch), fp(stats), &res, fp(out[0]), dual ? fp(out[2]) : nullptr, fp(out[1]),
                                       dual ? fp(out[3]) : nullptr, st));
    std::vector<OptTensor> saved{OptTensor(W_lrv), OptTensor(x2), OptTensor(x2max), OptTensor(lrv), OptTensor(ip), OptTensor(cat),
                                 OptTensor(y), OptTensor(stats), lrv_planes[1]};
    saved.insert(saved.end(), mlp_saved.begin(), mlp_saved.end());
    return {out, saved};
}

// gradients of x_a, x_v and their tangents, of l, r, v, of gamma and beta, and of the MLP's weights and biases
std::tuple<std::vector<OptTensor>, Tensors> painn_update_train_bwd(const at::Tensor& g_a, const OptTensor& g_at, const at::Tensor& g_v,
                                                                   const OptTensor& g_vt, const Tensors& W, int groups,
                                                                   const at::Tensor& gamma, const std::vector<OptTensor>& saved,
                                                                   bool residual) {
    const bool dual = g_at.has_value();
    check_input(g_a, "gradient of out_a");
    check_input(g_v, "gradient of out_v");
    for (const OptTensor& t : {g_at, g_vt})
        if (t.has_value()) check_input(*t, "gradient of a tangent");
    const int64_t B = g_a.size(0), N = g_a.size(1), n = g_a.size(2), R = B * N, copies = dual ? 2 : 1;
    c10::hip::HIPGuardMasqueradingAsCUDA guard(g_a.device());
    const at::Tensor &W_lrv = *saved[0], &x2 = *saved[1], &lrv = *saved[3], &ip = *saved[4], &cat = *saved[5], &y = *saved[6],
                     &stats = *saved[7];
    const std::vector<OptTensor> mlp_saved(saved.begin() + 9, saved.end());
    const mg_stream_t st = stream_of(g_a);
    long fwd = 0, bwd = 0;
    check(mg_painn_update_scratch_floats((int)B, (int)N, (int)n, groups, &fwd, &bwd));
    at::Tensor scratch = floats(g_a, {std::max<int64_t>(bwd, 1)});
    at::Tensor g_y = floats(y, y.sizes()), g_y_max = floats(y, {y.size(0), 1}), g_ip = floats(ip, ip.sizes());
    at::Tensor g_lrv = floats(lrv, lrv.sizes()), g_lrv_max = floats(lrv, {copies * R * 3, 1});
    at::Tensor d_gamma = floats(g_a, {n}), d_beta = floats(g_a, {n});
    check(mg_painn_update_post_bwd(fp(lrv), fp(ip), fp(y), fp(stats), fp(gamma), fp(g_a), fp(g_at), fp(g_v), fp(g_vt), (int)B, (int)N,
                                   (int)n, groups, dual, fp(scratch), fp(g_y), fp(g_y_max), fp(g_ip), fp(g_lrv), fp(d_gamma),
                                   fp(d_beta), st));
    auto [g_cat, mlp_params] = mlp_rows_bwd(g_y, OptTensor(g_y_max), cat, R, W, mlp_saved, true, true);
    at::Tensor g_xa = floats(g_a, {copies * R, n});
    mg_painn_rows add{};
    if (residual) add = rows_in({OptTensor(g_a), g_at, OptTensor(g_v), g_vt}, R, n);
    check(mg_painn_update_pre_add_bwd(fp(lrv), fp(g_ip), fp(*g_cat), R, (int)n, dual, fp(g_lrv), fp(g_lrv_max), &add, fp(g_xa), st));
    const OptTensor g_bound(g_lrv_max);
    const at::Tensor dW = rows_wgrad(g_lrv, x2, 0, false, g_bound, saved[2]).first;
    at::Tensor g_xv;
    const at::Tensor back = W_lrv.t();
    if (mg_get_linear_mode() == kModeF16x2 && f16x2_takes(copies * R * 3, 3 * n, n, g_lrv)) {
        g_xv = floats(g_a, {copies * R, n, 3});
        run_f16x2(back, 3 * n, fp(g_lrv), copies * R * 3, Bound{g_bound}, OptTensor(), kActNone, false, 3, g_xv, nullptr, false, -1,
                  saved[8]);
    } else {
        g_xv = rows_linear(back, OptTensor(), g_lrv, 0, Bound{g_bound}).reshape({copies * R, 3, n}).transpose(1, 2).contiguous();
    }
    const std::vector<int64_t> sv{B, N, n, 3};
    std::vector<OptTensor> g_x{OptTensor(on_storage(g_xa, 0, g_a.sizes())), second_half(g_xa, g_a.sizes(), dual),
                               OptTensor(on_storage(g_xv, 0, sv)), second_half(g_xv, sv, dual)};
    if (residual) {
        g_x[2]->add_(g_v.view(sv));
        if (dual) g_x[3]->add_(g_vt->view(sv));
    }
    Tensors params{on_storage(dW, 0, {n, n}), on_storage(dW, n * n, {n, n}), on_storage(dW, 2 * n * n, {n, n}), d_gamma, d_beta};
    params.insert(params.end(), mlp_params.begin(), mlp_params.end());
    return {g_x, params};
}

// (order, sorted keys) of a stable sort of int32 keys in 0 .. limit - 1; values: what order holds in the place of positions
std::pair<at::Tensor, at::Tensor> sort_values_by_key(const at::Tensor& keys, const OptTensor& values, int64_t limit) {
    at::Tensor order = at::empty_like(keys), sorted = at::empty_like(keys);
    size_t n = 0;
    check(mg_sort_by_key_workspace_bytes(keys.numel(), &n));
    at::Tensor ws = bytes_like(keys, n);
    check(mg_sort_values_by_key(keys.data_ptr<int>(), values.has_value() ? values->data_ptr<int>() : nullptr, keys.numel(), (int)limit,
                                ws.data_ptr(), order.data_ptr<int>(), sorted.data_ptr<int>(), stream_of(keys)));
    return {order, sorted};
}
std::pair<at::Tensor, at::Tensor> sort_by_key(const at::Tensor& keys, int64_t limit) {
    check_input(keys, "keys", at::kInt);
    c10::hip::HIPGuardMasqueradingAsCUDA guard(keys.device());
    return sort_values_by_key(keys, OptTensor(), limit);
}

// (d_table, d_actv, d_v) of the message interpolated from its grid; each only if wanted
std::tuple<OptTensor, OptTensor, OptTensor> painn_grid_message_bwd(const at::Tensor& table, const at::Tensor& actv,
                                                                   const at::Tensor& actv_sliced, const at::Tensor& v,
                                                                   const at::Tensor& r_ij, const at::Tensor& g_v, const at::Tensor& g_a,
                                                                   const at::Tensor& src, const at::Tensor& dst,
                                                                   const at::Tensor& row_ptr, const OptTensor& order,
                                                                   const OptTensor& node_order, double period, double epsilon,
                                                                   bool want_table, bool want_actv, bool want_v,
                                                                   const OptTensor& src_row_ptr, bool residual) {
    for (const at::Tensor& t : {table, actv, actv_sliced, v, r_ij, g_v, g_a}) check_input(t, "operand of the message");
    for (const at::Tensor& t : {src, dst, row_ptr}) check_input(t, "index", at::kInt);
    for (const OptTensor& t : {order, node_order, src_row_ptr})
        if (t.has_value()) check_input(*t, "order", at::kInt);
    const int64_t N = v.size(0), n = v.size(1), E = r_ij.size(0), rows = table.size(0);
    TORCH_CHECK(actv.numel() == N * 4 * n && actv_sliced.numel() == N * 4 * n && v.numel() == N * n * 3 && table.size(1) == 4 * n &&
                    g_v.numel() == N * n * 3 && g_a.numel() == N * n && r_ij.numel() == 3 * E && src.numel() == E && dst.numel() == E &&
                    row_ptr.numel() == N + 1 && (!order.has_value() || order->numel() == E) &&
                    (!node_order.has_value() || node_order->numel() == N) && (!src_row_ptr.has_value() || src_row_ptr->numel() == N + 1),
                "painn_grid_message_bwd: operand sizes");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(v.device());
    const mg_stream_t st = stream_of(v);
    size_t n_ws = 0;
    check(mg_painn_grid_grad_workspace_bytes((int)rows, (int)n, E, &n_ws));
    at::Tensor ws = bytes_like(v, n_ws);
    auto ints = [](const OptTensor& t) { return t.has_value() ? t->data_ptr<int>() : nullptr; };
    OptTensor d_table, d_actv, d_v;
    if (want_actv || want_v) {
        if (want_actv) d_actv = floats(v, {N, 4 * n});
        if (want_v) d_v = floats(v, v.sizes());
        // (v went past the message as well)
        check(mg_painn_grid_node_add_grad(row_ptr.data_ptr<int>(), ints(order), src.data_ptr<int>(), ints(node_order), (int)N, E,
                                      fp(r_ij), fp(table), (int)rows, (float)period, (float)epsilon, fp(g_v), fp(g_a), fp(actv), fp(v),
                                      (int)n, ws.data_ptr(), residual ? fp(g_v) : nullptr, want_actv ? fp(*d_actv) : nullptr, want_v ? fp(*d_v) : nullptr, st));
    }
    if (want_table) {
        d_table = floats(v, table.sizes());
        at::Tensor key = at::empty({E}, src.options()), ptr = at::empty({rows + 1}, src.options());
        OptTensor edge;
        if (node_order.has_value() && src_row_ptr.has_value()) {
            edge = at::empty({E}, src.options());
            size_t bytes = 0;
            check(mg_painn_grid_rows_by_node_workspace_bytes((int)N, &bytes));
            at::Tensor starts = bytes_like(v, bytes);
            check(mg_painn_grid_rows_by_node(fp(r_ij), E, src_row_ptr->data_ptr<int>(), node_order->data_ptr<int>(), (int)N, (int)rows,
                                             (float)period, starts.data_ptr(), key.data_ptr<int>(), edge->data_ptr<int>(), st));
        } else {
            check(mg_painn_grid_rows(fp(r_ij), E, (int)rows, (float)period, key.data_ptr<int>(), st));
        }
        auto [by_row, sorted] = sort_values_by_key(key, edge, rows);
        check(mg_segment_row_ptr(sorted.data_ptr<int>(), 0, E, (int)rows, ptr.data_ptr<int>(), st));
        check(mg_painn_grid_table_grad(by_row.data_ptr<int>(), ptr.data_ptr<int>(), src.data_ptr<int>(), dst.data_ptr<int>(), (int)N, E,
                                       fp(r_ij), (int)rows, (float)period, (float)epsilon, fp(g_v), fp(g_a), fp(actv_sliced), fp(v),
                                       (int)n, ws.data_ptr(), fp(*d_table), st));
    }
    return {d_table, d_actv, d_v};
}

// gradients of the rank-0/1/2 message products: (l_0, l_1, l_2), enc, rh.  dy: three gradients, operands and products
// component-major (mg_bee_message_grad_rows), or 13, all of them by channel (mg_bee_message_grad)
template <typename Args>
void bee_message_grad_fill(Args& a, const Tensors& left, Tensors& d_left, const at::Tensor& enc, const at::Tensor& rh,
                           const at::Tensor& row_ptr, const at::Tensor& dst, const at::Tensor& dst_row_ptr, const OptTensor& perm,
                           at::Tensor& ws, at::Tensor& d_enc, at::Tensor& d_rh) {
    a.l_0 = fp(left[0]);
    a.l_1 = fp(left[1]);
    a.l_2 = fp(left[2]);
    a.enc = fp(enc);
    a.rh = fp(rh);
    a.row_ptr = row_ptr.data_ptr<int>();
    a.dst = dst.data_ptr<int>();
    a.dst_row_ptr = dst_row_ptr.data_ptr<int>();
    a.perm = perm.has_value() ? perm->data_ptr<int>() : nullptr;
    a.E = enc.size(0);
    a.n_src = (int)row_ptr.numel() - 1;
    a.n_rows = (int)left[0].size(0);
    a.chan = (int)enc.size(1);
    a.workspace = ws.data_ptr();
    if (!d_left.empty()) {
        a.d_0 = fp(d_left[0]);
        a.d_1 = fp(d_left[1]);
        a.d_2 = fp(d_left[2]);
    }
    a.d_enc = d_enc.defined() ? fp(d_enc) : nullptr;
    a.d_rh = d_rh.defined() ? fp(d_rh) : nullptr;
}

std::tuple<Tensors, OptTensor, OptTensor> bee_message_bwd(const Tensors& left, const at::Tensor& enc, const at::Tensor& rh,
                                                          const Tensors& dy, const at::Tensor& row_ptr, const at::Tensor& dst,
                                                          const at::Tensor& dst_row_ptr, const OptTensor& perm, bool want_left,
                                                          bool want_enc, bool want_rh) {
    static const int rank_of[13] = {0, 0, 0, 1, 1, 1, 1, 2, 2, 2, 2, 1, 2};
    TORCH_CHECK(left.size() == 3 && (dy.size() == 3 || dy.size() == 13), "bee_message_bwd: three operands and 3 or 13 gradients expected");
    check_input(enc, "enc");
    check_input(rh, "rh");
    check_input(row_ptr, "row_ptr", at::kInt);
    check_input(dst, "dst", at::kInt);
    check_input(dst_row_ptr, "dst_row_ptr", at::kInt);
    if (perm.has_value()) check_input(*perm, "perm", at::kInt);
    TORCH_CHECK(enc.dim() == 2 && rh.dim() == 2, "bee_message_bwd: enc (edges, chan) and rh (edges, 3) expected");
    const bool rows_layout = dy.size() == 3;
    const int64_t E = enc.size(0), C = enc.size(1), rows = left[0].size(0), n_src = row_ptr.numel() - 1;
    const int64_t per_rank[3] = {C, 3 * C, 9 * C}, stacked[3] = {E * 3 * C, n_src * 15 * C, n_src * 45 * C};
    TORCH_CHECK(rh.numel() == 3 * E && dst.numel() == E && dst_row_ptr.numel() == rows + 1 && n_src >= 0 &&
                    (!perm.has_value() || perm->numel() == E),
                "bee_message_bwd: operand sizes");
    for (int k = 0; k < 3; k++) {
        check_input(left[k], "left operand");
        TORCH_CHECK(left[k].numel() == rows * per_rank[k], "bee_message_bwd: operand sizes");
    }
    for (size_t k = 0; k < dy.size(); k++) {
        check_input(dy[k], "gradient of the products");
        TORCH_CHECK(dy[k].numel() == (rows_layout ? stacked[k] : (rank_of[k] ? n_src : E) * per_rank[rank_of[k]]),
                    "bee_message_bwd: gradient sizes");
    }
    c10::hip::HIPGuardMasqueradingAsCUDA guard(enc.device());
    Tensors d_left;
    if (want_left)
        for (const at::Tensor& t : left) d_left.push_back(floats(t, t.sizes()));
    at::Tensor d_enc, d_rh;
    if (want_enc) d_enc = floats(enc, enc.sizes());
    if (want_rh) d_rh = floats(rh, rh.sizes());
    size_t bytes = 0;
    check(mg_bee_message_grad_workspace_bytes(E, (int)C, want_left, want_rh, &bytes));
    at::Tensor ws = bytes_like(enc, bytes);
    if (rows_layout) {
        mg_bee_message_grad_rows a{};
        bee_message_grad_fill(a, left, d_left, enc, rh, row_ptr, dst, dst_row_ptr, perm, ws, d_enc, d_rh);
        a.d_P0 = fp(dy[0]);
        a.d_S1 = fp(dy[1]);
        a.d_S2 = fp(dy[2]);
        check(mg_bee_message_grad_rows_run(&a, stream_of(enc)));
    } else {
        mg_bee_message_grad a{};
        bee_message_grad_fill(a, left, d_left, enc, rh, row_ptr, dst, dst_row_ptr, perm, ws, d_enc, d_rh);
        for (int k = 0; k < 13; k++) a.dy[k] = fp(dy[k]);
        check(mg_bee_message_grad_run(&a, stream_of(enc)));
    }
    return {d_left, want_enc ? OptTensor(d_enc) : OptTensor(), want_rh ? OptTensor(d_rh) : OptTensor()};
}

}  // namespace

void register_ops(pybind11::module_& m) {
    m.def("invalidate_weight_caches", [] { g_epoch.fetch_add(1); });
    m.def("packed_weight", &packed_weight);
    m.def("tens_norms", &tens_norms);
    m.def("row_absmax", &row_absmax);
    m.def("linear_f16x2", &linear_f16x2);
    m.def("linear_fwd", &linear_fwd);
    m.def("component_rows_take", &component_rows_take);
    m.def("linear_wgrad", &linear_wgrad);
    m.def("row_linears_fwd", &row_linears_fwd);
    m.def("row_linears_bwd", &row_linears_bwd);
    m.def("silu_order", &silu_order);
    m.def("linear_chain", &linear_chain);
    m.def("tens_norm_fwd", &tens_norm_fwd);
    m.def("tens_norm_bwd", &tens_norm_bwd);
    m.def("filter_grid", &filter_grid);
    m.def("filter_grids", &filter_grids);
    m.def("mlp_takes_rows", &mlp_takes_rows);
    m.def("painn_update", &painn_update);
    m.def("painn_message_grid", &painn_message_grid);
    m.def("painn_message_edges", &painn_message_edges);
    m.def("sort_by_key", &sort_by_key);
    m.def("painn_grid_message_bwd", &painn_grid_message_bwd);
    m.def("bee_message_bwd", &bee_message_bwd);
    m.def("mlp_silu_fwd", &mlp_silu_fwd);
    m.def("mlp_silu_bwd", &mlp_silu_bwd);
    m.def("mlp_leaky_takes", &mlp_leaky_takes);
    m.def("mlp_leaky_fwd", &mlp_leaky_fwd, py::arg("x"), py::arg("W"), py::arg("b"), py::arg("residual") = false);
    m.def("mlp_leaky_bwd", &mlp_leaky_bwd, py::arg("g"), py::arg("x"), py::arg("W"), py::arg("saved"), py::arg("want_x"),
          py::arg("want_params"), py::arg("residual") = false);
    m.def("edge_encode_fwd", &edge_encode_fwd);
    m.def("edge_encode_bwd", &edge_encode_bwd);
    m.def("combine_dual_fwd", &combine_dual_fwd);
    m.def("combine_dual_bwd", &combine_dual_bwd);
    m.def("painn_update_train_fwd", &painn_update_train_fwd);
    m.def("painn_update_train_bwd", &painn_update_train_bwd);
}
