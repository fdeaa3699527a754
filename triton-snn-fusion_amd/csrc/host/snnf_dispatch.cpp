// Native dispatch of the `snn_custom` operators and of the internal-layout entry points: the host side of a call that has
// been seen before.
//
// What bounds a small call is the host. An operator call through the Python implementations takes 12 us (one neuron step)
// to 50 us (a convolution with a 16-bit membrane), of which the kernel launch itself is 3: argument checks, reason strings,
// statistics, ctypes. All of that depends on the call's signature alone - shapes, dtypes, parameters, which operands are
// there -, so the first call of a signature runs the Python implementation, which stays the only place where calls are
// judged, refused and counted, and this file remembers a signature that ran natively together with the statistics it
// added. Later calls of the signature are a hash look-up, two allocations and the C ABI call (measured, batch-1 neuron
// step: 12.2 -> 5.9 us per call).
// A call whose signature is unknown, whose tensors are not plain contiguous GPU tensors, whose entry point returns an error, or
// that throws on its way (no memory, a weight that cannot be packed) goes through the Python implementation, which raises or
// falls back as it always did.
//
// State: the plan table (bounded; cleared when full), the hit counters, the packed weights of live weight tensors. All under
// one mutex: operator calls arrive without the interpreter lock and from any thread. The mutex is never held while the
// interpreter lock is requested.
#include <Python.h>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/python/pybind_utils.h>
#include <torch/extension.h>
#include <torch/library.h>

#include <array>
#include <atomic>
#include <cstring>
#include <list>
#include <memory>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "snnf.h"

namespace {

using at::Tensor;
using c10::IValue;
using torch::jit::Stack;

constexpr int kMaxSteps = 64;              // timesteps whose pointers fit on the stack of a call; longer sequences take the Python path
constexpr size_t kMaxPlans = 4096;
constexpr size_t kMaxWeights = 512;

// ------------------------------------------------------------------------------------------------------------------
// Signatures and plans
// ------------------------------------------------------------------------------------------------------------------
struct Key {
    std::array<int64_t, 64> v;
    int n = 0;
    bool plain = true;                     // false: something about the call keeps it off the fast path

    void add(int64_t x) {
        if (n < static_cast<int>(v.size())) v[n++] = x; else plain = false;
    }
    void add(double x) {
        int64_t bits;
        std::memcpy(&bits, &x, sizeof bits);
        add(bits);
    }
    void sizes(const Tensor& t) {
        add(t.dim());
        for (int64_t d : t.sizes()) add(d);
    }
    // A GPU operand that the kernels read in place. Inference tensors have signatures of their own: as weights they have no version by
    // which a packed copy could be known to be current, and the Python implementations refuse to pack them.
    void tensor(const Tensor& t) {
        if (!t.defined() || !t.is_cuda() || !t.is_contiguous()) {
            plain = false;
            return;
        }
        add((static_cast<int64_t>(t.scalar_type()) << 16) | (t.is_inference() ? 1 << 8 : 0) | t.device().index());
        sizes(t);
    }
    bool operator==(const Key& o) const { return n == o.n && std::memcmp(v.data(), o.v.data(), n * sizeof(int64_t)) == 0; }
};

struct KeyHash {
    size_t operator()(const Key& k) const {
        uint64_t h = 0x9e3779b97f4a7c15ull;
        for (int i = 0; i < k.n; ++i) {
            h ^= static_cast<uint64_t>(k.v[i]);
            h *= 0xff51afd7ed558ccdull;
            h ^= h >> 32;
        }
        return h;
    }
};

// What the first call of a signature established. `statistic` < 0 with `native` false: the call does not run natively.
struct Plan {
    bool native = false;
    int statistic = -1;                    // index into the hit counters, -1: the call counts nothing
    int route = 0;                         // internal-layout convolutions: bits of `Learnt`
};

std::mutex g_mutex;
std::unordered_map<Key, Plan, KeyHash> g_plans;
std::vector<int64_t> g_hits;
std::atomic<bool> g_enabled{false};

bool find_plan(const Key& key, Plan* out) {
    std::lock_guard<std::mutex> lock(g_mutex);
    auto it = g_plans.find(key);
    if (it == g_plans.end()) return false;
    *out = it->second;
    return true;
}

// A call on its way to the kernels: its signature, and after `known()` what is remembered about it.
struct Attempt : Key {
    Plan plan;
    bool searched = false, found = false;
    bool known() {
        if (!plain) return false;
        searched = true;
        found = find_plan(*this, &plan);
        return found && plan.native;
    }
    bool worth_learning() const { return plain && searched && !found; }
};

void remember(const Key& key, const Plan& plan) {
    std::lock_guard<std::mutex> lock(g_mutex);
    if (g_plans.size() >= kMaxPlans) g_plans.clear();
    g_plans[key] = plan;
}

void count(const Plan& plan) {
    if (plan.statistic < 0) return;
    std::lock_guard<std::mutex> lock(g_mutex);
    if (plan.statistic >= static_cast<int>(g_hits.size())) g_hits.resize(plan.statistic + 1, 0);
    ++g_hits[plan.statistic];
}

// ------------------------------------------------------------------------------------------------------------------
// Packed weights of live tensors (the Python backend packs; a tensor is looked up by identity, version and address, as there)
// ------------------------------------------------------------------------------------------------------------------
using WeakTensor = c10::weak_intrusive_ptr<c10::TensorImpl, c10::UndefinedTensorImpl>;

struct WeightKey {
    const void* w;
    const void* b;
    int64_t form;                          // packed element type, or the plane of a matrix form
    bool operator==(const WeightKey& o) const { return w == o.w && b == o.b && form == o.form; }
};
struct WeightHash {
    size_t operator()(const WeightKey& k) const {
        return reinterpret_cast<size_t>(k.w) * 31 + reinterpret_cast<size_t>(k.b) * 17 + static_cast<size_t>(k.form);
    }
};
struct WeightEntry {
    WeakTensor w, b;
    int64_t w_version, b_version;
    const void *w_data, *b_data;
    Tensor first, second;                  // packed weight, or matrix and bias row
    std::list<WeightKey>::iterator age;
};

std::unordered_map<WeightKey, WeightEntry, WeightHash> g_weights;
std::list<WeightKey> g_weight_ages;        // most recently used in front
py::object* g_pack = nullptr;              // _packed_weight(weight, bias, dtype)
py::object* g_plane = nullptr;             // _plane_matrix(weight, bias, H, W, ph, pw)

int64_t version_of(const Tensor& t) { return static_cast<int64_t>(t._version()); }

// Tensors that leave the table are released by the caller after the mutex: freeing one can need the interpreter lock.
using Released = std::vector<Tensor>;

void drop_weight(std::unordered_map<WeightKey, WeightEntry, WeightHash>::iterator it, Released* released) {
    released->push_back(std::move(it->second.first));
    released->push_back(std::move(it->second.second));
    g_weight_ages.erase(it->second.age);
    g_weights.erase(it);
}

bool find_weight(const WeightKey& key, const Tensor& w, const Tensor& b, Tensor* first, Tensor* second) {
    Released released;
    std::lock_guard<std::mutex> lock(g_mutex);
    auto it = g_weights.find(key);
    if (it == g_weights.end()) return false;
    WeightEntry& e = it->second;
    // An address can be handed to a new tensor once the old one is gone: an entry whose weak reference has expired is stale.
    if (e.w.expired() || e.b.expired() || e.w_version != version_of(w) || e.b_version != version_of(b) || e.w_data != w.data_ptr()
        || e.b_data != b.data_ptr()) {
        drop_weight(it, &released);
        return false;
    }
    if (e.age != g_weight_ages.begin()) g_weight_ages.splice(g_weight_ages.begin(), g_weight_ages, e.age);
    *first = e.first;
    if (second) *second = e.second;
    return true;
}

void keep_weight(const WeightKey& key, const Tensor& w, const Tensor& b, Tensor first, Tensor second) {
    Released released;
    std::lock_guard<std::mutex> lock(g_mutex);
    auto it = g_weights.find(key);
    if (it != g_weights.end()) drop_weight(it, &released);
    for (auto i = g_weights.begin(); i != g_weights.end();) {          // what dead tensors left behind
        auto next = std::next(i);
        if (i->second.w.expired() || i->second.b.expired()) drop_weight(i, &released);
        i = next;
    }
    while (g_weights.size() >= kMaxWeights) drop_weight(g_weights.find(g_weight_ages.back()), &released);
    g_weight_ages.push_front(key);
    g_weights.emplace(key, WeightEntry{WeakTensor(w.getIntrusivePtr()), WeakTensor(b.getIntrusivePtr()), version_of(w), version_of(b), w.data_ptr(),
                                       b.data_ptr(), std::move(first), std::move(second), g_weight_ages.begin()});
}

Tensor packed_weight(const Tensor& w, const Tensor& b, at::ScalarType dtype) {
    const WeightKey key{w.unsafeGetTensorImpl(), b.unsafeGetTensorImpl(), -1 - static_cast<int64_t>(dtype)};
    Tensor packed;
    if (find_weight(key, w, b, &packed, nullptr)) return packed;
    py::gil_scoped_acquire gil;
    packed = (*g_pack)(w, b, py::reinterpret_borrow<py::object>(reinterpret_cast<PyObject*>(torch::getTHPDtype(dtype)))).cast<Tensor>();
    keep_weight(key, w, b, packed, Tensor());
    return packed;
}

void plane_matrix(const Tensor& w, const Tensor& b, int64_t H, int64_t W, int64_t ph, int64_t pw, Tensor* matrix, Tensor* row) {
    const WeightKey key{w.unsafeGetTensorImpl(), b.unsafeGetTensorImpl(), ((H * 64 + W) * 64 + ph) * 64 + pw};
    if (find_weight(key, w, b, matrix, row)) return;
    py::gil_scoped_acquire gil;
    auto pair = (*g_plane)(w, b, H, W, ph, pw).cast<std::pair<Tensor, Tensor>>();
    *matrix = pair.first;
    *row = pair.second;
    keep_weight(key, w, b, pair.first, pair.second);
}

// ------------------------------------------------------------------------------------------------------------------
// Workspaces of the split linear kernel: owned by the Python backend, which never frees one (a captured graph may hold its
// address); remembered here per (device, stream, capturing).
// ------------------------------------------------------------------------------------------------------------------
struct Workspace {
    void* data;
    size_t bytes;
};
struct WorkspaceSlot {
    int device;
    void* stream;
    bool capturing;
    Workspace space;
};
std::vector<WorkspaceSlot> g_workspaces;
py::object* g_workspace = nullptr;         // _split_workspace(lib, device, T, M, Fin, Fout), lib bound

Workspace split_workspace(const Tensor& like, hipStream_t stream, int64_t T, int64_t M, int64_t fin, int64_t fout) {
    const size_t need = snnf_linear_lif_workspace_bytes(static_cast<int>(T), static_cast<int>(M), static_cast<int>(fin), static_cast<int>(fout));
    if (need == 0) return {nullptr, 0};
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    (void)hipStreamIsCapturing(stream, &status);
    const bool capturing = status != hipStreamCaptureStatusNone;
    // A capture's stream exists only for the capture: captured calls share one workspace per device.
    void* const tag = capturing ? nullptr : static_cast<void*>(stream);
    const int device = like.device().index();
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        for (const WorkspaceSlot& s : g_workspaces)
            if (s.device == device && s.stream == tag && s.capturing == capturing && s.space.bytes >= need) return s.space;
    }
    py::gil_scoped_acquire gil;
    py::object got = (*g_workspace)(py::cast(like).attr("device"), T, M, fin, fout);
    if (got.is_none()) return {nullptr, 0};
    const Tensor t = got.cast<Tensor>();
    const Workspace space{t.data_ptr(), static_cast<size_t>(t.numel())};
    std::lock_guard<std::mutex> lock(g_mutex);
    for (WorkspaceSlot& s : g_workspaces)
        if (s.device == device && s.stream == tag && s.capturing == capturing) {
            s.space = space;
            return space;
        }
    if (g_workspaces.size() >= 64) g_workspaces.clear();
    g_workspaces.push_back({device, tag, capturing, space});
    return space;
}

// ------------------------------------------------------------------------------------------------------------------
// Small helpers
// ------------------------------------------------------------------------------------------------------------------
bool dtype_code(at::ScalarType t, int* code) {
    switch (t) {
        case at::kFloat: *code = SNNF_F32; return true;
        case at::kBFloat16: *code = SNNF_BF16; return true;
        case at::kHalf: *code = SNNF_F16; return true;
        default: return false;
    }
}

int code_of(at::ScalarType t) {
    int code = SNNF_F32;
    dtype_code(t, &code);
    return code;
}

hipStream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor empty(at::IntArrayRef sizes, at::ScalarType dtype, const Tensor& like) {
    return at::empty(sizes, at::TensorOptions().dtype(dtype).device(like.device()));
}

struct Lif {
    double v_threshold, v_reset, tau;
};

// The membrane of a call: dtype (membrane_dtype in _lib.py) and, when it does not start from zeros, the tensor it starts from.
struct Membrane {
    at::ScalarType dtype;
    const Tensor* from = nullptr;
};

Membrane membrane_of(const Tensor& x, const Tensor& v) {
    const bool chooses = (v.scalar_type() == at::kFloat || v.scalar_type() == x.scalar_type()) && v.device() == x.device();
    return {chooses ? v.scalar_type() : x.scalar_type(), nullptr};
}

// Adds `v_init` to the key; a tensor state has to be one that the kernels read in place.
Membrane add_membrane(Key& key, const Tensor& x, const Tensor& v, at::IntArrayRef shape) {
    Membrane m = membrane_of(x, v);
    key.add((static_cast<int64_t>(v.scalar_type()) << 8) | (v.dim() == 0 ? 0 : 1) | (v.device() == x.device() ? 2 : 0));
    if (v.dim() != 0) {
        if (v.device() != x.device() || v.scalar_type() != m.dtype || v.sizes() != shape || !v.is_contiguous()) key.plain = false;
        m.from = &v;
    }
    return m;
}

const void* data_or_null(const Tensor* t) { return t ? t->data_ptr() : nullptr; }

// More steps than a launch takes hand the membrane from launch to launch through the output: a 16-bit one then works in float32
// and is rounded once at the end.
struct WorkMembrane {
    Tensor out, work, start;
    const void* from;
    WorkMembrane(const Tensor& x, const Membrane& m, at::IntArrayRef shape, bool wide) : out(empty(shape, m.dtype, x)), from(data_or_null(m.from)) {
        work = out;
        if (wide) widen(x, m, shape);
    }
    void widen(const Tensor& x, const Membrane& m, at::IntArrayRef shape) {
        work = empty(shape, at::kFloat, x);
        if (m.from) {
            start = m.from->to(at::kFloat);
            from = start.data_ptr();
        }
    }
    int code() const { return code_of(work.scalar_type()); }
    void finish() {
        if (work.unsafeGetTensorImpl() != out.unsafeGetTensorImpl()) out.copy_(work);
    }
};

// ------------------------------------------------------------------------------------------------------------------
// Operators
// ------------------------------------------------------------------------------------------------------------------
enum Op { kStep, kScan, kTail, kLinear, kLinearPacked, kConv, kPointwise, kDepthwise, kDepthwiseAlias, kConvAdd, kConvAddDepthwise, kConvSingle };

py::object* g_slow = nullptr;              // slow(name, args, learn) -> (result, statistic or None)

// The Python implementation. `learn`: remember the signature when the call ran natively.
void call_python(const c10::OperatorHandle& op, Stack* stack, const Key* learn) {
    const size_t n = op.schema().arguments().size();
    Plan plan;
    Tensor first, second;
    {
        py::gil_scoped_acquire gil;
        py::list args;
        for (size_t i = stack->size() - n; i < stack->size(); ++i) args.append(torch::jit::toPyObject((*stack)[i]));
        py::tuple answer = (*g_slow)(op.schema().name(), args, learn != nullptr).cast<py::tuple>();
        py::tuple result = answer[0].cast<py::tuple>();
        first = result[0].cast<Tensor>();
        second = result[1].cast<Tensor>();
        if (!answer[1].is_none()) {
            plan.native = true;
            plan.statistic = answer[1].cast<int>();
        }
    }
    if (learn) remember(*learn, plan);
    torch::jit::drop(*stack, n);
    torch::jit::push(*stack, std::move(first), std::move(second));
}

struct Call {
    Stack* stack;
    size_t base;
    const IValue& at(size_t i) const { return (*stack)[base + i]; }
    Lif lif(size_t i) const { return {at(i).toDouble(), at(i + 1).toDouble(), at(i + 2).toDouble()}; }
};

void add_lif(Key& key, const Call& c, size_t i) {
    for (size_t k = 0; k < 3; ++k) key.add(c.at(i + k).toDouble());
    key.add(static_cast<int64_t>(c.at(i + 3).toBool()));
}

using Pair = std::pair<Tensor, Tensor>;

// A native route that throws ends there, with nothing handed out: the Python implementation then runs the call, and raises what
// there is to raise, of the type that it always had, or counts a fallback. Only what is no error (an interrupt) leaves here.
template <typename Body>
auto run_native(Body&& body) -> decltype(body()) {
    try {
        return body();
    } catch (py::error_already_set& e) {
        py::gil_scoped_acquire gil;
        if (!e.matches(PyExc_Exception)) throw;
    } catch (const std::exception&) {
    }
    return {};
}

// Each operator builds its signature and, when that is known to run natively, enqueues the kernels and returns true.
bool step_call(const Call& c, Attempt& key, Pair* out) {
    const Tensor x = c.at(0).toTensor(), v = c.at(1).toTensor();
    const Lif lif = c.lif(2);
    int code;
    // One GPU operand is enough for a call to arrive here: a state on the GPU does not make the input one.
    key.tensor(x);
    if (!key.plain || !dtype_code(x.scalar_type(), &code) || x.numel() == 0 || lif.tau == 0.0) return false;
    const Membrane m = membrane_of(x, v);
    // A state of another shape, device or dtype starts from zeros.
    const bool continues = v.dim() != 0 && v.sizes() == x.sizes() && v.device() == x.device() && v.scalar_type() == m.dtype;
    if (continues && !v.is_contiguous()) return false;
    Tensor spikes = at::empty_like(x), next = empty(x.sizes(), m.dtype, x);
    const void* xs = x.data_ptr();
    const int64_t n = x.numel();
    if (snnf_lif_scan(&xs, 1, n, code, continues ? v.data_ptr() : nullptr, code_of(m.dtype), spikes.data_ptr(), n, next.data_ptr(),
                      static_cast<float>(lif.v_threshold), static_cast<float>(lif.v_reset), static_cast<float>(lif.tau), stream_of(x)) != 0)
        return false;
    *out = {std::move(spikes), std::move(next)};
    return true;
}

// Where the T steps of a contiguous tensor start. Of a single step `stride(0)` says nothing: a size-1 dimension of a contiguous
// tensor may have any stride, so the size of a step is always the product of its extents.
void packed_steps(const Tensor& x, int64_t T, const void** steps) {
    const char* base = static_cast<const char*>(x.data_ptr());
    const int64_t bytes = x.stride(0) * static_cast<int64_t>(x.element_size());
    for (int64_t t = 0; t < T; ++t) steps[t] = base + t * bytes;
}

// Whether all of several timesteps read the same tensor: such a convolution runs once, on the dense kernels, without scratch memory.
bool one_frame(const void* const* steps, int64_t T) {
    for (int64_t t = 1; t < T; ++t)
        if (steps[t] != steps[0]) return false;
    return T > 1;
}

// Scratch memory of a convolution from the pool of the current stream; none where the allocator has none left: such a call runs on the dense
// kernels. (A DataPtr, not a tensor: that costs another microsecond.)
c10::DataPtr scratch_memory(const Tensor& like, size_t bytes) {
    if (bytes == 0) return {};
    const c10::DeviceGuard guard(like.device());
    try {
        return c10::GetAllocator(c10::kCUDA)->allocate(bytes);
    } catch (const c10::OutOfMemoryError&) {
        return {};
    }
}

bool scan_call(const Call& c, Attempt& key, Pair* out) {
    const Tensor x = c.at(0).toTensor(), v = c.at(1).toTensor();
    key.tensor(x);
    if (!key.plain || x.dim() != 5 || x.size(0) > kMaxSteps) {
        key.plain = false;
        return false;
    }
    const auto shape = x.sizes().slice(1);
    const Membrane m = add_membrane(key, x, v, shape);
    add_lif(key, c, 2);
    if (!key.known()) return false;
    const int64_t T = x.size(0), n = c10::multiply_integers(shape);
    const void* steps[kMaxSteps];
    packed_steps(x, T, steps);
    const Lif lif = c.lif(2);
    Tensor spikes = at::empty_like(x);
    WorkMembrane w(x, m, shape, m.dtype != at::kFloat && T > SNNF_MAX_T_PER_LAUNCH);
    if (snnf_lif_scan(steps, static_cast<int>(T), n, code_of(x.scalar_type()), w.from, w.code(), spikes.data_ptr(), n, w.work.data_ptr(),
                      static_cast<float>(lif.v_threshold), static_cast<float>(lif.v_reset), static_cast<float>(lif.tau), stream_of(x)) != 0)
        return false;
    w.finish();
    *out = {std::move(spikes), std::move(w.out)};
    return true;
}

// An optional bias: absent or empty means none.
bool add_bias(Key& key, const IValue& v, Tensor* bias) {
    if (v.isTensor() && v.toTensor().defined() && v.toTensor().numel() > 0) {
        *bias = v.toTensor();
        key.tensor(*bias);
        return true;
    }
    key.add(static_cast<int64_t>(-1));
    return false;
}

bool tail_call(const Call& c, Attempt& key, Pair* out) {
    const Tensor x = c.at(0).toTensor(), v = c.at(1).toTensor(), fw = c.at(2).toTensor();
    key.tensor(x);
    key.tensor(fw);
    if (!key.plain || x.dim() != 5 || x.size(0) > kMaxSteps) {
        key.plain = false;
        return false;
    }
    Tensor fb;
    const bool biased = add_bias(key, c.at(3), &fb);
    const auto shape = x.sizes().slice(1);
    const Membrane m = add_membrane(key, x, v, shape);
    add_lif(key, c, 4);
    if (!key.known()) return false;
    const int T = static_cast<int>(x.size(0)), N = static_cast<int>(x.size(1)), C = static_cast<int>(x.size(2));
    const void* steps[kMaxSteps];
    packed_steps(x, T, steps);
    const Lif lif = c.lif(4);
    const int64_t K = fw.size(0);
    Tensor sum = empty({N, K}, x.scalar_type(), x), next = empty(shape, m.dtype, x);
    const size_t bytes = snnf_lif_pool_linear_workspace_bytes(N, C);
    Tensor workspace = empty({static_cast<int64_t>(bytes)}, at::kByte, x);
    if (snnf_lif_pool_linear(steps, T, N, C, static_cast<int>(x.size(3)), static_cast<int>(x.size(4)), code_of(x.scalar_type()), data_or_null(m.from),
                             code_of(m.dtype), fw.data_ptr(), biased ? fb.data_ptr() : nullptr, static_cast<int>(K), code_of(fw.scalar_type()),
                             sum.data_ptr(), next.data_ptr(), workspace.data_ptr(), bytes, static_cast<float>(lif.v_threshold),
                             static_cast<float>(lif.v_reset), static_cast<float>(lif.tau), stream_of(x)) != 0)
        return false;
    *out = {std::move(sum), std::move(next)};
    return true;
}

// The T inputs of a list operator: plain tensors of one shape, dtype and device. Returns T, or 0.
int64_t list_steps(Key& key, const IValue& v, const void** steps, Tensor* first) {
    if (!v.isTensorList()) {
        key.plain = false;
        return 0;
    }
    const auto list = v.toTensorList();
    const int64_t T = static_cast<int64_t>(list.size());
    if (T < 1 || T > kMaxSteps) {
        key.plain = false;
        return 0;
    }
    *first = list.get(0);
    key.tensor(*first);
    key.add(T);
    if (!key.plain) return 0;
    steps[0] = first->data_ptr();
    for (int64_t t = 1; t < T; ++t) {
        const Tensor x = list.get(t);
        if (x.sizes() != first->sizes() || x.scalar_type() != first->scalar_type() || x.device() != first->device() || !x.is_contiguous()) {
            key.plain = false;
            return 0;
        }
        steps[t] = x.data_ptr();
    }
    return T;
}

bool linear_call(const Call& c, Attempt& key, bool packed, Pair* out) {
    const void* steps[kMaxSteps];
    Tensor x;
    int64_t T, M, fin;
    if (packed) {
        x = c.at(0).toTensor();
        key.tensor(x);
        if (!key.plain || x.dim() != 3 || x.size(0) < 1 || x.size(0) > kMaxSteps) {
            key.plain = false;
            return false;
        }
        T = x.size(0), M = x.size(1), fin = x.size(2);
        packed_steps(x, T, steps);
    } else {
        T = list_steps(key, c.at(0), steps, &x);
        if (!key.plain || x.dim() != 2) {
            key.plain = false;
            return false;
        }
        M = x.size(0), fin = x.size(1);
    }
    const Tensor w = c.at(1).toTensor(), v = c.at(3).toTensor();
    key.tensor(w);
    if (!key.plain || w.dim() != 2) {
        key.plain = false;
        return false;
    }
    Tensor bias;
    const bool biased = add_bias(key, c.at(2), &bias);
    const int64_t fout = w.size(0);
    const std::array<int64_t, 2> shape{M, fout};
    const Membrane m = add_membrane(key, x, v, shape);
    add_lif(key, c, 4);
    if (!key.known()) return false;
    const Lif lif = c.lif(4);
    const hipStream_t stream = stream_of(x);
    const Workspace space = split_workspace(x, stream, T, M, fin, fout);
    Tensor spikes = empty({T, M, fout}, x.scalar_type(), x);
    WorkMembrane wm(x, m, shape, m.dtype != at::kFloat && T > SNNF_MAX_T_PER_LAUNCH);
    if (snnf_linear_lif_ws(steps, static_cast<int>(T), static_cast<int>(M), static_cast<int>(fin), fin, code_of(x.scalar_type()), w.data_ptr(),
                           biased ? bias.data_ptr() : nullptr, static_cast<int>(fout), code_of(w.scalar_type()), wm.from, wm.code(),
                           spikes.data_ptr(), M * fout, wm.work.data_ptr(), static_cast<float>(lif.v_threshold), static_cast<float>(lif.v_reset),
                           static_cast<float>(lif.tau), space.data, space.bytes, stream) != 0)
        return false;
    wm.finish();
    *out = {std::move(spikes), std::move(wm.out)};
    return true;
}

bool conv_call(const Call& c, Attempt& key, Op op, Pair* out) {
    const bool residual = op == kConvAdd || op == kConvAddDepthwise;
    const void* steps[kMaxSteps];
    const void* rs[kMaxSteps];
    Tensor x, r;
    int64_t T = 1;
    size_t i = 1;
    if (op == kConvSingle) {
        x = c.at(0).toTensor();
        key.tensor(x);
        if (key.plain) steps[0] = x.data_ptr();
    } else {
        T = list_steps(key, c.at(0), steps, &x);
        if (residual && key.plain && list_steps(key, c.at(i++), rs, &r) != T) key.plain = false;
    }
    if (!key.plain) return false;
    const Tensor w = c.at(i).toTensor(), b = c.at(i + 1).toTensor(), v = c.at(i + 2).toTensor();
    key.tensor(w);
    key.tensor(b);
    if (!key.plain || x.dim() != 4 || w.dim() != 4) {
        key.plain = false;
        return false;
    }
    int64_t geometry[6];                   // stride, padding, dilation
    for (int k = 0; k < 3; ++k) {
        const auto pair = c.at(i + 3 + k).toIntList();
        if (pair.size() != 2) {
            key.plain = false;
            return false;
        }
        geometry[2 * k] = pair.get(0);
        geometry[2 * k + 1] = pair.get(1);
    }
    const int64_t groups = c.at(i + 6).toInt();
    for (int64_t g : geometry) key.add(g);
    key.add(groups);
    const int64_t sh = geometry[0], sw = geometry[1], ph = geometry[2], pw = geometry[3];
    const int64_t kh = w.size(2), kw = w.size(3);
    if (sh < 1 || sw < 1) {
        key.plain = false;
        return false;
    }
    const std::array<int64_t, 4> shape{x.size(0), w.size(0), (x.size(2) + 2 * ph - kh) / sh + 1, (x.size(3) + 2 * pw - kw) / sw + 1};
    const Membrane m = add_membrane(key, x, v, shape);
    add_lif(key, c, i + 7);
    if (!key.known()) return false;
    const Lif lif = c.lif(i + 7);
    const bool depthwise = groups > 1;     // the only grouped convolutions that run natively
    const hipStream_t stream = stream_of(x);
    const int N = static_cast<int>(x.size(0)), cin = static_cast<int>(x.size(1)), H = static_cast<int>(x.size(2)), W = static_cast<int>(x.size(3));
    const int64_t step = shape[0] * shape[1] * shape[2] * shape[3];
    Tensor spikes = op == kConvSingle ? empty(shape, x.scalar_type(), x) : empty({T, shape[0], shape[1], shape[2], shape[3]}, x.scalar_type(), x);
    const void* const* residuals = residual ? rs : nullptr;
    const auto scratch_bytes = [&](int v_code) -> size_t {
        if (depthwise || one_frame(steps, T)) return 0;
        return snnf_conv_lif_scratch_bytes(static_cast<int>(T), N, cin, H, W, code_of(x.scalar_type()), static_cast<int>(shape[1]), static_cast<int>(kh),
                                           static_cast<int>(kw), static_cast<int>(sh), static_cast<int>(sw), static_cast<int>(ph), static_cast<int>(pw),
                                           v_code, residual ? 1 : 0);
    };
    // With scratch memory the library keeps a 16-bit membrane wide between its launches by itself.
    const bool narrow = m.dtype != at::kFloat && T > (depthwise ? SNNF_MAX_T_PER_LAUNCH : 1);
    size_t bytes = scratch_bytes(code_of(m.dtype));
    WorkMembrane wm(x, m, shape, narrow && bytes == 0);
    int status;
    if (depthwise) {
        status = snnf_dwconv3x3_lif(steps, residuals, static_cast<int>(T), N, cin, H, W, static_cast<int>(sh), code_of(x.scalar_type()), w.data_ptr(),
                                    b.data_ptr(), code_of(w.scalar_type()), wm.from, wm.code(), spikes.data_ptr(), step, wm.work.data_ptr(),
                                    static_cast<float>(lif.v_threshold), static_cast<float>(lif.v_reset), static_cast<float>(lif.tau), stream);
    } else {
        const Tensor packed = packed_weight(w, b, x.scalar_type());
        const c10::DataPtr workspace = scratch_memory(x, bytes);
        if (bytes > 0 && !workspace) {
            bytes = 0;
            if (narrow) wm.widen(x, m, shape);
        }
        status = snnf_conv_lif_ws(steps, residuals, static_cast<int>(T), N, cin, H, W, code_of(x.scalar_type()), packed.data_ptr(),
                                  static_cast<int>(shape[1]), static_cast<int>(kh), static_cast<int>(kw), static_cast<int>(sh), static_cast<int>(sw),
                                  static_cast<int>(ph), static_cast<int>(pw), wm.from, wm.code(), spikes.data_ptr(), step, wm.work.data_ptr(),
                                  static_cast<float>(lif.v_threshold), static_cast<float>(lif.v_reset), static_cast<float>(lif.tau),
                                  workspace.get(), bytes, stream);
    }
    if (status != 0) return false;
    wm.finish();
    *out = {std::move(spikes), std::move(wm.out)};
    return true;
}

template <Op OP>
void dispatch(const c10::OperatorHandle& op, Stack* stack) {
    const size_t n = op.schema().arguments().size();
    const Call c{stack, stack->size() - n};
    Pair out;
    Attempt attempt;
    bool ran = false;
    if (g_enabled.load(std::memory_order_relaxed)) {
        attempt.add(static_cast<int64_t>(OP));
        ran = run_native([&]() -> bool {
            if constexpr (OP == kStep) return step_call(c, attempt, &out);      // counts nothing, and its conditions are few: no plan
            else if constexpr (OP == kScan) return scan_call(c, attempt, &out);
            else if constexpr (OP == kTail) return tail_call(c, attempt, &out);
            else if constexpr (OP == kLinear || OP == kLinearPacked) return linear_call(c, attempt, OP == kLinearPacked, &out);
            else return conv_call(c, attempt, OP, &out);
        });
    }
    if (!ran) return call_python(op, stack, attempt.worth_learning() ? &attempt : nullptr);
    count(attempt.plan);
    torch::jit::drop(*stack, n);
    torch::jit::push(*stack, std::move(out.first), std::move(out.second));
}

TORCH_LIBRARY_IMPL(snn_custom, CUDA, m) {
    m.impl("lif_forward_state", torch::CppFunction::makeFromBoxedFunction<&dispatch<kStep>>());
    m.impl("fused_conv_lif_state", torch::CppFunction::makeFromBoxedFunction<&dispatch<kConvSingle>>());
    m.impl("fused_temporal_conv_lif_state", torch::CppFunction::makeFromBoxedFunction<&dispatch<kConv>>());
    m.impl("fused_temporal_pointwise_conv_lif_state", torch::CppFunction::makeFromBoxedFunction<&dispatch<kPointwise>>());
    m.impl("fused_temporal_depthwise_conv_lif_state", torch::CppFunction::makeFromBoxedFunction<&dispatch<kDepthwise>>());
    m.impl("fused_temporal_conv_lif_state_depthwise", torch::CppFunction::makeFromBoxedFunction<&dispatch<kDepthwiseAlias>>());
    m.impl("fused_temporal_conv_add_lif_state", torch::CppFunction::makeFromBoxedFunction<&dispatch<kConvAdd>>());
    m.impl("fused_temporal_conv_add_lif_state_depthwise", torch::CppFunction::makeFromBoxedFunction<&dispatch<kConvAddDepthwise>>());
    m.impl("fused_temporal_lif_state", torch::CppFunction::makeFromBoxedFunction<&dispatch<kScan>>());
    m.impl("fused_temporal_lif_avgpool_linear", torch::CppFunction::makeFromBoxedFunction<&dispatch<kTail>>());
    m.impl("fused_temporal_lif_tail", torch::CppFunction::makeFromBoxedFunction<&dispatch<kTail>>());
    m.impl("fused_temporal_linear_lif_state", torch::CppFunction::makeFromBoxedFunction<&dispatch<kLinear>>());
    m.impl("fused_temporal_linear_lif_state_packed", torch::CppFunction::makeFromBoxedFunction<&dispatch<kLinearPacked>>());
}

// ------------------------------------------------------------------------------------------------------------------
// Internal layouts (hip_blocked_backend.py): plain functions, called with the interpreter lock held, which they give back while they
// allocate and launch. Each takes what the Python entry point has in hand and returns the result, or None for a call that is not
// known: the Python entry point then runs it and, when it ran, calls again with what it learnt in the last argument.
// ------------------------------------------------------------------------------------------------------------------
enum Blocked { kBlockedConv = 100, kBlockedShortcut, kBlockedAvgPool, kBlockedPool, kBlockedHead, kDenseConvBias, kDensePool };
enum Learnt { kRoutePlane = 1, kAllocateV = 2, kReturnV = 4 };     // the last argument; -1: run

struct Args {
    PyObject* const* v;
    Py_ssize_t n;
    bool fine = true;
    std::array<Tensor, 8> held;
    int n_held = 0;

    int64_t number(Py_ssize_t i) {
        const long long x = PyLong_AsLongLong(v[i]);
        if (x == -1 && PyErr_Occurred()) {
            PyErr_Clear();
            fine = false;
        }
        return x;
    }
    double real(Py_ssize_t i) {
        const double x = PyFloat_AsDouble(v[i]);
        if (x == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            fine = false;
        }
        return x;
    }
    // The tensors are held here: the kernels are launched without the interpreter lock.
    const Tensor* tensor(Py_ssize_t i) {
        if (!THPVariable_Check(v[i]) || n_held == static_cast<int>(held.size())) {
            fine = false;
            return nullptr;
        }
        held[n_held] = THPVariable_Unpack(v[i]);
        return &held[n_held++];
    }
    // a pair of numbers, or one number for both
    void pair(Py_ssize_t i, int64_t* a, int64_t* b) {
        PyObject* o = v[i];
        if (PyLong_Check(o)) {
            *a = *b = number(i);
            return;
        }
        if ((!PyList_Check(o) && !PyTuple_Check(o)) || PySequence_Fast_GET_SIZE(o) != 2) {
            fine = false;
            return;
        }
        PyObject** items = PySequence_Fast_ITEMS(o);
        *a = PyLong_AsLongLong(items[0]);
        *b = PyLong_AsLongLong(items[1]);
        if (PyErr_Occurred()) {
            PyErr_Clear();
            fine = false;
        }
    }
    // three numbers, or None: no neuron
    bool lif(Py_ssize_t i, Lif* out) {
        PyObject* o = v[i];
        *out = {1.0, 0.0, 2.0};
        if (o == Py_None) return false;
        if ((!PyList_Check(o) && !PyTuple_Check(o)) || PySequence_Fast_GET_SIZE(o) != 3) {
            fine = false;
            return false;
        }
        PyObject** items = PySequence_Fast_ITEMS(o);
        *out = {PyFloat_AsDouble(items[0]), PyFloat_AsDouble(items[1]), PyFloat_AsDouble(items[2])};
        if (PyErr_Occurred()) {
            PyErr_Clear();
            fine = false;
        }
        return true;
    }
    at::ScalarType dtype(Py_ssize_t i) {
        if (!THPDtype_Check(v[i])) {
            fine = false;
            return at::kFloat;
        }
        return reinterpret_cast<THPDtype*>(v[i])->scalar_type;
    }
};

// One operand in an internal layout: its tensor and T, N, C, H, W.
struct Frames {
    const Tensor* data;
    int layout;
    bool shared;
    int T, N, C, H, W;
    const void* steps[kMaxSteps];

    // reads arguments i ... i + 7: data, layout, shared, T, N, C, H, W
    bool read(Args& a, Key& key, Py_ssize_t i) {
        data = a.tensor(i);
        layout = static_cast<int>(a.number(i + 1));
        shared = a.number(i + 2) != 0;
        T = static_cast<int>(a.number(i + 3));
        N = static_cast<int>(a.number(i + 4));
        C = static_cast<int>(a.number(i + 5));
        H = static_cast<int>(a.number(i + 6));
        W = static_cast<int>(a.number(i + 7));
        if (!a.fine) return false;
        key.tensor(*data);
        for (int64_t x : {layout, static_cast<int>(shared), T, N, C, H, W}) key.add(x);
        if (!key.plain || T < 1 || T > kMaxSteps || data->dim() < 1) return key.plain = false;
        const char* base = static_cast<const char*>(data->data_ptr());
        const int64_t bytes = shared ? 0 : data->stride(0) * static_cast<int64_t>(data->element_size());
        for (int t = 0; t < T; ++t) steps[t] = base + t * bytes;
        return true;
    }
};

Tensor empty_frames(int layout, int64_t T, int64_t N, int64_t C, int64_t H, int64_t W, at::ScalarType dtype, const Tensor& like) {
    const int64_t c8 = (C + 7) / 8;
    if (layout == SNNF_LAYOUT_BITS) return empty({T, N, c8, H, W}, at::kByte, like);
    if (layout == SNNF_LAYOUT_C8) return empty({T, N, c8, H, W, 8}, dtype, like);
    return empty({T, N, C, H, W}, dtype, like);
}

int64_t step_bytes(const Tensor& t) { return t.stride(0) * static_cast<int64_t>(t.element_size()); }

PyObject* none() { Py_RETURN_NONE; }

// Runs `body` without the interpreter lock: other Python threads go on while it allocates and launches.
template <typename Body>
bool unlocked(Body&& body) {
    py::gil_scoped_release nogil;
    return body();
}

// The answer of a convolution or pool: (output data, channels, Ho, Wo, route, membrane or None).
PyObject* frames_answer(const Tensor& out, int64_t channels, int64_t ho, int64_t wo, int route, const Tensor& v) {
    PyObject* tuple = PyTuple_New(6);
    PyTuple_SET_ITEM(tuple, 0, THPVariable_Wrap(out));
    PyTuple_SET_ITEM(tuple, 1, PyLong_FromLongLong(channels));
    PyTuple_SET_ITEM(tuple, 2, PyLong_FromLongLong(ho));
    PyTuple_SET_ITEM(tuple, 3, PyLong_FromLongLong(wo));
    PyTuple_SET_ITEM(tuple, 4, PyLong_FromLong(route));
    if (v.defined()) {
        PyTuple_SET_ITEM(tuple, 5, THPVariable_Wrap(v));
    } else {
        Py_INCREF(Py_None);
        PyTuple_SET_ITEM(tuple, 5, Py_None);
    }
    return tuple;
}

// Common end of the three convolution forms: what is known, or what is to be remembered.
bool proceed(Attempt& key, const Args& a, int64_t learnt) {
    if (!a.fine || !key.plain) return false;
    if (learnt >= 0) {
        Plan plan;
        plan.native = true;
        plan.route = static_cast<int>(learnt);
        remember(key, plan);
        return false;
    }
    return key.known();
}

PyObject* guarded(PyObject* (*body)(Args&), PyObject* const* args, Py_ssize_t n, Py_ssize_t expected) {
    if (g_pack == nullptr) {
        PyErr_SetString(PyExc_RuntimeError, "snnf dispatch: not connected to the Python implementations");
        return nullptr;
    }
    if (n != expected) {
        PyErr_SetString(PyExc_TypeError, "snnf dispatch: wrong number of arguments");
        return nullptr;
    }
    try {
        PyObject* answer = run_native([&] {
            Args a{args, n};
            return body(a);
        });
        return answer != nullptr || PyErr_Occurred() ? answer : none();
    } catch (py::error_already_set& e) {
        e.restore();
        return nullptr;
    }
}

// data, layout, shared, T, N, C, H, W, dtype, weight, bias, stride, padding, lif, residual data | None, residual layout,
// residual C, residual H, residual W, out layout, want_v, learnt
PyObject* blocked_conv(Args& a) {
    Attempt key;
    key.add(static_cast<int64_t>(kBlockedConv));
    Frames x;
    if (!x.read(a, key, 0)) return none();
    const at::ScalarType dtype = a.dtype(8);
    const Tensor *w = a.tensor(9), *b = a.tensor(10);
    int64_t sh = 1, sw = 1, ph = 0, pw = 0;
    a.pair(11, &sh, &sw);
    a.pair(12, &ph, &pw);
    Lif lif;
    const bool neuron = a.lif(13, &lif);
    const bool residual = a.v[14] != Py_None;
    const Tensor* r = residual ? a.tensor(14) : nullptr;
    const int res_layout = residual ? static_cast<int>(a.number(15)) : 0;
    const int out_layout = static_cast<int>(a.number(19));
    const bool want_v = a.number(20) != 0;
    const int64_t learnt = a.number(21);
    if (!a.fine) return none();
    key.tensor(*w);
    key.tensor(*b);
    for (int64_t k : {static_cast<int64_t>(dtype), sh, sw, ph, pw, static_cast<int64_t>(neuron), static_cast<int64_t>(out_layout),
                      static_cast<int64_t>(want_v), static_cast<int64_t>(residual)})
        key.add(k);
    key.add(lif.v_threshold);
    key.add(lif.v_reset);
    key.add(lif.tau);
    if (residual) {
        key.tensor(*r);
        for (Py_ssize_t i = 15; i < 19; ++i) key.add(a.number(i));
    }
    if (!proceed(key, a, learnt)) return none();
    const int64_t cout = w->size(0), kh = w->size(2), kw = w->size(3);
    const int64_t ho = (x.H + 2 * ph - kh) / sh + 1, wo = (x.W + 2 * pw - kw) / sw + 1;
    const int route = key.plan.route;
    Tensor out, v;
    const bool ran = unlocked([&] {
        const hipStream_t stream = stream_of(*x.data);
        out = empty_frames(out_layout, x.T, x.N, cout, ho, wo, dtype, *x.data);
        int status;
        if (route & kRoutePlane) {
            Tensor matrix, row;
            plane_matrix(*w, *b, x.H, x.W, ph, pw, &matrix, &row);
            const int64_t fin = static_cast<int64_t>(x.C) * x.H * x.W, fout = cout * x.H * x.W;
            const Workspace space = split_workspace(*x.data, stream, x.T, x.N, fin, fout);
            const bool bits = x.layout == SNNF_LAYOUT_BITS;
            status = snnf_linear_lif_bits(x.steps, bits ? 1 : 0, x.T, x.N, static_cast<int>(fin), bits ? fin / 8 : fin, code_of(dtype), matrix.data_ptr(),
                                          row.data_ptr(), static_cast<int>(fout), nullptr, out.data_ptr(), step_bytes(out), nullptr,
                                          static_cast<float>(lif.v_threshold), static_cast<float>(lif.v_reset), static_cast<float>(lif.tau),
                                          space.data, space.bytes, stream);
        } else {
            const Tensor packed = packed_weight(*w, *b, dtype);
            const void* rs[kMaxSteps];
            if (residual) packed_steps(*r, x.T, rs);
            if (route & kAllocateV) v = empty({x.N, cout, ho, wo}, at::kFloat, *x.data);
            status = snnf_conv_lif_blocked(x.steps, x.layout, residual ? rs : nullptr, res_layout, x.T, x.N, x.C, x.H, x.W, code_of(dtype),
                                           packed.data_ptr(), static_cast<int>(cout), static_cast<int>(kh), static_cast<int>(kw),
                                           static_cast<int>(sh), static_cast<int>(sw), static_cast<int>(ph), static_cast<int>(pw), nullptr,
                                           out.data_ptr(), out_layout, step_bytes(out), v.defined() ? v.data_ptr() : nullptr, neuron ? 1 : 0,
                                           static_cast<float>(lif.v_threshold), static_cast<float>(lif.v_reset), static_cast<float>(lif.tau), stream);
        }
        return status == 0;
    });
    return ran ? frames_answer(out, cout, ho, wo, route, route & kReturnV ? v : Tensor()) : none();
}

// data, layout, shared, T, N, C, H, W, dtype, weight, bias, padding, lif, shortcut: data, layout, shared, T, N, C, H, W, weight, bias,
// stride, out layout, want_v, learnt
PyObject* blocked_shortcut(Args& a) {
    Attempt key;
    key.add(static_cast<int64_t>(kBlockedShortcut));
    Frames x, s;
    if (!x.read(a, key, 0) || !s.read(a, key, 13)) return none();
    const at::ScalarType dtype = a.dtype(8);
    const Tensor *w = a.tensor(9), *b = a.tensor(10), *sw_ = a.tensor(21), *sb = a.tensor(22);
    int64_t ph = 0, pw = 0, ssh = 1, ssw = 1;
    a.pair(11, &ph, &pw);
    a.pair(23, &ssh, &ssw);
    Lif lif;
    const bool neuron = a.lif(12, &lif);
    const int out_layout = static_cast<int>(a.number(24));
    const bool want_v = a.number(25) != 0;
    const int64_t learnt = a.number(26);
    if (!a.fine) return none();
    for (const Tensor* t : {w, b, sw_, sb}) key.tensor(*t);
    for (int64_t k : {static_cast<int64_t>(dtype), ph, pw, ssh, ssw, static_cast<int64_t>(neuron), static_cast<int64_t>(out_layout),
                      static_cast<int64_t>(want_v)})
        key.add(k);
    key.add(lif.v_threshold);
    key.add(lif.v_reset);
    key.add(lif.tau);
    if (!proceed(key, a, learnt)) return none();
    const int64_t cout = w->size(0);
    const int route = key.plan.route;
    Tensor out, v;
    const bool ran = unlocked([&] {
        const Tensor packed = packed_weight(*w, *b, dtype), packed_sc = packed_weight(*sw_, *sb, dtype);
        out = empty_frames(out_layout, x.T, x.N, cout, x.H, x.W, dtype, *x.data);
        if (route & kAllocateV) v = empty({x.N, cout, x.H, x.W}, at::kFloat, *x.data);
        return snnf_conv_lif_blocked_shortcut(x.steps, s.steps, x.T, x.N, x.C, x.H, x.W, code_of(dtype), packed.data_ptr(), static_cast<int>(cout),
                                              static_cast<int>(w->size(2)), static_cast<int>(w->size(3)), static_cast<int>(ph), static_cast<int>(pw), s.C,
                                              s.H, s.W, static_cast<int>(ssh), static_cast<int>(ssw), packed_sc.data_ptr(), nullptr, out.data_ptr(),
                                              out_layout, step_bytes(out), v.defined() ? v.data_ptr() : nullptr, neuron ? 1 : 0,
                                              static_cast<float>(lif.v_threshold), static_cast<float>(lif.v_reset), static_cast<float>(lif.tau),
                                              stream_of(*x.data)) == 0;
    });
    return ran ? frames_answer(out, cout, x.H, x.W, route, route & kReturnV ? v : Tensor()) : none();
}

// data, layout, shared, T, N, C, H, W, dtype, weight, bias, stride, padding, lif, want_v, learnt
PyObject* blocked_avgpool(Args& a) {
    Attempt key;
    key.add(static_cast<int64_t>(kBlockedAvgPool));
    Frames x;
    if (!x.read(a, key, 0)) return none();
    const at::ScalarType dtype = a.dtype(8);
    const Tensor *w = a.tensor(9), *b = a.tensor(10);
    int64_t sh = 1, sw = 1, ph = 0, pw = 0;
    a.pair(11, &sh, &sw);
    a.pair(12, &ph, &pw);
    Lif lif;
    if (!a.lif(13, &lif)) return none();
    const bool want_v = a.number(14) != 0;
    const int64_t learnt = a.number(15);
    if (!a.fine) return none();
    key.tensor(*w);
    key.tensor(*b);
    for (int64_t k : {static_cast<int64_t>(dtype), sh, sw, ph, pw, static_cast<int64_t>(want_v)}) key.add(k);
    key.add(lif.v_threshold);
    key.add(lif.v_reset);
    key.add(lif.tau);
    if (!proceed(key, a, learnt)) return none();
    const int64_t cout = w->size(0), kh = w->size(2), kw = w->size(3);
    const int64_t ho = (x.H + 2 * ph - kh) / sh + 1, wo = (x.W + 2 * pw - kw) / sw + 1;
    const int route = key.plan.route;
    Tensor out, v;
    const bool ran = unlocked([&] {
        const Tensor packed = packed_weight(*w, *b, dtype);
        out = empty_frames(SNNF_LAYOUT_C8, x.T, x.N, cout, ho / 2, wo / 2, dtype, *x.data);
        if (route & kAllocateV) v = empty({x.N, cout, ho, wo}, at::kFloat, *x.data);
        return snnf_conv_lif_blocked_avgpool(x.steps, x.layout, x.T, x.N, x.C, x.H, x.W, code_of(dtype), packed.data_ptr(), static_cast<int>(cout),
                                             static_cast<int>(kh), static_cast<int>(kw), static_cast<int>(sh), static_cast<int>(sw), static_cast<int>(ph),
                                             static_cast<int>(pw), out.data_ptr(), step_bytes(out), v.defined() ? v.data_ptr() : nullptr,
                                             static_cast<float>(lif.v_threshold), static_cast<float>(lif.v_reset), static_cast<float>(lif.tau),
                                             stream_of(*x.data)) == 0;
    });
    return ran ? frames_answer(out, cout, ho / 2, wo / 2, route, route & kReturnV ? v : Tensor()) : none();
}

// data, layout, shared, T, N, C, H, W, dtype, kernel, stride, padding, is_max, out layout, learnt
PyObject* blocked_pool(Args& a) {
    Attempt key;
    key.add(static_cast<int64_t>(kBlockedPool));
    Frames x;
    if (!x.read(a, key, 0)) return none();
    const at::ScalarType dtype = a.dtype(8);
    const int64_t k = a.number(9), s = a.number(10), p = a.number(11), is_max = a.number(12), out_layout = a.number(13), learnt = a.number(14);
    for (int64_t v : {static_cast<int64_t>(dtype), k, s, p, is_max, out_layout}) key.add(v);
    if (!proceed(key, a, learnt)) return none();
    const int64_t frames = x.data->size(0), ho = (x.H + 2 * p - k) / s + 1, wo = (x.W + 2 * p - k) / s + 1;
    Tensor out;
    const bool ran = unlocked([&] {
        out = empty_frames(static_cast<int>(out_layout), frames, x.N, x.C, ho, wo, dtype, *x.data);
        return snnf_pool2d_blocked(x.data->data_ptr(), x.layout, out.data_ptr(), static_cast<int>(out_layout), frames * x.N, x.C, x.H, x.W,
                                   static_cast<int>(k), static_cast<int>(s), static_cast<int>(p), is_max != 0 ? 1 : 0, code_of(dtype),
                                   stream_of(*x.data)) == 0;
    });
    return ran ? frames_answer(out, x.C, ho, wo, 0, Tensor()) : none();
}

// data, layout, shared, T, N, C, H, W, dtype, weight, bias | None, scale, learnt
PyObject* blocked_head(Args& a) {
    Attempt key;
    key.add(static_cast<int64_t>(kBlockedHead));
    Frames x;
    if (!x.read(a, key, 0)) return none();
    const at::ScalarType dtype = a.dtype(8);
    const Tensor* w = a.tensor(9);
    const bool biased = a.v[10] != Py_None;
    const Tensor* b = biased ? a.tensor(10) : nullptr;
    const double scale = a.real(11);
    const int64_t learnt = a.number(12);
    if (!a.fine) return none();
    key.tensor(*w);
    key.add(static_cast<int64_t>(dtype));
    key.add(static_cast<int64_t>(biased));
    if (biased) key.tensor(*b);
    if (!proceed(key, a, learnt)) return none();
    Tensor out;
    const bool ran = unlocked([&] {
        out = empty({x.N, w->size(0)}, dtype, *x.data);
        return snnf_spike_pool_linear(x.steps, x.T, x.N, x.C, x.H, x.W, w->data_ptr(), biased ? b->data_ptr() : nullptr, static_cast<int>(w->size(0)),
                                      code_of(dtype), out.data_ptr(), static_cast<float>(scale), stream_of(*x.data)) == 0;
    });
    return ran ? THPVariable_Wrap(out) : none();
}

// x [T, N, C, H, W] dense, weight, bias, stride, padding, learnt: the convolution without a neuron
PyObject* dense_conv_bias(Args& a) {
    Attempt key;
    key.add(static_cast<int64_t>(kDenseConvBias));
    const Tensor *x = a.tensor(0), *w = a.tensor(1), *b = a.tensor(2);
    int64_t sh = 1, sw = 1, ph = 0, pw = 0;
    a.pair(3, &sh, &sw);
    a.pair(4, &ph, &pw);
    const int64_t learnt = a.number(5);
    if (!a.fine) return none();
    for (const Tensor* t : {x, w, b}) key.tensor(*t);
    for (int64_t k : {sh, sw, ph, pw}) key.add(k);
    if (!key.plain || x->dim() != 5 || w->dim() != 4 || x->size(0) > kMaxSteps || !proceed(key, a, learnt)) return none();
    const int64_t T = x->size(0), N = x->size(1), H = x->size(3), W = x->size(4), cout = w->size(0), kh = w->size(2), kw = w->size(3);
    const int64_t ho = (H + 2 * ph - kh) / sh + 1, wo = (W + 2 * pw - kw) / sw + 1;
    const void* steps[kMaxSteps];
    packed_steps(*x, T, steps);
    Tensor out;
    const bool ran = unlocked([&] {
        const Tensor packed = packed_weight(*w, *b, x->scalar_type());
        out = empty({T, N, cout, ho, wo}, x->scalar_type(), *x);
        size_t bytes = snnf_conv_bias_workspace_bytes(static_cast<int>(T), static_cast<int>(N), static_cast<int>(x->size(2)), static_cast<int>(H),
                                                      static_cast<int>(W), code_of(x->scalar_type()), static_cast<int>(cout), static_cast<int>(kh),
                                                      static_cast<int>(kw), static_cast<int>(sh), static_cast<int>(sw), static_cast<int>(ph),
                                                      static_cast<int>(pw), 0);
        const c10::DataPtr workspace = scratch_memory(*x, bytes);
        if (!workspace) bytes = 0;
        return snnf_conv_bias_ws(steps, nullptr, static_cast<int>(T), static_cast<int>(N), static_cast<int>(x->size(2)), static_cast<int>(H), static_cast<int>(W),
                                 code_of(x->scalar_type()), packed.data_ptr(), static_cast<int>(cout), static_cast<int>(kh), static_cast<int>(kw),
                                 static_cast<int>(sh), static_cast<int>(sw), static_cast<int>(ph), static_cast<int>(pw), out.data_ptr(), out.stride(0),
                                 workspace.get(), bytes, stream_of(*x)) == 0;
    });
    return ran ? THPVariable_Wrap(out) : none();
}

// x [..., H, W] dense, is_max, kernel, stride, padding, learnt
PyObject* dense_pool(Args& a) {
    Attempt key;
    key.add(static_cast<int64_t>(kDensePool));
    const Tensor* x = a.tensor(0);
    const int64_t is_max = a.number(1), k = a.number(2), s = a.number(3), p = a.number(4), learnt = a.number(5);
    if (!a.fine) return none();
    key.tensor(*x);
    for (int64_t v : {is_max, k, s, p}) key.add(v);
    if (!key.plain || x->dim() < 3 || !proceed(key, a, learnt)) return none();
    const int64_t H = x->size(-2), W = x->size(-1), ho = (H + 2 * p - k) / s + 1, wo = (W + 2 * p - k) / s + 1;
    c10::SmallVector<int64_t, 6> shape(x->sizes().begin(), x->sizes().end());
    shape[shape.size() - 2] = ho;
    shape[shape.size() - 1] = wo;
    Tensor out;
    const bool ran = unlocked([&] {
        out = empty(shape, x->scalar_type(), *x);
        return snnf_pool2d(x->data_ptr(), out.data_ptr(), x->numel() / (H * W), static_cast<int>(H), static_cast<int>(W), static_cast<int>(k), static_cast<int>(s),
                           static_cast<int>(p), is_max != 0 ? 1 : 0, code_of(x->scalar_type()), stream_of(*x)) == 0;
    });
    return ran ? THPVariable_Wrap(out) : none();
}

PyObject* py_conv(PyObject*, PyObject* const* args, Py_ssize_t n) { return guarded(blocked_conv, args, n, 22); }
PyObject* py_shortcut(PyObject*, PyObject* const* args, Py_ssize_t n) { return guarded(blocked_shortcut, args, n, 27); }
PyObject* py_avgpool(PyObject*, PyObject* const* args, Py_ssize_t n) { return guarded(blocked_avgpool, args, n, 16); }
PyObject* py_pool(PyObject*, PyObject* const* args, Py_ssize_t n) { return guarded(blocked_pool, args, n, 15); }
PyObject* py_head(PyObject*, PyObject* const* args, Py_ssize_t n) { return guarded(blocked_head, args, n, 13); }

PyObject* py_conv_bias(PyObject*, PyObject* const* args, Py_ssize_t n) { return guarded(dense_conv_bias, args, n, 6); }
PyObject* py_dense_pool(PyObject*, PyObject* const* args, Py_ssize_t n) { return guarded(dense_pool, args, n, 6); }

PyMethodDef g_fast_methods[] = {
    {"blocked_conv", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(py_conv)), METH_FASTCALL, nullptr},
    {"blocked_shortcut", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(py_shortcut)), METH_FASTCALL, nullptr},
    {"blocked_avgpool", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(py_avgpool)), METH_FASTCALL, nullptr},
    {"blocked_pool", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(py_pool)), METH_FASTCALL, nullptr},
    {"blocked_head", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(py_head)), METH_FASTCALL, nullptr},
    {"dense_conv_bias", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(py_conv_bias)), METH_FASTCALL, nullptr},
    {"dense_pool", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(py_dense_pool)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

void keep(py::object** slot, py::object value) {
    if (*slot == nullptr) *slot = new py::object();        // lives as long as the process: no destructor after the interpreter
    **slot = std::move(value);
}

}  // namespace

PYBIND11_MODULE(_snnf_dispatch, m) {
    PyModule_AddFunctions(m.ptr(), g_fast_methods);
    m.def("connect", [](py::object slow, py::object pack, py::object plane, py::object workspace) {
        keep(&g_slow, std::move(slow));
        keep(&g_pack, std::move(pack));
        keep(&g_plane, std::move(plane));
        keep(&g_workspace, std::move(workspace));
    });
    m.def("connected", [] { return g_pack != nullptr; });
    m.def("enable", [](bool on) { g_enabled.store(on && g_pack != nullptr); });
    m.def("hits", [] {
        std::lock_guard<std::mutex> lock(g_mutex);
        return g_hits;
    });
    m.def("reset_hits", [] {
        std::lock_guard<std::mutex> lock(g_mutex);
        g_hits.clear();
    });
    m.def("forget_plans", [] {
        std::lock_guard<std::mutex> lock(g_mutex);
        g_plans.clear();
    });
    m.def("forget_weights", [] {
        Released released;
        std::lock_guard<std::mutex> lock(g_mutex);
        while (!g_weights.empty()) drop_weight(g_weights.begin(), &released);
    });
}
