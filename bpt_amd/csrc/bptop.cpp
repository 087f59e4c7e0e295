// bptop — the host side of a call whose plan is known, in native code: checks, plan lookup, allocation, launch, autograd.
//
// A step's kernels take 50 to 300 us, its Python host work took 220 (55 forward, 80 backward, the rest autograd and the hand-over
// of the interpreter lock to autograd's thread and back): the GPU waited for the host in every case but the largest.  Here the
// same work is some microseconds a call, and the backward runs on autograd's thread without the interpreter.
//
// Nothing is decided here.  bpt_amd/graphop.py chooses kernels and builds plans; each time it has done so it leaves what it
// chose in the table below (`remember`), under the index tensors' addresses, sizes and versions, the shape and the type.  The
// plan cache (bpt_amd/plan.py) lets an entry in only while it holds the entry's plans, and drops the entry when it drops one of
// them (`forget`); an entry holds its index tensors too, so that their addresses mean nothing else as long as it stands.
// Changing a switch clears the table.  A call that is not in the table, or has an argument that a check refuses, goes to
// the Python function, which raises, or builds, chooses and remembers.  Every call is checked anew.
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <optional>
#include <unordered_map>
#include <vector>

#include "../../include/bptattn.h"
#include "../../include/bptbuild.h"
#include "../../include/bptplan.h"

namespace py = pybind11;
using at::Tensor;

namespace {

enum Kind { ATTN_FWD = 0, ATTN_BWD = 1, ATTN_FWD_NARROW = 2, ATTN_BWD_NARROW = 3, MM_FWD = 4, MM_BWD = 5, SPMM_FWD = 6, SPMM_BWD = 7, SOFTMAX = 8, REL_FWD = 9, REL_TRAIN = 10 };

constexpr size_t MAX_TENSORS = 9, MAX_EXTRA = 7, MAX_ENTRIES = 512;

struct Key {                          // compared and hashed as bytes: always zeroed first
    int64_t kind, device;
    std::array<int64_t, MAX_TENSORS> ptr, numel, version;
    std::array<int64_t, MAX_EXTRA> extra;
    bool operator==(const Key &o) const { return std::memcmp(this, &o, sizeof(Key)) == 0; }
};
static_assert(sizeof(Key) == 8 * (2 + 3 * MAX_TENSORS + MAX_EXTRA), "no padding");

struct KeyHash {
    size_t operator()(const Key &k) const {
        const auto *w = reinterpret_cast<const uint64_t *>(&k);
        uint64_t h = 0x9E3779B97F4A7C15ull;
        for (size_t i = 0; i < sizeof(Key) / 8; ++i) {
            h ^= w[i];
            h *= 0xBF58476D1CE4E5B9ull;
            h ^= h >> 29;
        }
        return (size_t)h;
    }
};

struct Entry {
    bpt_plan a{}, b{}, c{};
    std::vector<Tensor> more;         // REL_*: the index tensors of the score term (RelTensor)
    std::vector<PyObject *> plans;    // owned: what the structs point into lives as long as the entry
    std::vector<Tensor> index;        // whose addresses the key holds: they are not given to other tensors meanwhile
    std::atomic<bool> used{false};
    ~Entry() {
        if (plans.empty() || !Py_IsInitialized()) return;
        py::gil_scoped_acquire gil;
        for (PyObject *p : plans) Py_DECREF(p);
    }
};
using EntryPtr = std::shared_ptr<Entry>;

std::mutex g_mutex;                   // never held while the interpreter lock is taken
int64_t g_generation = 0;             // (under g_mutex) how often the table was cleared
std::unordered_map<Key, EntryPtr, KeyHash> &table() {
    static auto *t = new std::unordered_map<Key, EntryPtr, KeyHash>();       // (lives on: entries may outlast static destruction)
    return *t;
}

EntryPtr find(const Key &k) {
    std::lock_guard<std::mutex> lock(g_mutex);
    auto it = table().find(k);
    if (it == table().end()) return nullptr;
    it->second->used.store(true, std::memory_order_relaxed);
    return it->second;
}

int dtype_code(at::ScalarType t) { return t == at::kFloat ? BPT_F32 : t == at::kBFloat16 ? BPT_BF16 : t == at::kDouble ? BPT_F64 : -1; }

bool index_ok(const Tensor &t, const at::Device &dev) {
    return t.scalar_type() == at::kLong && t.dim() == 1 && t.is_cuda() && t.device() == dev && t.is_contiguous() && !t.is_inference();
}

bool like(const Tensor &t, const Tensor &q) {
    return t.scalar_type() == q.scalar_type() && t.device() == q.device() && t.is_contiguous();
}

bool float_matrix(const Tensor &t, const at::Device &dev, int64_t rows, int64_t columns) {
    return t.scalar_type() == at::kFloat && t.device() == dev && t.is_contiguous() && t.dim() == 2 && t.size(0) == rows && t.size(1) == columns;
}

// false: an index tensor is not what the kernels take
bool make_key(Key &k, Kind kind, const std::vector<const Tensor *> &index, const at::Device &dev, std::initializer_list<int64_t> extra) {
    std::memset(static_cast<void *>(&k), 0, sizeof(Key));
    k.kind = kind;
    k.device = dev.index();
    size_t i = 0;
    for (const Tensor *t : index) {
        if (!index_ok(*t, dev)) return false;
        k.ptr[i] = reinterpret_cast<int64_t>(t->data_ptr());
        k.numel[i] = t->numel();
        k.version[i++] = (int64_t)t->_version();
    }
    i = 0;
    for (int64_t x : extra) k.extra[i++] = x;
    return true;
}

void *stream_of(const at::Device &dev) { return (void *)c10::hip::getCurrentHIPStream(dev.index()).stream(); }

struct Workspace {
    Tensor t;
    void *ptr = nullptr;
    int64_t bytes = 0;
    Workspace(int op, const bpt_plan *a, const bpt_plan *b, int h, int d, int dt, const Tensor &like) {
        bytes = bpt_workspace_bytes(op, a, b, h, d, dt);
        if (bytes > 0) {
            t = at::empty({bytes}, like.options().dtype(at::kByte));
            ptr = t.data_ptr();
        }
    }
};

// ---- fused attention -------------------------------------------------------------------------------------------------------
struct Shape {
    int64_t nq, nk;
    int h, d, dt;
};

bool attention_shape(const Tensor &q, const Tensor &k, const Tensor &v, double p, Shape &s) {
    if (q.dim() != 3 || k.dim() != 3 || !q.is_cuda() || !q.is_contiguous() || !like(k, q) || !like(v, q)) return false;
    if (k.size(1) != q.size(1) || k.size(2) != q.size(2) || v.sizes() != k.sizes() || !(p >= 0.0 && p < 1.0)) return false;
    s = Shape{q.size(0), k.size(0), (int)q.size(1), (int)q.size(2), dtype_code(q.scalar_type())};
    return s.dt >= 0;
}

std::optional<std::tuple<Tensor, Tensor>> attention_forward_known(const Tensor &col, const Tensor &indptr, const Tensor &eid, const Tensor &indices,
                                                                  const Tensor &q, const Tensor &k, const Tensor &v, double scale, double p,
                                                                  uint64_t seed) {
    Shape s;
    if (!attention_shape(q, k, v, p, s) || indices.sizes() != eid.sizes()) return std::nullopt;
    Key key;
    if (!make_key(key, ATTN_FWD, {&col, &indptr, &eid, &indices}, q.device(), {s.nq, s.nk, s.h, s.d, s.dt, p > 0.0})) return std::nullopt;
    const EntryPtr e = find(key);
    if (!e) return std::nullopt;
    c10::DeviceGuard guard(q.device());
    Tensor o = at::empty_like(q), lse = at::empty({s.nq, s.h}, q.options().dtype(at::kFloat));
    Workspace ws(BPT_OP_ATTN_FWD, &e->a, nullptr, s.h, s.d, s.dt, q);
    const int st = bpt_attention_forward(&e->a, q.data_ptr(), k.data_ptr(), v.data_ptr(), nullptr, o.data_ptr(), (float *)lse.data_ptr(), ws.ptr,
                                         ws.bytes, (float)scale, (float)p, seed, s.h, s.d, s.dt, stream_of(q.device()));
    if (st != BPT_OK) return std::nullopt;                   // (the Python function meets the same status and names it)
    return std::make_tuple(o, lse);
}

using Three = std::tuple<Tensor, Tensor, Tensor>;

std::optional<Three> attention_backward_known(const Tensor &row, const Tensor &indptr_r, const Tensor &eid_r, const Tensor &indices_r,
                                              const Tensor &col, const Tensor &indptr_c, const Tensor &eid_c, const Tensor &indices_c,
                                              const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &o, const Tensor &lse,
                                              const Tensor &d_o, double scale, double p, uint64_t seed) {
    Shape s;
    if (!attention_shape(q, k, v, p, s) || !like(o, q) || !like(d_o, q) || o.sizes() != q.sizes() || d_o.sizes() != q.sizes()) return std::nullopt;
    if (lse.scalar_type() != at::kFloat || lse.device() != q.device() || !lse.is_contiguous() || lse.dim() != 2 || lse.size(0) != s.nq ||
        lse.size(1) != s.h)
        return std::nullopt;
    if (indices_c.sizes() != eid_c.sizes() || indices_r.sizes() != eid_r.sizes() || eid_r.sizes() != eid_c.sizes()) return std::nullopt;
    Key key;
    if (!make_key(key, ATTN_BWD, {&row, &indptr_r, &eid_r, &indices_r, &col, &indptr_c, &eid_c, &indices_c}, q.device(),
                  {s.nq, s.nk, s.h, s.d, s.dt, p > 0.0}))
        return std::nullopt;
    const EntryPtr e = find(key);
    if (!e) return std::nullopt;
    c10::DeviceGuard guard(q.device());
    Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    Workspace ws(BPT_OP_ATTN_BWD_PLAIN, &e->a, &e->b, s.h, s.d, s.dt, q);
    const int st = bpt_attention_backward(&e->a, &e->b, q.data_ptr(), k.data_ptr(), v.data_ptr(), nullptr, o.data_ptr(), d_o.data_ptr(),
                                          (const float *)lse.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), nullptr, ws.ptr, ws.bytes,
                                          (float)scale, (float)p, seed, s.h, s.d, s.dt, stream_of(q.device()));
    if (st != BPT_OK) return std::nullopt;
    return Three{dq, dk, dv};
}

py::object python(const char *name) { return py::module_::import("bpt_amd.graphop").attr(name); }

// Python's exceptions leave autograd's thread as themselves
template <typename F> auto with_python(F &&f) {
    py::gil_scoped_acquire gil;
    try {
        return f();
    } catch (py::error_already_set &e) {
        e.restore();
        python_error err;
        err.persist();
        throw std::move(err);
    }
}

std::tuple<Tensor, Tensor> attention_forward(const Tensor &col, const Tensor &indptr, const Tensor &eid, const Tensor &indices, const Tensor &q,
                                             const Tensor &k, const Tensor &v, double scale, double p, uint64_t seed) {
    auto r = attention_forward_known(col, indptr, eid, indices, q, k, v, scale, p, seed);
    if (!r) r = python("attention_forward")(col, indptr, eid, indices, q, k, v, scale, p, seed).cast<std::tuple<Tensor, Tensor>>();
    return *r;
}

// (its forward runs with the interpreter lock held, its backward without)
struct Attention : torch::autograd::Function<Attention> {
    static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &row, const Tensor &indptr_r, const Tensor &eid_r,
                          const Tensor &indices_r, const Tensor &col, const Tensor &indptr_c, const Tensor &eid_c, const Tensor &indices_c,
                          const Tensor &q, const Tensor &k, const Tensor &v, double scale, double p, int64_t seed) {
        auto r = attention_forward_known(col, indptr_c, eid_c, indices_c, q, k, v, scale, p, (uint64_t)seed);
        if (!r) {                                             // a new graph: both sides' plans at once
            python("prepare_training")(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, p);
            r = attention_forward(col, indptr_c, eid_c, indices_c, q, k, v, scale, p, (uint64_t)seed);
        }
        const auto [o, lse] = *r;
        ctx->save_for_backward({row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, o, lse});
        ctx->saved_data["scale"] = scale;
        ctx->saved_data["p"] = p;
        ctx->saved_data["seed"] = seed;
        return o;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        const auto t = ctx->get_saved_variables();
        const double scale = ctx->saved_data["scale"].toDouble(), p = ctx->saved_data["p"].toDouble();
        const uint64_t seed = (uint64_t)ctx->saved_data["seed"].toInt();
        const Tensor d_o = grads[0].contiguous();
        auto r = attention_backward_known(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], t[9], t[10], t[11], t[12], d_o, scale, p, seed);
        if (!r)
            r = with_python([&] {
                return python("attention_backward")(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], t[9], t[10], t[11], t[12], d_o, scale, p,
                                                    seed).template cast<Three>();
            });
        torch::autograd::variable_list out(14);
        std::tie(out[8], out[9], out[10]) = *r;
        return out;
    }
};

// Through the autograd function also where a tangent of forward-mode differentiation is carried: the function refuses it, the bare
// forward would drop it.
bool differentiated(std::initializer_list<const Tensor *> tensors) {
    for (const Tensor *t : tensors)
        if ((at::GradMode::is_enabled() && t->requires_grad()) || t->_fw_grad(/*level=*/0).defined()) return true;
    return false;
}

// op.BPTAttention with the host work in native code: the same call, the same result
Tensor attention(const Tensor &row, const Tensor &indptr_r, const Tensor &eid_r, const Tensor &indices_r, const Tensor &col, const Tensor &indptr_c,
                 const Tensor &eid_c, const Tensor &indices_c, const Tensor &q, const Tensor &k, const Tensor &v, double scale, double p, uint64_t seed) {
    if (differentiated({&q, &k, &v}))
        return Attention::apply(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, scale, p, (int64_t)seed);
    return std::get<0>(attention_forward(col, indptr_c, eid_c, indices_c, q, k, v, scale, p, seed));
}

// ---- fused attention with heads of fewer than 64 columns, h: the heads it is computed as if padded to -------------------------
// keep: tensors that become copies of q, k, v and of the result (graphop._attention_forward_narrow)
using Copies = std::array<std::optional<Tensor>, 4>;

std::optional<std::tuple<Tensor, Tensor>> narrow_forward_known(const Tensor &col, const Tensor &indptr, const Tensor &eid, const Tensor &indices,
                                                               const Tensor &q, const Tensor &k, const Tensor &v, int h, double scale, double p,
                                                               uint64_t seed, const Copies &keep) {
    Shape s;
    if (!attention_shape(q, k, v, p, s) || indices.sizes() != eid.sizes()) return std::nullopt;
    void *copies[4] = {};
    for (size_t i = 0; i < 4; ++i) {
        if (!keep[i]) continue;
        if (!like(*keep[i], q) || keep[i]->sizes() != (i == 1 || i == 2 ? k : q).sizes()) return std::nullopt;
        copies[i] = keep[i]->data_ptr();
    }
    Key key;
    if (!make_key(key, ATTN_FWD_NARROW, {&col, &indptr, &eid, &indices}, q.device(), {s.nq, s.nk, h, s.d, s.dt, p > 0.0, s.h}))
        return std::nullopt;
    const EntryPtr e = find(key);
    if (!e) return std::nullopt;
    c10::DeviceGuard guard(q.device());
    Tensor o = at::empty_like(q), lse = at::empty({s.nq, h}, q.options().dtype(at::kFloat));
    Workspace ws(BPT_OP_ATTN_FWD, &e->a, nullptr, h, 64, s.dt, q);
    const int st = bpt_attention_forward_narrow_keep(&e->a, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), (float *)lse.data_ptr(), copies,
                                                     s.nq, s.nk, ws.ptr, ws.bytes, (float)scale, (float)p, seed, s.h, s.d, h, s.dt,
                                                     stream_of(q.device()));
    if (st != BPT_OK) return std::nullopt;
    return std::make_tuple(o, lse);
}

std::optional<Three> narrow_backward_known(const Tensor &row, const Tensor &indptr_r, const Tensor &eid_r, const Tensor &indices_r,
                                           const Tensor &col, const Tensor &indptr_c, const Tensor &eid_c, const Tensor &indices_c, const Tensor &q,
                                           const Tensor &k, const Tensor &v, const Tensor &o, const Tensor &lse, const Tensor &d_o, int h,
                                           double scale, double p, uint64_t seed) {
    Shape s;
    if (!attention_shape(q, k, v, p, s) || !like(o, q) || !like(d_o, q) || o.sizes() != q.sizes() || d_o.sizes() != q.sizes()) return std::nullopt;
    if (lse.scalar_type() != at::kFloat || lse.device() != q.device() || !lse.is_contiguous() || lse.dim() != 2 || lse.size(0) != s.nq ||
        lse.size(1) != h)
        return std::nullopt;
    if (indices_c.sizes() != eid_c.sizes() || indices_r.sizes() != eid_r.sizes() || eid_r.sizes() != eid_c.sizes()) return std::nullopt;
    Key key;
    if (!make_key(key, ATTN_BWD_NARROW, {&row, &indptr_r, &eid_r, &indices_r, &col, &indptr_c, &eid_c, &indices_c}, q.device(),
                  {s.nq, s.nk, h, s.d, s.dt, p > 0.0, s.h}))
        return std::nullopt;
    const EntryPtr e = find(key);
    if (!e) return std::nullopt;
    c10::DeviceGuard guard(q.device());
    Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    Workspace ws(BPT_OP_ATTN_BWD, &e->a, &e->b, h, 64, s.dt, q);
    const int st = bpt_attention_backward_narrow(&e->a, &e->b, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_o.data_ptr(),
                                                 (const float *)lse.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), ws.ptr, ws.bytes,
                                                 (float)scale, (float)p, seed, s.h, s.d, h, s.dt, stream_of(q.device()));
    if (st != BPT_OK) return std::nullopt;
    return Three{dq, dk, dv};
}

// a contiguous tensor that starts on 4 bytes, as the kernels' loads need (a bfloat16 view may start on 2)
Tensor rows(const Tensor &x) {
    Tensor y = x.contiguous();
    return y.is_cuda() && (reinterpret_cast<uintptr_t>(y.data_ptr()) & 3) ? y.clone() : y;
}

// Memory for a copy of rows(x) that is nobody else's, where rows(x) is not one already.  A backward needs the rows as the forward saw
// them, and a layer on padded copies let its caller write to q, k, v and o after the forward (an activation or a residual in
// place); so does this one.  The forward's launches fill the copies.
std::optional<Tensor> room_for_copy(const Tensor &x, const Tensor &rows_of_x) {
    if (!rows_of_x.is_alias_of(x)) return std::nullopt;
    return at::empty_like(rows_of_x);
}

// The forward is a call of graphop.attention_forward, as that of the padded copies was: q, k, v stand for the padded shape there.
std::tuple<Tensor, Tensor> narrow_forward(const Tensor &col, const Tensor &indptr, const Tensor &eid, const Tensor &indices, const Tensor &q,
                                          const Tensor &k, const Tensor &v, int64_t h, double scale, double p, int64_t seed, const Copies &keep) {
    const auto meta = at::TensorOptions().dtype(q.dtype()).device(at::kMeta);
    const Tensor qp = at::empty({q.size(0), h, 64}, meta), kp = at::empty({k.size(0), h, 64}, meta);
    py::dict kw;
    kw["narrow"] = py::make_tuple(q, k, v);
    kw["keep"] = py::make_tuple(keep[0], keep[1], keep[2], keep[3]);
    return python("attention_forward")(col, indptr, eid, indices, qp, kp, kp, scale, p, (uint64_t)seed, **kw).cast<std::tuple<Tensor, Tensor>>();
}

bool narrow_known(const Tensor &col, const Tensor &indptr, const Tensor &eid, const Tensor &indices, const Tensor &q, const Tensor &k, int64_t h,
                  double p) {
    Key key;
    return q.is_cuda() && q.dim() == 3 &&
           make_key(key, ATTN_FWD_NARROW, {&col, &indptr, &eid, &indices}, q.device(),
                    {q.size(0), k.size(0), h, q.size(2), dtype_code(q.scalar_type()), p > 0.0, q.size(1)}) &&
           find(key) != nullptr;
}

struct NarrowAttention : torch::autograd::Function<NarrowAttention> {
    static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &row, const Tensor &indptr_r, const Tensor &eid_r,
                          const Tensor &indices_r, const Tensor &col, const Tensor &indptr_c, const Tensor &eid_c, const Tensor &indices_c,
                          const Tensor &q, const Tensor &k, const Tensor &v, int64_t h, double scale, double p, int64_t seed) {
        const Tensor qr = rows(q), kr = rows(k), vr = rows(v);
        if (!narrow_known(col, indptr_c, eid_c, indices_c, qr, kr, h, p))
            python("prepare_training")(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, qr, kr, p, h);
        const Copies keep{room_for_copy(q, qr), room_for_copy(k, kr), room_for_copy(v, vr), at::empty_like(qr)};
        const auto [o, lse] = narrow_forward(col, indptr_c, eid_c, indices_c, qr, kr, vr, h, scale, p, seed, keep);
        ctx->save_for_backward({row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, keep[0].value_or(qr), keep[1].value_or(kr),
                                keep[2].value_or(vr), *keep[3], lse});
        ctx->saved_data["h"] = h;
        ctx->saved_data["scale"] = scale;
        ctx->saved_data["p"] = p;
        ctx->saved_data["seed"] = seed;
        return o;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        const auto t = ctx->get_saved_variables();
        const double scale = ctx->saved_data["scale"].toDouble(), p = ctx->saved_data["p"].toDouble();
        const uint64_t seed = (uint64_t)ctx->saved_data["seed"].toInt();
        const int h = (int)ctx->saved_data["h"].toInt();
        const Tensor d_o = rows(grads[0]);
        auto r = narrow_backward_known(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], t[9], t[10], t[11], t[12], d_o, h, scale, p, seed);
        if (!r)
            r = with_python([&] {
                return python("attention_backward_narrow")(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], t[9], t[10], t[11], t[12], d_o, h,
                                                           scale, p, seed).template cast<Three>();
            });
        torch::autograd::variable_list out(15);
        std::tie(out[8], out[9], out[10]) = *r;
        return out;
    }
};

Tensor attention_narrow(const Tensor &row, const Tensor &indptr_r, const Tensor &eid_r, const Tensor &indices_r, const Tensor &col,
                        const Tensor &indptr_c, const Tensor &eid_c, const Tensor &indices_c, const Tensor &q, const Tensor &k, const Tensor &v,
                        int64_t h, double scale, double p, uint64_t seed) {
    if (differentiated({&q, &k, &v}))
        return NarrowAttention::apply(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, h, scale, p, (int64_t)seed);
    return std::get<0>(narrow_forward(col, indptr_c, eid_c, indices_c, rows(q), rows(k), rows(v), h, scale, p, (int64_t)seed, Copies{}));
}

// ---- fused attention with the relative-position term, in the order of the tile plan's pairs (op.BPTRelAttention) ---------------
// A training pass through the Python function cost the host 157 or 267 us by the process (89 forward and 113 backward at its best), L = 100 as
// L = 8192, whose kernels take 225.  Passes on a machine of the slower kind: L = 100 267 -> 109 us, L = 2048 16 heads bfloat16 277 -> 110, 6 x 50 on padded
// copies, 16 graphs, 444 -> 249; with the gradient's kernel of now L = 8192, k = 8 both ways 905 -> 785, L = 32768 bfloat16 576 -> 515.
// An entry holds what both passes need (REL_FWD: the forward only), and the autograd node keeps the entry: its backward looks nothing up.
enum RelTensor { REL_USED_TYPES = 0, REL_PAIR_TYPES = 1, REL_USED = 2, REL_ROWS_SLOT = 3, REL_NUMBER_SLOT = 4 };

EntryPtr rel_entry(Kind kind, const Tensor &row, const Tensor &indptr_r, const Tensor &eid_r, const Tensor &indices_r, const Tensor &col,
                   const Tensor &indptr_c, const Tensor &eid_c, const Tensor &indices_c, const Tensor &q, const Tensor &k, const Tensor &v, double p,
                   const Tensor &table, const Tensor &etype) {
    Shape s;
    if (!attention_shape(q, k, v, p, s) || indices_c.sizes() != eid_c.sizes() || indices_r.sizes() != eid_r.sizes() || eid_r.sizes() != eid_c.sizes())
        return nullptr;
    if (!like(table, q) || table.dim() != 2 || table.size(1) != s.d) return nullptr;
    Key key;
    if (!make_key(key, kind, {&row, &indptr_r, &eid_r, &indices_r, &col, &indptr_c, &eid_c, &indices_c, &etype}, q.device(),
                  {s.nq, s.nk, s.h, s.d, s.dt, p > 0.0, table.size(0)}))
        return nullptr;
    return find(key);
}

// (o, lse, the term)
std::optional<Three> rel_forward_known(const EntryPtr &e, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &table, double scale, double p,
                                       uint64_t seed) {
    const int h = (int)q.size(1), d = (int)q.size(2), dt = dtype_code(q.scalar_type());
    c10::DeviceGuard guard(q.device());
    void *stream = stream_of(q.device());
    Tensor bias = at::empty({h, e->a.n_edges}, q.options().dtype(at::kFloat));
    const Tensor &types = e->more[REL_USED_TYPES];
    if (bpt_rel_bias_forward_tiles(&e->a, q.data_ptr(), table.data_ptr(), types.const_data_ptr<int32_t>(), types.numel(),
                                   e->more[REL_PAIR_TYPES].const_data_ptr<int32_t>(), bias.data_ptr<float>(), h, d, dt, stream) != BPT_OK)
        return std::nullopt;
    Tensor o = at::empty_like(q), lse = at::empty({q.size(0), h}, q.options().dtype(at::kFloat));
    Workspace ws(BPT_OP_ATTN_FWD, &e->a, nullptr, h, d, dt, q);
    if (bpt_attention_forward(&e->a, q.data_ptr(), k.data_ptr(), v.data_ptr(), bias.data_ptr<float>(), o.data_ptr(), lse.data_ptr<float>(), ws.ptr, ws.bytes,
                              (float)scale, (float)p, seed, h, d, dt, stream) != BPT_OK)
        return std::nullopt;
    return Three{o, lse, bias};
}

std::optional<std::array<Tensor, 4>> rel_backward_known(const EntryPtr &e, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &o,
                                                        const Tensor &lse, const Tensor &bias, const Tensor &table, const Tensor &d_o, double scale,
                                                        double p, uint64_t seed) {
    // (the entry was found for the forward's tensors; a hook on saved tensors may give back others)
    Shape s;
    if (!attention_shape(q, k, v, p, s) || !like(o, q) || !like(d_o, q) || o.sizes() != q.sizes() || d_o.sizes() != q.sizes()) return std::nullopt;
    if (s.nq != e->a.n_rows || s.nk != e->b.n_rows || !float_matrix(lse, q.device(), s.nq, s.h) || !float_matrix(bias, q.device(), s.h, e->a.n_edges) ||
        !like(table, q) || table.dim() != 2 || table.size(0) != e->more[REL_USED].numel() || table.size(1) != s.d)
        return std::nullopt;
    const int h = s.h, d = s.d, dt = s.dt;
    c10::DeviceGuard guard(q.device());
    void *stream = stream_of(q.device());
    Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v), ds = at::empty_like(bias), dtable = at::empty_like(table);
    {
        Workspace ws(BPT_OP_ATTN_BWD, &e->a, &e->b, h, d, dt, q);
        if (bpt_attention_backward(&e->a, &e->b, q.data_ptr(), k.data_ptr(), v.data_ptr(), bias.data_ptr<float>(), o.data_ptr(), d_o.data_ptr(),
                                   lse.data_ptr<float>(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), ds.data_ptr<float>(), ws.ptr, ws.bytes,
                                   (float)scale, (float)p, seed, h, d, dt, stream) != BPT_OK)
            return std::nullopt;
    }
    const Tensor &types = e->more[REL_USED_TYPES];
    const int64_t bytes = std::max<int64_t>(bpt_rel_bias_backward_workspace_bytes(&e->c, types.numel(), h), 16);
    Tensor ws = at::empty({bytes}, q.options().dtype(at::kByte));
    if (bpt_rel_bias_backward(&e->c, ds.data_ptr<float>(), q.data_ptr(), table.data_ptr(), e->more[REL_USED].const_data_ptr<int32_t>(),
                              types.const_data_ptr<int32_t>(), table.size(0), types.numel(), dq.data_ptr(), dtable.data_ptr(), ws.data_ptr(), bytes, h, d, dt,
                              stream) != BPT_OK)
        return std::nullopt;
    return std::array<Tensor, 4>{dq, dk, dv, dtable};
}

struct RelHold : torch::CustomClassHolder {
    EntryPtr e;
    explicit RelHold(EntryPtr x) : e(std::move(x)) {}
};

// (r: what the forward has computed already: a call that the library refuses never becomes a node)
struct RelAttention : torch::autograd::Function<RelAttention> {
    static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &row, const Tensor &indptr_r, const Tensor &eid_r,
                          const Tensor &indices_r, const Tensor &col, const Tensor &indptr_c, const Tensor &eid_c, const Tensor &indices_c,
                          const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &table, const EntryPtr &e, const Three &r, double scale,
                          double p, int64_t seed) {
        const auto &[o, lse, bias] = r;
        ctx->save_for_backward({row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, o, lse, bias, table});
        ctx->saved_data["entry"] = c10::IValue::make_capsule(c10::make_intrusive<RelHold>(e));
        ctx->saved_data["scale"] = scale;
        ctx->saved_data["p"] = p;
        ctx->saved_data["seed"] = seed;
        return o;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        const auto t = ctx->get_saved_variables();
        const double scale = ctx->saved_data["scale"].toDouble(), p = ctx->saved_data["p"].toDouble();
        const uint64_t seed = (uint64_t)ctx->saved_data["seed"].toInt();
        const EntryPtr e = c10::static_intrusive_pointer_cast<RelHold>(ctx->saved_data["entry"].toCapsule())->e;
        const Tensor d_o = grads[0].contiguous();
        auto r = rel_backward_known(e, t[8], t[9], t[10], t[11], t[12], t[13], t[14], d_o, scale, p, seed);
        if (!r)
            r = with_python([&] {
                const auto four = py::module_::import("bpt_amd.op").attr("_rel_backward")(
                                       t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], t[9], t[10], t[11], t[12], t[13], t[14], d_o, scale, p, seed,
                                       e->more[REL_ROWS_SLOT], e->more[REL_NUMBER_SLOT], e->more[REL_USED], e->more[REL_USED_TYPES])
                                      .template cast<std::vector<Tensor>>();
                return std::array<Tensor, 4>{four[0], four[1], four[2], four[3]};
            });
        torch::autograd::variable_list out(17);
        for (int i = 0; i < 4; ++i) out[8 + i] = (*r)[i];
        return out;
    }
};

// op.BPTRelAttention of a call whose plans are known, or None
std::optional<Tensor> rel_attention(const Tensor &row, const Tensor &indptr_r, const Tensor &eid_r, const Tensor &indices_r, const Tensor &col,
                                    const Tensor &indptr_c, const Tensor &eid_c, const Tensor &indices_c, const Tensor &q, const Tensor &k,
                                    const Tensor &v, double scale, double p, uint64_t seed, const Tensor &table, const Tensor &etype) {
    const bool train = differentiated({&q, &k, &v, &table});
    EntryPtr e = rel_entry(REL_TRAIN, row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, p, table, etype);
    if (!e && !train) e = rel_entry(REL_FWD, row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, p, table, etype);
    if (!e) return std::nullopt;
    const auto r = rel_forward_known(e, q, k, v, table, scale, p, seed);
    if (!r) return std::nullopt;
    if (!train) return std::get<0>(*r);
    return RelAttention::apply(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, table, e, *r, scale, p, (int64_t)seed);
}

// ---- the separate operators (modules/op.py:10-58 of the reference) -----------------------------------------------------------
// masked_mm, sparse_softmax and vec_spmm of (n, h, d) rows and (E, h) edge tensors whose plans are known and cover every edge.  A
// training pass through the chain cost the host 325 us in Python, at L = 512 as at L = 8192: three calls of its autograd functions,
// and their backwards on autograd's thread, which has to be handed the interpreter for each.
using Two = std::tuple<Tensor, Tensor>;

bool rows_of_heads(const Tensor &a) { return a.dim() == 3 && a.is_cuda() && a.is_contiguous() && dtype_code(a.scalar_type()) >= 0; }
bool same_heads(const Tensor &b, const Tensor &a) { return b.dim() == 3 && like(b, a) && b.size(1) == a.size(1) && b.size(2) == a.size(2); }
bool per_edge(const Tensor &e, const Tensor &a, const Tensor &eid) {
    return e.dim() == 2 && like(e, a) && e.size(0) == eid.numel() && e.size(1) == a.size(1);
}

std::optional<Tensor> masked_mm_known(const Tensor &row, const Tensor &indptr, const Tensor &eid, const Tensor &indices, const Tensor &a, const Tensor &b) {
    if (!rows_of_heads(a) || !same_heads(b, a) || indices.sizes() != eid.sizes()) return std::nullopt;
    const int h = (int)a.size(1), d = (int)a.size(2), dt = dtype_code(a.scalar_type());
    Key key;
    if (!make_key(key, MM_FWD, {&row, &indptr, &eid, &indices}, a.device(), {a.size(0), b.size(0), h, d, dt})) return std::nullopt;
    const EntryPtr e = find(key);
    if (!e) return std::nullopt;
    c10::DeviceGuard guard(a.device());
    Tensor y = at::empty({eid.numel(), h}, a.options());
    if (bpt_maskedmm_csr_forward(&e->a, a.data_ptr(), b.data_ptr(), y.data_ptr(), h, d, dt, stream_of(a.device())) != BPT_OK) return std::nullopt;
    return y;
}

std::optional<Two> masked_mm_backward_known(const Tensor &row, const Tensor &indptr_r, const Tensor &eid_r, const Tensor &indices_r, const Tensor &col,
                                            const Tensor &indptr_c, const Tensor &eid_c, const Tensor &indices_c, const Tensor &a, const Tensor &b,
                                            const Tensor &dy) {
    if (!rows_of_heads(a) || !same_heads(b, a) || indices_r.sizes() != eid_r.sizes() || indices_c.sizes() != eid_c.sizes() ||
        eid_c.sizes() != eid_r.sizes() || !per_edge(dy, a, eid_r))
        return std::nullopt;
    const int h = (int)a.size(1), d = (int)a.size(2), dt = dtype_code(a.scalar_type());
    Key key;
    if (!make_key(key, MM_BWD, {&row, &indptr_r, &eid_r, &indices_r, &col, &indptr_c, &eid_c, &indices_c}, a.device(), {a.size(0), b.size(0), h, d, dt}))
        return std::nullopt;
    const EntryPtr e = find(key);
    if (!e) return std::nullopt;
    c10::DeviceGuard guard(a.device());
    Tensor da = at::empty_like(a), db = at::empty_like(b);
    Workspace ws(BPT_OP_MASKEDMM_BWD, &e->a, &e->b, h, d, dt, a);
    if (bpt_maskedmm_csr_backward(&e->a, &e->b, a.data_ptr(), b.data_ptr(), dy.data_ptr(), da.data_ptr(), db.data_ptr(), ws.ptr, ws.bytes, h, d, dt,
                                  stream_of(a.device())) != BPT_OK)
        return std::nullopt;
    return Two{da, db};
}

std::optional<Tensor> softmax_known(const Tensor &row, const Tensor &indptr, const Tensor &eid, const Tensor &x, const Tensor *dy) {
    // forward of x, or with dy the backward of the probabilities x
    if (x.dim() != 2 || !x.is_cuda() || !x.is_contiguous() || dtype_code(x.scalar_type()) < 0 || x.size(0) != eid.numel()) return std::nullopt;
    if (dy && (!like(*dy, x) || dy->sizes() != x.sizes())) return std::nullopt;
    const int h = (int)x.size(1), dt = dtype_code(x.scalar_type());
    Key key;
    if (!make_key(key, SOFTMAX, {&row, &indptr, &eid}, x.device(), {h, dt})) return std::nullopt;
    const EntryPtr e = find(key);
    if (!e) return std::nullopt;
    c10::DeviceGuard guard(x.device());
    Tensor y = at::empty_like(x);
    Workspace ws(dy ? BPT_OP_SOFTMAX_BWD : BPT_OP_SOFTMAX_FWD, &e->a, nullptr, h, 1, dt, x);
    const int st = dy ? bpt_sparse_softmax_backward(&e->a, x.data_ptr(), dy->data_ptr(), y.data_ptr(), ws.ptr, ws.bytes, h, dt, stream_of(x.device()))
                      : bpt_sparse_softmax_forward(&e->a, x.data_ptr(), y.data_ptr(), ws.ptr, ws.bytes, h, dt, stream_of(x.device()));
    if (st != BPT_OK) return std::nullopt;
    return y;
}

std::optional<Tensor> vec_spmm_known(const Tensor &row, const Tensor &indptr, const Tensor &eid, const Tensor &indices, const Tensor &w, const Tensor &x) {
    if (!rows_of_heads(x) || !per_edge(w, x, eid) || indices.sizes() != eid.sizes()) return std::nullopt;
    const int h = (int)x.size(1), d = (int)x.size(2), dt = dtype_code(x.scalar_type());
    Key key;
    if (!make_key(key, SPMM_FWD, {&row, &indptr, &eid, &indices}, x.device(), {x.size(0), h, d, dt})) return std::nullopt;
    const EntryPtr e = find(key);
    if (!e) return std::nullopt;
    c10::DeviceGuard guard(x.device());
    Tensor y = at::empty_like(x);
    Workspace ws(BPT_OP_SPMM_FWD, &e->a, nullptr, h, d, dt, x);
    if (bpt_vector_spmm_forward(&e->a, w.data_ptr(), x.data_ptr(), y.data_ptr(), ws.ptr, ws.bytes, h, d, dt, stream_of(x.device())) != BPT_OK)
        return std::nullopt;
    return y;
}

std::optional<Two> vec_spmm_backward_known(const Tensor &row, const Tensor &indptr, const Tensor &eid, const Tensor &indices, const Tensor &col,
                                           const Tensor &indptr_t, const Tensor &eid_t, const Tensor &indices_t, const Tensor &w, const Tensor &dy,
                                           const Tensor &x) {
    if (!rows_of_heads(x) || !per_edge(w, x, eid) || !same_heads(dy, x) || dy.size(0) != x.size(0) || indices.sizes() != eid.sizes() ||
        indices_t.sizes() != eid_t.sizes() || eid_t.sizes() != eid.sizes())
        return std::nullopt;
    const int h = (int)x.size(1), d = (int)x.size(2), dt = dtype_code(x.scalar_type());
    Key key;
    if (!make_key(key, SPMM_BWD, {&row, &indptr, &eid, &indices, &col, &indptr_t, &eid_t, &indices_t}, x.device(), {x.size(0), h, d, dt})) return std::nullopt;
    const EntryPtr e = find(key);
    if (!e) return std::nullopt;
    c10::DeviceGuard guard(x.device());
    Tensor dw = at::empty_like(w), dx = at::empty_like(x);
    Workspace ws(BPT_OP_SPMM_BWD, &e->a, &e->b, h, d, dt, x);
    if (bpt_vector_spmm_backward(&e->a, &e->b, w.data_ptr(), dy.data_ptr(), x.data_ptr(), dw.data_ptr(), dx.data_ptr(), ws.ptr, ws.bytes, h, d, dt,
                                 stream_of(x.device())) != BPT_OK)
        return std::nullopt;
    return Two{dw, dx};
}

struct MaskedMM : torch::autograd::Function<MaskedMM> {
    static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &row, const Tensor &indptr_r, const Tensor &eid_r,
                          const Tensor &indices_r, const Tensor &col, const Tensor &indptr_c, const Tensor &eid_c, const Tensor &indices_c,
                          const Tensor &a, const Tensor &b) {
        ctx->save_for_backward({row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, a, b});
        auto r = masked_mm_known(row, indptr_r, eid_r, indices_r, a, b);
        if (!r) {                                             // a new graph: both sides' plans at once
            python("prepare_products")(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, a, b);
            r = python("maskedmm_csr_forward")(row, indptr_r, eid_r, indices_r, a, b).cast<Tensor>();
        }
        return *r;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        const auto t = ctx->get_saved_variables();
        const Tensor dy = grads[0].contiguous();
        auto r = masked_mm_backward_known(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], t[9], dy);
        if (!r)
            r = with_python([&] {
                const auto two = python("maskedmm_csr_backward")(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], t[9], dy,
                                                                       py::arg("_native_call") = true)
                                     .template cast<std::vector<Tensor>>();
                return Two{two[0], two[1]};
            });
        torch::autograd::variable_list out(10);
        std::tie(out[8], out[9]) = *r;
        return out;
    }
};

struct EdgeSoftmax : torch::autograd::Function<EdgeSoftmax> {
    static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &row, const Tensor &indptr, const Tensor &eid, const Tensor &x) {
        auto y = softmax_known(row, indptr, eid, x, nullptr);
        if (!y) y = python("sparse_softmax_forward")(row, indptr, eid, x, py::arg("_native_call") = true).cast<Tensor>();
        ctx->save_for_backward({row, indptr, eid, *y});
        return *y;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        const auto t = ctx->get_saved_variables();
        const Tensor dy = grads[0].contiguous();
        auto dx = softmax_known(t[0], t[1], t[2], t[3], &dy);
        if (!dx)
            dx = with_python([&] {
                return python("sparse_softmax_backward")(t[0], t[1], t[2], t[3], dy, py::arg("_native_call") = true).template cast<Tensor>();
            });
        return {Tensor(), Tensor(), Tensor(), *dx};
    }
};

struct VecSpmm : torch::autograd::Function<VecSpmm> {
    static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &row, const Tensor &indptr, const Tensor &eid, const Tensor &indices,
                          const Tensor &col, const Tensor &indptr_t, const Tensor &eid_t, const Tensor &indices_t, const Tensor &w, const Tensor &x) {
        ctx->save_for_backward({row, indptr, eid, indices, col, indptr_t, eid_t, indices_t, w, x});
        auto y = vec_spmm_known(row, indptr, eid, indices, w, x);
        if (!y) y = python("vector_spmm_forward")(row, indptr, eid, indices, w, x, py::arg("_native_call") = true).cast<Tensor>();
        return *y;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        const auto t = ctx->get_saved_variables();
        const Tensor dy = grads[0].contiguous();
        auto r = vec_spmm_backward_known(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], dy, t[9]);
        if (!r)
            r = with_python([&] {
                const auto two = python("vector_spmm_backward")(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], dy, t[9],
                                                                       py::arg("_native_call") = true)
                                     .template cast<std::vector<Tensor>>();
                return Two{two[0], two[1]};
            });
        torch::autograd::variable_list out(10);
        std::tie(out[8], out[9]) = *r;
        return out;
    }
};

Tensor masked_mm(const Tensor &row, const Tensor &indptr_r, const Tensor &eid_r, const Tensor &indices_r, const Tensor &col, const Tensor &indptr_c,
                 const Tensor &eid_c, const Tensor &indices_c, const Tensor &a, const Tensor &b) {
    if (differentiated({&a, &b})) return MaskedMM::apply(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, a, b);
    auto y = masked_mm_known(row, indptr_r, eid_r, indices_r, a, b);
    if (!y) {
        python("prepare_products")(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, a, b);
        y = python("maskedmm_csr_forward")(row, indptr_r, eid_r, indices_r, a, b).cast<Tensor>();
    }
    return *y;
}

Tensor sparse_softmax(const Tensor &row, const Tensor &indptr, const Tensor &eid, const Tensor &x) {
    if (differentiated({&x})) return EdgeSoftmax::apply(row, indptr, eid, x);
    auto y = softmax_known(row, indptr, eid, x, nullptr);
    if (!y) y = python("sparse_softmax_forward")(row, indptr, eid, x, py::arg("_native_call") = true).cast<Tensor>();
    return *y;
}

Tensor vec_spmm(const Tensor &row, const Tensor &indptr, const Tensor &eid, const Tensor &indices, const Tensor &col, const Tensor &indptr_t,
                const Tensor &eid_t, const Tensor &indices_t, const Tensor &w, const Tensor &x) {
    if (differentiated({&w, &x})) return VecSpmm::apply(row, indptr, eid, indices, col, indptr_t, eid_t, indices_t, w, x);
    auto y = vec_spmm_known(row, indptr, eid, indices, w, x);
    if (!y) y = python("vector_spmm_forward")(row, indptr, eid, indices, w, x, py::arg("_native_call") = true).cast<Tensor>();
    return *y;
}

// ---- tile plans ---------------------------------------------------------------------------------------------------------------
// The tile plans of one side of a graph or of both (the second linked to the first: what a training step needs), built in shared
// launches.  One wait, for the counts; the caller waits for the finished plans before anybody else may use them.
struct SideIn {
    Tensor row, indptr, eid, indices;
    int64_t n_rows, n_index;
    int seg_len, by_mask;
};
constexpr int PAD_ENTRIES = 8;

void check_build(int st, const char *what) {
    if (st != BPT_OK) throw std::runtime_error(std::string(what) + ": status " + std::to_string(st));
}

void wait_for(void *stream) {
    py::gil_scoped_release nogil;
    check_build(bpt_build_wait(stream), "bpt_build_wait");
}

// graphbuilder.get_csrs_device behind its checks: the five arrays of the out- and of the in-side, and (error, units) of each
std::tuple<std::vector<Tensor>, std::vector<Tensor>, std::vector<int>> build_csrs(const Tensor &src, const Tensor &dst, int64_t n, int chunk) {
    const int64_t E = src.numel();
    c10::DeviceGuard guard(src.device());
    int64_t bounds[2];
    check_build(bpt_csr_device_bounds(E, n, chunk, bounds), "bpt_csr_device_bounds");
    std::vector<Tensor> side[2];
    int64_t *ptr[2][5];
    for (int i = 0; i < 2; ++i) {
        int j = 0;
        for (int64_t size : {n + 1, E, E, bounds[0], bounds[0] + 1}) {
            side[i].push_back(at::empty({std::max<int64_t>(size, 1)}, src.options()));
            ptr[i][j] = side[i][j].data_ptr<int64_t>();
            ++j;
        }
    }
    Tensor ws = at::empty({bounds[1]}, src.options().dtype(at::kByte));
    Tensor info = at::empty({4}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));      // (written by the last kernel: no copy to wait for)
    void *stream = stream_of(src.device());
    check_build(bpt_build_csrs_device(src.const_data_ptr<int64_t>(), dst.const_data_ptr<int64_t>(), E, n, chunk, ptr[0], ptr[1],
                                      info.data_ptr<int32_t>(), ws.data_ptr(), bounds[1], stream),
                "bpt_build_csrs_device");
    wait_for(stream);
    const int32_t *c = info.data_ptr<int32_t>();
    return {side[0], side[1], {c[0], c[1], c[2], c[3]}};
}

// how many rows of one or two CSR sides (their units' rows and pointers) have edges; one wait
std::vector<int64_t> count_rows(const std::vector<std::tuple<Tensor, Tensor>> &in) {
    const int n = (int)in.size();
    if (n < 1 || n > 2) throw std::invalid_argument("one or two sides");
    const at::Device dev = std::get<0>(in[0]).device();
    const int64_t *row[2] = {}, *indptr[2] = {};
    int64_t units[2] = {};
    for (int i = 0; i < n; ++i) {
        const auto &[r, p] = in[i];
        if (!index_ok(r, dev) || !index_ok(p, dev) || p.numel() != r.numel() + 1)
            throw std::invalid_argument("row and indptr: contiguous int64 on one GPU, one indptr more than rows");
        row[i] = r.const_data_ptr<int64_t>();
        indptr[i] = p.const_data_ptr<int64_t>();
        units[i] = r.numel();
    }
    c10::DeviceGuard guard(dev);
    Tensor parts = at::empty({n * BPT_COUNT_PARTS}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
    void *stream = stream_of(dev);
    check_build(bpt_build_count_rows(row, indptr, units, n, parts.data_ptr<int32_t>(), stream), "bpt_build_count_rows");
    wait_for(stream);
    std::vector<int64_t> counts(n, 0);
    for (int i = 0; i < n * BPT_COUNT_PARTS; ++i) counts[i / BPT_COUNT_PARTS] += parts.data_ptr<int32_t>()[i];
    return counts;
}

// The arrays of a side's base plan, for the largest numbers of items and split rows that its sizes allow
std::vector<Tensor> base_arrays(const bpt_build_side &s, const at::TensorOptions &i32) {
    const int64_t E = std::max<int64_t>(s.n_edges, 1), items = std::max<int64_t>(s.n_rows + s.n_edges / s.seg_len, 1);
    return {at::empty({s.n_rows + 1}, i32), at::empty({E}, i32), at::empty({E}, i32), at::empty({items, 4}, i32), at::empty({items, 2}, i32),
            at::empty({std::max<int64_t>(s.n_edges / (s.seg_len + 1), 1), 3}, i32), at::empty({16}, i32)};
}
void point_at(bpt_build_side &s, const std::vector<Tensor> &base, const Tensor &row, const Tensor &indptr, const Tensor &eid, const Tensor &indices) {
    s.row = row.const_data_ptr<int64_t>(); s.indptr_units = indptr.const_data_ptr<int64_t>();
    s.eid = eid.const_data_ptr<int64_t>(); s.indices = indices.const_data_ptr<int64_t>();
    int32_t **to[7] = {&s.rowptr, &s.idx32, &s.eid32, &s.items, &s.item_bounds, &s.heavy, &s.info};
    for (int j = 0; j < 7; ++j) *to[j] = base[j].data_ptr<int32_t>();
}

// The base plans of one or two sides, in one launch where they are small and with one wait: per side its info block and base arrays, or None where
// an array is not what the kernels read.
py::object build_plans(const std::vector<std::tuple<Tensor, Tensor, Tensor, Tensor, int64_t, int64_t, int>> &in) {
    const int n = (int)in.size();
    if (n < 1 || n > 2) throw std::invalid_argument("one or two sides");
    const at::Device dev = std::get<2>(in[0]).device();
    for (const auto &[row, indptr, eid, indices, n_rows, n_index, seg] : in)
        for (const Tensor *t : {&row, &indptr, &eid, &indices})
            if (!index_ok(*t, dev)) return py::none();
    c10::DeviceGuard guard(dev);
    const auto i32 = at::TensorOptions().dtype(at::kInt).device(dev);
    bpt_build_side sides[2] = {};
    std::vector<std::vector<Tensor>> base(n);
    for (int i = 0; i < n; ++i) {
        const auto &[row, indptr, eid, indices, n_rows, n_index, seg] = in[i];
        bpt_build_side &s = sides[i];
        s.n_units = row.numel(); s.n_edges = eid.numel(); s.n_rows = n_rows; s.n_index_nodes = n_index; s.seg_len = seg;
        if (indptr.numel() != s.n_units + 1 || indices.numel() != s.n_edges || n_rows < 0 || n_index < 0 || seg < 1) return py::none();
    }
    int64_t bytes = 0;
    if (bpt_build_plans_bounds(sides, n, &bytes) != BPT_OK) return py::none();
    for (int i = 0; i < n; ++i) {
        const auto &[row, indptr, eid, indices, n_rows, n_index, seg] = in[i];
        base[i] = base_arrays(sides[i], i32);
        point_at(sides[i], base[i], row, indptr, eid, indices);
    }
    Tensor ws = at::empty({bytes}, i32.dtype(at::kByte));
    Tensor infos = at::empty({16 * n}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
    void *stream = stream_of(dev);
    check_build(bpt_build_plans(sides, n, infos.data_ptr<int32_t>(), ws.data_ptr(), bytes, stream), "bpt_build_plans");
    wait_for(stream);
    py::list result;
    for (int i = 0; i < n; ++i) {
        const int32_t *c = infos.data_ptr<int32_t>() + 16 * i;
        result.append(py::make_tuple(std::vector<int>(c, c + 16), base[i]));
    }
    return result;
}

// None where the short form does not build them; else (per side: its info block, base arrays, group arrays; the pair mapping of
// the second side).  A side's info block holds an error where its arrays are malformed (then nothing else is valid).
py::object build_tile_plans(const std::vector<std::tuple<Tensor, Tensor, Tensor, Tensor, int64_t, int64_t, int, int>> &in) {
    const int n = (int)in.size();
    if (n < 1 || n > 2) throw std::invalid_argument("one or two sides");
    const at::Device dev = std::get<2>(in[0]).device();
    for (const auto &[row, indptr, eid, indices, n_rows, n_index, seg, mask] : in)
        for (const Tensor *t : {&row, &indptr, &eid, &indices})
            if (!index_ok(*t, dev)) return py::none();
    c10::DeviceGuard guard(dev);
    const auto i32 = at::TensorOptions().dtype(at::kInt).device(dev);
    bpt_build_side sides[2] = {};
    std::vector<std::vector<Tensor>> base(n), groups(n);
    for (int i = 0; i < n; ++i) {
        const auto &[row, indptr, eid, indices, n_rows, n_index, seg, mask] = in[i];
        const int64_t E = eid.numel(), U = row.numel();
        if (indptr.numel() != U + 1 || indices.numel() != E || n_rows < 0 || n_index < 0 || seg < 1) return py::none();
        bpt_build_side &s = sides[i];
        s.n_units = U; s.n_edges = E; s.n_rows = n_rows; s.n_index_nodes = n_index; s.seg_len = seg; s.by_mask = mask;
    }
    int64_t bytes = 0;
    if (bpt_build_tiles_bounds(sides, n, &bytes) != BPT_OK) return py::none();
    for (int i = 0; i < n; ++i) {
        const auto &[row, indptr, eid, indices, n_rows, n_index, seg, mask] = in[i];
        base[i] = base_arrays(sides[i], i32);
        point_at(sides[i], base[i], row, indptr, eid, indices);
    }
    Tensor ws = at::empty({bytes}, i32.dtype(at::kByte));
    Tensor counts = at::empty({32 * n}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
    void *stream = stream_of(dev);
    check_build(bpt_build_tiles_count(sides, n, counts.data_ptr<int32_t>(), ws.data_ptr(), bytes, stream), "bpt_build_tiles_count");
    wait_for(stream);
    const int32_t *c = counts.data_ptr<int32_t>();
    bool good = true;
    for (int i = 0; i < n; ++i) good = good && c[32 * i] == 0;
    Tensor pairs, number;
    if (good) {
        bpt_build_tiles out[2] = {};
        const bool link = n == 2 && (c[5] & 1) && (c[37] & 1) && sides[0].n_edges == sides[1].n_edges;
        for (int i = 0; i < n; ++i) {
            const int64_t ng = c[32 * i + 16], ne = c[32 * i + 17];
            groups[i] = {at::empty({ng, 16, 2}, i32), at::empty({ng + 1}, i32), at::empty({ne + 1, 4}, i32), at::empty({sides[i].n_edges}, i32),
                         at::empty({(ne + PAD_ENTRIES) * 16}, i32), at::empty({9}, i32), at::empty({16}, i32)};
            int32_t **to[7] = {&out[i].members, &out[i].grp_ptr, &out[i].entries, &out[i].pair_eid, &out[i].grp_eids, &out[i].chunks, &out[i].group_info};
            for (int j = 0; j < 7; ++j) *to[j] = groups[i][j].data_ptr<int32_t>();
        }
        if (link) {
            number = at::empty({std::max<int64_t>(sides[0].n_edges, 1)}, i32);
            pairs = at::empty({groups[1][4].numel()}, i32);
            out[0].number = number.data_ptr<int32_t>();
        }
        check_build(bpt_build_tiles_write(sides, n, c, out, PAD_ENTRIES, link ? pairs.data_ptr<int32_t>() : nullptr, ws.data_ptr(), bytes, stream),
                    "bpt_build_tiles_write");
    }
    py::list result;
    for (int i = 0; i < n; ++i) {
        py::list info;
        for (int j = 0; j < 32; ++j) info.append(c[32 * i + j]);
        result.append(py::make_tuple(info, base[i], groups[i]));
    }
    return py::make_tuple(result, pairs.defined() ? py::cast(pairs) : py::none());
}

// ---- the table ---------------------------------------------------------------------------------------------------------------
// `kind`'s choice for these index tensors and numbers: the bpt_plan structs at the addresses a and b (0: none), which point into
// what `plans` holds.  generation: what generation() said before the choice was begun; a table that was cleared since does not take
// it, since a switch may have changed under it.  True if it was taken.
bool remember_more(int64_t generation, int kind, const std::vector<Tensor> &index, const std::vector<int64_t> &extra, int64_t a, int64_t b, int64_t c,
                   const std::vector<Tensor> &more, py::tuple plans) {
    if (index.empty() || index.size() > MAX_TENSORS || extra.size() > MAX_EXTRA || !index[0].defined() || !index[0].is_cuda() || !a) return false;
    std::vector<const Tensor *> ptrs;
    for (const Tensor &t : index) ptrs.push_back(&t);
    Key key;
    if (!make_key(key, (Kind)kind, ptrs, index[0].device(), {})) return false;
    std::copy(extra.begin(), extra.end(), key.extra.begin());
    auto e = std::make_shared<Entry>();
    std::memcpy(&e->a, reinterpret_cast<const void *>(a), sizeof(bpt_plan));
    if (b) std::memcpy(&e->b, reinterpret_cast<const void *>(b), sizeof(bpt_plan));
    if (c) std::memcpy(&e->c, reinterpret_cast<const void *>(c), sizeof(bpt_plan));
    e->more = more;
    for (auto p : plans) e->plans.push_back(p.inc_ref().ptr());
    e->index = index;
    e->used.store(true);
    std::vector<EntryPtr> dropped;                           // (destroyed behind the lock)
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        if (generation != g_generation) return false;
        if (table().size() >= MAX_ENTRIES) {
            for (auto &kv : table()) dropped.push_back(std::move(kv.second));
            table().clear();
        }
        EntryPtr &slot = table()[key];
        dropped.push_back(std::move(slot));
        slot = e;
    }
    return true;
}

bool remember(int64_t generation, int kind, const std::vector<Tensor> &index, const std::vector<int64_t> &extra, int64_t a, int64_t b, py::tuple plans) {
    return remember_more(generation, kind, index, extra, a, b, 0, {}, std::move(plans));
}

// the same for the attention with relative positions: c, the plan of the term's gradient, and the term's index tensors in the order of RelTensor
bool remember_rel(int64_t generation, int kind, const std::vector<Tensor> &index, const std::vector<int64_t> &extra, int64_t a, int64_t b, int64_t c,
                  const std::vector<Tensor> &more, py::tuple plans) {
    if (kind != REL_FWD && kind != REL_TRAIN) return false;
    if (more.size() != (kind == REL_FWD ? 2 : 5) || (kind == REL_TRAIN && (!b || !c))) return false;
    for (const Tensor &t : more)
        if (!t.is_cuda() || t.dim() != 1 || !t.is_contiguous()) return false;
    for (RelTensor i : {REL_USED_TYPES, REL_PAIR_TYPES, REL_USED})
        if ((size_t)i < more.size() && more[i].scalar_type() != at::kInt) return false;
    return remember_more(generation, kind, index, extra, a, b, c, more, std::move(plans));
}

// drops what was chosen with this plan object
void forget(py::object plan) {
    std::vector<EntryPtr> dropped;
    std::lock_guard<std::mutex> lock(g_mutex);
    for (auto it = table().begin(); it != table().end();) {
        bool hit = false;
        for (PyObject *p : it->second->plans) hit = hit || p == plan.ptr();
        if (hit) {
            dropped.push_back(std::move(it->second));
            it = table().erase(it);
        } else {
            ++it;
        }
    }
}

void clear() {
    std::vector<EntryPtr> dropped;
    std::lock_guard<std::mutex> lock(g_mutex);
    ++g_generation;
    for (auto &kv : table()) dropped.push_back(std::move(kv.second));
    table().clear();
}

int64_t generation() {
    std::lock_guard<std::mutex> lock(g_mutex);
    return g_generation;
}

// the plan objects whose entries served a call since the last time this was asked
std::vector<py::object> take_used() {
    std::vector<EntryPtr> hit;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        for (auto &kv : table())
            if (kv.second->used.exchange(false)) hit.push_back(kv.second);
    }
    std::vector<py::object> out;
    for (auto &e : hit)
        for (PyObject *p : e->plans) out.push_back(py::reinterpret_borrow<py::object>(p));
    return out;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.attr("ATTN_FWD") = (int)ATTN_FWD;
    m.attr("ATTN_BWD") = (int)ATTN_BWD;
    m.attr("ATTN_FWD_NARROW") = (int)ATTN_FWD_NARROW;
    m.attr("ATTN_BWD_NARROW") = (int)ATTN_BWD_NARROW;
    m.attr("MM_FWD") = (int)MM_FWD;
    m.attr("MM_BWD") = (int)MM_BWD;
    m.attr("SPMM_FWD") = (int)SPMM_FWD;
    m.attr("SPMM_BWD") = (int)SPMM_BWD;
    m.attr("SOFTMAX") = (int)SOFTMAX;
    m.attr("REL_FWD") = (int)REL_FWD;
    m.attr("REL_TRAIN") = (int)REL_TRAIN;
    m.def("masked_mm", &masked_mm);
    m.def("sparse_softmax", &sparse_softmax);
    m.def("vec_spmm", &vec_spmm);
    m.def("attention", &attention);
    m.def("attention_narrow", &attention_narrow);
    m.def("attention_forward_narrow", &narrow_forward_known);
    m.def("attention_forward", &attention_forward_known);
    m.def("attention_backward", &attention_backward_known);
    m.def("build_csrs", &build_csrs);
    m.def("build_plans", &build_plans);
    m.def("build_tile_plans", &build_tile_plans);
    m.def("count_rows", &count_rows);
    m.def("rel_attention", &rel_attention);
    m.def("remember", &remember);
    m.def("remember_rel", &remember_rel);
    m.def("forget", &forget);
    m.def("clear", &clear);
    m.def("generation", &generation);
    m.def("take_used", &take_used);
    m.def("plan_bytes", [] { return (int64_t)sizeof(bpt_plan); });
}
