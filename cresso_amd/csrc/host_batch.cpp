// Host-side bookkeeping of the scalar plan's steady state, in C++.
//
// One optimizer step of a group of many small tensors (the C3 case: 840) is a
// single kernel sequence on the GPU, but the per-step Python work around it
// (checking that the group is unchanged, collecting the fresh grad pointers
// that autograd allocates, advancing every state["step"]) costs about 0.2 us
// per tensor and per item in CPython, which is as long as the GPU step itself.
// BatchGuard does the same checks and writes in one pass over the Python
// objects: gather() verifies each parameter (same object, storage, shape and
// dtype, contiguous), its grad (defined, contiguous, the parameter's shape and
// device, the planned dtype) and its state (the planned dict, tensors, storage
// and step count: the plan holds their addresses) and writes the grad pointers
// into a host array; bump() adds 1 to state["step"].  Any mismatch makes
// gather() return false and the caller rebuilds the plan.
//
// SpectralGuard does the same for a group's spectral tensors: fill() verifies
// each parameter, its grad and every tensor of its state dict again on every
// step and writes their descriptors for the C ABI (in Python about 8 us a
// tensor: a step of 9 convolution weights and 42 small tensors took 648 us on
// the host, as long as on the GPU).
#include <torch/extension.h>

#include <cstdint>
#include <stdexcept>
#include <vector>

#include "../../include/cresso_hip.h"

namespace {

// The version of a dict's contents: a number that no dict has had before,
// new with every change of an entry.  0: this Python keeps none.
uint64_t dict_version(PyObject* d) {
#if PY_VERSION_HEX < 0x030C0000
    return reinterpret_cast<PyDictObject*>(d)->ma_version_tag;
#else
    (void)d;
    return 0;
#endif
}

struct BatchGuard {
    // A planned state tensor and the storage it had at plan time.  The
    // references keep both alive: no other tensor can take their addresses
    // while the guard lives, and the plan's pointers stay valid memory.
    struct Planned {
        at::Tensor tensor;
        c10::Storage storage;
        const void* data;
    };
    // Where in the storage it was, if not all of it, and a field's form.
    struct View {
        const c10::TensorImpl* x;
        int64_t offset, numel;
        caffe2::TypeMeta dtype;
    };
    struct Item {
        py::object param, dict, keys;   // keys: a tuple; the state's planned entries, from planned[first] on
        size_t first;
        const void* pptr;
        std::vector<int64_t> sizes;
        int pdtype, gdtype, device;
        int64_t step0;                // state["step"] at plan time
        mutable uint64_t version;     // the dict's, when its entries were last compared (or written by bump)
    };
    std::vector<Item> items;
    std::vector<Planned> planned;
    std::vector<View> views;
    bool with_state = false;
    int64_t ran = 0;                      // steps since plan time (bump)
    mutable uint64_t state_version = 0;   // the optimizer's state dict's, when its items were last compared

    // states: empty, or one dict per parameter; keys: each state's planned keys.
    BatchGuard(const py::list& ps, const py::list& states, const py::list& keys) {
        const size_t n = ps.size();
        if ((states.size() != 0 && states.size() != n) || keys.size() != states.size())
            throw std::invalid_argument("BatchGuard: one state and its keys per parameter");
        with_state = states.size() != 0;
        items.reserve(n);
        planned.reserve(with_state ? 8 * n : 0);
        for (size_t i = 0; i < n; ++i) {
            PyObject* o = ps[i].ptr();
            if (!THPVariable_Check(o)) throw std::invalid_argument("BatchGuard: parameters must be tensors");
            const at::Tensor& t = THPVariable_Unpack(o);
            const at::Tensor& g = t.grad();
            if (!g.defined()) throw std::invalid_argument("BatchGuard: every parameter needs a grad at plan time");
            // A strong reference: the parameter cannot be freed (and a new
            // object created at its address) while the guard lives, so the
            // identity test is exact.
            Item it{};
            it.param = py::reinterpret_borrow<py::object>(o);
            it.pptr = t.data_ptr();
            it.sizes = t.sizes().vec();
            it.pdtype = static_cast<int>(t.scalar_type());
            it.gdtype = static_cast<int>(g.scalar_type());
            it.device = t.device().index();
            if (with_state) plan_state(it, states[i].ptr(), keys[i].ptr());
            items.push_back(std::move(it));
        }
    }

    static PyObject* step_key() {
        static PyObject* const key = PyUnicode_InternFromString("step");
        return key;
    }

    // state["step"], or -1
    static int64_t step_of(PyObject* st) {
        PyObject* v = PyDict_GetItemWithError(st, step_key());   // borrowed
        const int64_t s = v && PyLong_Check(v) ? PyLong_AsLongLong(v) : -1;
        if (s == -1) PyErr_Clear();
        return s;
    }

    void plan_state(Item& it, PyObject* st, PyObject* keys) {
        if (!PyDict_Check(st) || !PyTuple_Check(keys)) throw std::invalid_argument("BatchGuard: a state must be a dict, its keys a tuple");
        it.dict = py::reinterpret_borrow<py::object>(st);
        it.keys = py::reinterpret_borrow<py::object>(keys);
        it.first = planned.size();
        for (Py_ssize_t k = 0; k < PyTuple_GET_SIZE(keys); ++k) {
            PyObject* v = PyDict_GetItemWithError(st, PyTuple_GET_ITEM(keys, k));   // borrowed
            if (!v && PyErr_Occurred()) throw py::error_already_set();
            if (!v || !THPVariable_Check(v)) throw std::invalid_argument("BatchGuard: a state lacks a planned tensor");
            const at::Tensor& x = THPVariable_Unpack(v);
            planned.push_back(Planned{x, x.storage(), x.storage().data()});
            if (x.numel() != 1 || x.storage().nbytes() != x.itemsize())
                views.push_back(View{x.unsafeGetTensorImpl(), x.storage_offset(), x.numel(), x.dtype()});
        }
        it.step0 = step_of(st);
        if (it.step0 < 0) throw std::invalid_argument("BatchGuard: a state lacks its step count");
        it.version = dict_version(st);
    }

    // Whether a state dict holds the planned tensors and step count.
    bool entries_hold(const Item& it) const {
        const uint64_t version = dict_version(it.dict.ptr());
        if (version != 0 && version == it.version) return true;
        for (Py_ssize_t k = 0; k < PyTuple_GET_SIZE(it.keys.ptr()); ++k) {
            PyObject* v = PyDict_GetItemWithError(it.dict.ptr(), PyTuple_GET_ITEM(it.keys.ptr(), k));   // borrowed
            if (!v && PyErr_Occurred()) throw py::error_already_set();
            if (!v || !THPVariable_Check(v) || !THPVariable_Unpack(v).is_same(planned[it.first + (size_t)k].tensor)) return false;
        }
        if (step_of(it.dict.ptr()) != it.step0 + ran) return false;
        it.version = version;
        return true;
    }

    // Whether the optimizer's state holds what the plan was made from.
    bool states_hold(PyObject* state) const {
        if (!PyDict_Check(state)) return false;
        const uint64_t version = dict_version(state);
        if (version == 0 || version != state_version) {
            for (const Item& it : items) {
                PyObject* st = PyDict_GetItemWithError(state, it.param.ptr());   // borrowed
                if (!st && PyErr_Occurred()) throw py::error_already_set();
                if (st != it.dict.ptr()) return false;
            }
            state_version = version;
        }
        for (const Item& it : items)
            if (!entries_hold(it)) return false;
        for (const Planned& p : planned)
            if (p.tensor.unsafeGetTensorImpl()->unsafe_storage().unsafeGetStorageImpl() != p.storage.unsafeGetStorageImpl() ||
                p.storage.data() != p.data)
                return false;
        for (const View& v : views)
            if (v.x->storage_offset() != v.offset ||
                (v.numel != 1 && (v.x->numel() != v.numel || v.x->dtype() != v.dtype || !v.x->is_contiguous())))
                return false;
        return true;
    }

    // Whether the parameters and, given the optimizer's state, their states
    // are those of plan time.
    bool holds(const py::list& ps, const py::object& state) const {
        if (ps.size() != items.size()) return false;
        for (size_t i = 0; i < items.size(); ++i) {
            const Item& it = items[i];
            if (PyList_GET_ITEM(ps.ptr(), i) != it.param.ptr()) return false;
            const at::Tensor& t = THPVariable_Unpack(it.param.ptr());
            if (t.data_ptr() != it.pptr || static_cast<int>(t.scalar_type()) != it.pdtype ||
                t.sizes() != c10::IntArrayRef(it.sizes) || !t.is_contiguous())
                return false;
        }
        return !with_state || state.is_none() || states_hold(state.ptr());
    }

    // Writes params[i].grad.data_ptr() to out[i]; false if anything differs
    // from plan time (then out is partially written and must not be used).
    bool gather(const py::list& ps, uintptr_t out_addr, const py::object& state) const {
        if (!holds(ps, state)) return false;
        void** out = reinterpret_cast<void**>(out_addr);
        for (size_t i = 0; i < items.size(); ++i) {
            const Item& it = items[i];
            const at::Tensor& t = THPVariable_Unpack(it.param.ptr());
            const at::Tensor& g = t.grad();
            if (!g.defined() || static_cast<int>(g.scalar_type()) != it.gdtype || g.sizes() != t.sizes() ||
                g.device().index() != it.device || !g.device().is_cuda() || g.is_sparse() || !g.is_contiguous())
                return false;
            out[i] = g.data_ptr();
        }
        return true;
    }

    // state["step"] += 1 for each state dict (the library advanced its own copy).
    void bump(const py::list& states) {
        PyObject* const key = step_key();
        ++ran;
        size_t i = 0;
        for (const py::handle& h : states) {
            PyObject* d = h.ptr();
            PyObject* v = PyDict_GetItemWithError(d, key);   // borrowed
            if (!v) {
                if (PyErr_Occurred()) throw py::error_already_set();
                throw std::invalid_argument("BatchGuard: a state has no 'step'");
            }
            const long long s = PyLong_AsLongLong(v);
            if (s == -1 && PyErr_Occurred()) throw py::error_already_set();
            PyObject* nv = PyLong_FromLongLong(s + 1);
            if (!nv) throw py::error_already_set();
            // (the step's own write keeps the entries compared, if they were)
            const bool known = with_state && i < items.size() && d == items[i].dict.ptr() &&
                               dict_version(d) == items[i].version && s + 1 == items[i].step0 + ran;
            const int rc = PyDict_SetItem(d, key, nv);
            Py_DECREF(nv);
            if (rc != 0) throw py::error_already_set();
            if (known) items[i].version = dict_version(d);
            ++i;
        }
    }
};

struct SpectralGuard {
    struct Item {
        py::object param, freqs;
        std::vector<int64_t> sizes;
        int pdtype, gdtype, sdtype, device;
        int64_t rank;
        int32_t pcode, gcode, hard, hash;
    };
    std::vector<Item> items;
    int64_t bins, tables;

    // freqs[i]: the state's frequency table the parameter's plan was made
    // from; codes[i] = (param, grad) dtype codes of the C ABI; hard[i], hash[i]:
    // the descriptor's hard channel, and whether it carries hash state.
    SpectralGuard(const py::list& ps, const py::list& freqs, const std::vector<std::pair<int, int>>& codes,
                  const std::vector<int>& hard, const std::vector<int>& hash, int64_t bins_, int64_t tables_)
        : bins(bins_), tables(tables_) {
        for (size_t i = 0; i < ps.size(); ++i) {
            PyObject* o = ps[i].ptr();
            if (!THPVariable_Check(o)) throw std::invalid_argument("SpectralGuard: parameters must be tensors");
            const at::Tensor& t = THPVariable_Unpack(o);
            const at::Tensor& g = t.grad();
            if (!g.defined()) throw std::invalid_argument("SpectralGuard: every parameter needs a grad at plan time");
            PyObject* f = freqs[i].ptr();
            if (!THPVariable_Check(f)) throw std::invalid_argument("SpectralGuard: freqs must be tensors");
            Item it;
            it.param = py::reinterpret_borrow<py::object>(o);
            it.freqs = py::reinterpret_borrow<py::object>(f);
            it.sizes = t.sizes().vec();
            it.pdtype = (int)t.scalar_type();
            it.gdtype = (int)g.scalar_type();
            it.sdtype = (int)(t.scalar_type() == at::kDouble ? at::kDouble : at::kFloat);
            it.device = t.device().index();
            it.rank = THPVariable_Unpack(f).size(0);
            it.pcode = codes[i].first;
            it.gcode = codes[i].second;
            it.hard = hard[i];
            it.hash = hash[i];
            items.push_back(std::move(it));
        }
    }

    // The state's tensor under `key` as the plan expects it (dtype, device,
    // contiguous, numel); nullptr otherwise.
    static void* entry(PyObject* st, PyObject* key, const Item& it, int64_t numel) {
        PyObject* v = PyDict_GetItemWithError(st, key);   // borrowed
        if (!v || !THPVariable_Check(v)) return nullptr;
        const at::Tensor& t = THPVariable_Unpack(v);
        if ((int)t.scalar_type() != it.sdtype || t.numel() != numel || !t.is_contiguous() || !t.device().is_cuda() ||
            t.device().index() != it.device)
            return nullptr;
        return t.data_ptr();
    }

    // Writes the descriptors (step: state["step"] + 1) to out; false if
    // anything differs from plan time (then out must not be used).
    bool fill(const py::dict& state, uintptr_t out_addr) const {
        static PyObject* const scalars[4] = {PyUnicode_InternFromString("force_rms"), PyUnicode_InternFromString("drive_energy"),
                                             PyUnicode_InternFromString("surprise"), PyUnicode_InternFromString("action")};
        static PyObject* const vecs[12] = {
            PyUnicode_InternFromString("omega"), PyUnicode_InternFromString("q_cos"), PyUnicode_InternFromString("q_sin"),
            PyUnicode_InternFromString("p_cos"), PyUnicode_InternFromString("p_sin"), PyUnicode_InternFromString("metric_cos"),
            PyUnicode_InternFromString("metric_sin"), PyUnicode_InternFromString("metric_p_cos"),
            PyUnicode_InternFromString("metric_p_sin"), PyUnicode_InternFromString("calcium_cos"),
            PyUnicode_InternFromString("calcium_sin"), PyUnicode_InternFromString("mode_confidence")};
        static PyObject* const hashes[3] = {PyUnicode_InternFromString("hash_energy"), PyUnicode_InternFromString("hash_impulse"),
                                            PyUnicode_InternFromString("hash_refractory")};
        static PyObject* const k_step = PyUnicode_InternFromString("step");
        static PyObject* const k_freqs = PyUnicode_InternFromString("freqs");
        cresso_spectral_desc* out = reinterpret_cast<cresso_spectral_desc*>(out_addr);
        for (size_t i = 0; i < items.size(); ++i) {
            const Item& it = items[i];
            const at::Tensor& t = THPVariable_Unpack(it.param.ptr());
            const at::Tensor& g = t.grad();
            if ((int)t.scalar_type() != it.pdtype || t.sizes().vec() != it.sizes || !t.is_contiguous() ||
                !t.device().is_cuda() || t.device().index() != it.device)
                return false;
            if (!g.defined() || g.is_sparse() || (int)g.scalar_type() != it.gdtype || g.sizes() != t.sizes() ||
                !g.is_contiguous() || g.device() != t.device())
                return false;
            PyObject* st = PyDict_GetItemWithError(state.ptr(), it.param.ptr());   // borrowed
            if (!st) {
                if (PyErr_Occurred()) throw py::error_already_set();
                return false;
            }
            if (!PyDict_Check(st) || PyDict_GetItemWithError(st, k_freqs) != it.freqs.ptr()) return false;
            PyObject* v = PyDict_GetItemWithError(st, k_step);
            if (!v || !PyLong_Check(v)) return false;
            const long long s = PyLong_AsLongLong(v);
            if (s < 0 || s >= INT32_MAX) {
                PyErr_Clear();
                return false;
            }
            cresso_spectral_desc d{};
            d.param = t.data_ptr();
            d.grad = g.data_ptr();
            d.param_dtype = it.pcode;
            d.grad_dtype = it.gcode;
            d.numel = t.numel();
            d.step = (int32_t)(s + 1);
            d.hard = it.hard;
            void** const sc[4] = {&d.force_rms, &d.drive_energy, &d.surprise, &d.action};
            for (int k = 0; k < 4; ++k)
                if (!(*sc[k] = entry(st, scalars[k], it, 1))) return false;
            void* omega = entry(st, vecs[0], it, it.rank);
            if (!omega) return false;
            d.omega = omega;
            void** const vc[11] = {&d.q_cos, &d.q_sin, &d.p_cos, &d.p_sin, &d.metric_cos, &d.metric_sin,
                                   &d.metric_p_cos, &d.metric_p_sin, &d.calcium_cos, &d.calcium_sin, &d.mode_confidence};
            for (int k = 0; k < 11; ++k)
                if (!(*vc[k] = entry(st, vecs[k + 1], it, it.rank))) return false;
            if (it.hash) {
                void** const hs[3] = {&d.hash_energy, &d.hash_impulse, &d.hash_refractory};
                for (int k = 0; k < 3; ++k) {
                    if (!(*hs[k] = entry(st, hashes[k], it, tables * bins))) return false;
                    const at::Tensor& x = THPVariable_Unpack(PyDict_GetItemWithError(st, hashes[k]));
                    if (x.dim() != 2 || x.size(0) != tables || x.size(1) != bins) return false;
                }
            }
            out[i] = d;
        }
        return true;
    }

    // state["step"] += 1 for every item (after fill() returned true)
    void bump(const py::dict& state) const {
        static PyObject* const k_step = PyUnicode_InternFromString("step");
        for (const Item& it : items) {
            PyObject* st = PyDict_GetItemWithError(state.ptr(), it.param.ptr());
            if (!st) {
                if (PyErr_Occurred()) throw py::error_already_set();
                throw std::invalid_argument("SpectralGuard: a parameter has no state");
            }
            PyObject* v = PyDict_GetItemWithError(st, k_step);
            if (!v) throw std::invalid_argument("SpectralGuard: a state has no 'step'");
            PyObject* nv = PyLong_FromLongLong(PyLong_AsLongLong(v) + 1);
            if (!nv) throw py::error_already_set();
            const int rc = PyDict_SetItem(st, k_step, nv);
            Py_DECREF(nv);
            if (rc != 0) throw py::error_already_set();
        }
    }
};

// Dtype code of the C ABI; -1: none.
int dtype_code(at::ScalarType t) {
    return t == at::kFloat ? CRESSO_F32 : t == at::kDouble ? CRESSO_F64 : t == at::kHalf ? CRESSO_F16 : t == at::kBFloat16 ? CRESSO_BF16 : -1;
}

// Writes the scalar plan's descriptors of these tensors to out.  False (out
// must not be used) unless every state holds, under each of its keys (the
// descriptor's order), a tensor of the work dtype (fp64 for fp64 parameters,
// else fp32) on the parameter's device: of one element, or, for the first
// fields[i] keys (a micro tensor's), contiguous in the parameter's shape; and
// "step".  (In Python 3 us a tensor, as long again as the rest of a plan.)
bool scalar_descs(const py::list& ps, const py::list& grads, const py::list& states, const py::list& keys,
                  const std::vector<int>& fields, uintptr_t out_addr) {
    const size_t n = ps.size();
    if (grads.size() != n || states.size() != n || keys.size() != n || fields.size() != n) return false;
    PyObject* const k_step = PyUnicode_InternFromString("step");
    const py::object hold = py::reinterpret_steal<py::object>(k_step);
    cresso_scalar_desc* out = reinterpret_cast<cresso_scalar_desc*>(out_addr);
    for (size_t i = 0; i < n; ++i) {
        PyObject *o = PyList_GET_ITEM(ps.ptr(), i), *go = PyList_GET_ITEM(grads.ptr(), i);
        PyObject *st = PyList_GET_ITEM(states.ptr(), i), *ks = PyList_GET_ITEM(keys.ptr(), i);
        if (!THPVariable_Check(o) || !THPVariable_Check(go) || !PyDict_Check(st) || !PyTuple_Check(ks)) return false;
        const at::Tensor &p = THPVariable_Unpack(o), &g = THPVariable_Unpack(go);
        const at::ScalarType want = p.scalar_type() == at::kDouble ? at::kDouble : at::kFloat;
        cresso_scalar_desc d{};
        d.param = p.data_ptr();
        d.grad = g.data_ptr();
        d.param_dtype = dtype_code(p.scalar_type());
        d.grad_dtype = dtype_code(g.scalar_type());
        d.route = fields[i] > 0 ? 1 : 0;
        if (p.dim() > 8 || PyTuple_GET_SIZE(ks) > 8 || d.param_dtype < 0 || d.grad_dtype < 0) return false;
        d.ndim = (int32_t)p.dim();
        d.numel = p.numel();
        for (int a = 0; a < d.ndim; ++a) d.shape[a] = p.size(a);
        for (Py_ssize_t k = 0; k < PyTuple_GET_SIZE(ks); ++k) {
            PyObject* v = PyDict_GetItemWithError(st, PyTuple_GET_ITEM(ks, k));   // borrowed
            if (!v && PyErr_Occurred()) throw py::error_already_set();
            if (!v || !THPVariable_Check(v)) return false;
            const at::Tensor& x = THPVariable_Unpack(v);
            if (x.scalar_type() != want || x.device() != p.device()) return false;
            if (k < fields[i] ? x.sizes() != p.sizes() || !x.is_contiguous() : x.numel() != 1) return false;
            d.state[k] = x.data_ptr();
        }
        PyObject* v = PyDict_GetItemWithError(st, k_step);   // borrowed
        const long long s = v && PyLong_Check(v) ? PyLong_AsLongLong(v) : -1;
        if (s < 0 || s >= INT32_MAX) {
            PyErr_Clear();
            return false;
        }
        d.step = (int32_t)s;
        out[i] = d;
    }
    return true;
}

// Whether two lists hold the same objects.
bool same_objects(const py::list& a, const py::list& b) {
    if (a.size() != b.size()) return false;
    for (size_t i = 0; i < a.size(); ++i)
        if (PyList_GET_ITEM(a.ptr(), i) != PyList_GET_ITEM(b.ptr(), i)) return false;
    return true;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.doc() = "Per-step host bookkeeping of the CRESSO5 scalar plan";
    py::class_<BatchGuard>(m, "BatchGuard")
        .def(py::init<const py::list&, const py::list&, const py::list&>(), py::arg("params"),
             py::arg("states") = py::list(), py::arg("keys") = py::list())
        .def("holds", &BatchGuard::holds, py::arg("params"), py::arg("state") = py::none())
        .def("gather", &BatchGuard::gather, py::arg("params"), py::arg("out"), py::arg("state") = py::none())
        .def("bump", &BatchGuard::bump);
    py::class_<SpectralGuard>(m, "SpectralGuard")
        .def(py::init<const py::list&, const py::list&, const std::vector<std::pair<int, int>>&, const std::vector<int>&,
                      const std::vector<int>&, int64_t, int64_t>())
        .def("fill", &SpectralGuard::fill)
        .def("bump", &SpectralGuard::bump);
    m.def("same_objects", &same_objects);
    m.def("scalar_descs", &scalar_descs);
}
