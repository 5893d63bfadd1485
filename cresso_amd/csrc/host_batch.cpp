// Host-side bookkeeping of the scalar plan's steady state, in C++.
//
// One optimizer step of a group of many small tensors (the C3 case: 840) is a
// single kernel sequence on the GPU, but the per-step Python work around it
// (checking that the group is unchanged, collecting the fresh grad pointers
// that autograd allocates, advancing every state["step"]) costs about 0.2 us
// per tensor and per item in CPython, which is as long as the GPU step itself.
// BatchGuard does the same checks and writes in one pass over the Python
// objects: gather() verifies each parameter (same object, same storage) and
// its grad (defined, contiguous, same dtype/device/numel as at plan time) and
// writes the grad pointers into a host array; bump() adds 1 to state["step"].
// Any mismatch makes gather() return false and the caller rebuilds the plan.
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

struct BatchGuard {
    // Strong references: a parameter cannot be freed (and a new object created
    // at its address) while the guard lives, so the identity test is exact.
    std::vector<py::object> params;
    std::vector<const void*> pptr;   // param storage at plan time
    std::vector<int> gdtype;         // grad dtype at plan time (c10::ScalarType)
    std::vector<int64_t> numel;
    std::vector<int> device;

    explicit BatchGuard(const py::list& ps) {
        const size_t n = ps.size();
        params.reserve(n);
        for (size_t i = 0; i < n; ++i) {
            PyObject* o = ps[i].ptr();
            if (!THPVariable_Check(o)) throw std::invalid_argument("BatchGuard: parameters must be tensors");
            const at::Tensor& t = THPVariable_Unpack(o);
            const at::Tensor& g = t.grad();
            if (!g.defined()) throw std::invalid_argument("BatchGuard: every parameter needs a grad at plan time");
            params.push_back(py::reinterpret_borrow<py::object>(o));
            pptr.push_back(t.data_ptr());
            gdtype.push_back(static_cast<int>(g.scalar_type()));
            numel.push_back(t.numel());
            device.push_back(t.device().index());
        }
    }

    // Writes params[i].grad.data_ptr() to out[i]; false if anything differs
    // from plan time (then out is partially written and must not be used).
    bool gather(const py::list& ps, uintptr_t out_addr) const {
        const size_t n = params.size();
        if (ps.size() != n) return false;
        void** out = reinterpret_cast<void**>(out_addr);
        for (size_t i = 0; i < n; ++i) {
            PyObject* o = ps[i].ptr();
            if (o != params[i].ptr()) return false;
            const at::Tensor& t = THPVariable_Unpack(o);
            if (t.data_ptr() != pptr[i]) return false;
            const at::Tensor& g = t.grad();
            if (!g.defined() || static_cast<int>(g.scalar_type()) != gdtype[i] || g.numel() != numel[i] ||
                g.device().index() != device[i] || !g.device().is_cuda() || g.is_sparse() || !g.is_contiguous())
                return false;
            out[i] = g.data_ptr();
        }
        return true;
    }

    // state["step"] += 1 for each state dict (the library advanced its own copy).
    void bump(const py::list& states) const {
        static PyObject* key = PyUnicode_InternFromString("step");
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
            const int rc = PyDict_SetItem(d, key, nv);
            Py_DECREF(nv);
            if (rc != 0) throw py::error_already_set();
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
        .def(py::init<const py::list&>())
        .def("gather", &BatchGuard::gather)
        .def("bump", &BatchGuard::bump);
    py::class_<SpectralGuard>(m, "SpectralGuard")
        .def(py::init<const py::list&, const py::list&, const std::vector<std::pair<int, int>>&, const std::vector<int>&,
                      const std::vector<int>&, int64_t, int64_t>())
        .def("fill", &SpectralGuard::fill)
        .def("bump", &SpectralGuard::bump);
    m.def("same_objects", &same_objects);
}
