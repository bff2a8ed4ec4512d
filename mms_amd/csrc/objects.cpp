// Python objects into flat arrays: what the searches hand over (lists of placements, lists of requests), read through
// CPython's C API.  Only the plain forms are read here, exact lists, tuples, ints and floats; anything else returns None
// and is left to the caller's own, general code, which then also says what is wrong with it.
//
// What bounds it: a look at each object, and the memory it lies in.  4096 placements, 131072 groups, 400000 model ids: 10
// ms with iterators over all of them that numpy reads, 3.7 here (asking for rows ahead of their turn: no gain); 30000
// requests: 4.4 / 0.7 ms.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <exception>
#include <vector>

namespace {

struct Ref {  // owns a reference
    PyObject *p = nullptr;
    explicit Ref(PyObject *o) : p(o) {}
    Ref(Ref &&o) noexcept : p(o.p) { o.p = nullptr; }
    Ref(const Ref &) = delete;
    Ref &operator=(const Ref &) = delete;
    ~Ref() { Py_XDECREF(p); }
};

bool is_row(PyObject *o) { return PyList_CheckExact(o) || PyTuple_CheckExact(o); }
// (of an exact list or tuple)
Py_ssize_t length(PyObject *row) { return PySequence_Fast_GET_SIZE(row); }
PyObject *item(PyObject *row, Py_ssize_t i) { return PySequence_Fast_GET_ITEM(row, i); }

bool int32_of(PyObject *o, int32_t *out) {  // an exact int of 32 bits
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    const long v = PyLong_AsLongAndOverflow(o, &overflow);
    if (overflow != 0 || v < INT32_MIN || v > INT32_MAX) return false;
    *out = (int32_t)v;
    return true;
}

template <typename T>
PyObject *bytes_of(const std::vector<T> &v) {
    return PyByteArray_FromStringAndSize(reinterpret_cast<const char *>(v.data()), (Py_ssize_t)(v.size() * sizeof(T)));
}

PyObject *g_configs, *g_models, *g_model_name, *g_slo;  // attribute names

// pack(sols, index, config_id) -> (Gmax, groups of each placement i32, configuration ids i32 [][Gmax], where each group's
// models start i64 [][Gmax+1], model ids i32), or None.  index: {configuration: id}; config_id(configuration) adds one.
PyObject *pack(PyObject *, PyObject *args) {
    PyObject *sols, *index, *config_id;
    if (!PyArg_ParseTuple(args, "OO!O", &sols, &PyDict_Type, &index, &config_id)) return nullptr;
    if (!is_row(sols)) Py_RETURN_NONE;
    try {
        std::vector<int32_t> groups, cfg_ids, ids;
        std::vector<int64_t> sizes;
        // Placements share their configuration objects: those met in this call are found by address, without hashing
        // (and kept alive meanwhile: looking one up may run its own code).
        struct Met {
            PyObject *cfg = nullptr;
            int32_t id = 0;
            ~Met() { Py_XDECREF(cfg); }
        } met[64];
        for (Py_ssize_t b = 0; b < length(sols); ++b) {
            Ref sol(Py_NewRef(item(sols, b)));
            Ref cfgs(PyObject_GetAttr(sol.p, g_configs));
            if (!cfgs.p) return nullptr;
            Ref models(PyObject_GetAttr(sol.p, g_models));
            if (!models.p) return nullptr;
            if (!is_row(cfgs.p) || !is_row(models.p) || length(cfgs.p) > INT32_MAX) Py_RETURN_NONE;
            const Py_ssize_t n = length(cfgs.p);
            groups.push_back((int32_t)n);
            for (Py_ssize_t g = 0; g < n; ++g) {
                if (g >= length(cfgs.p)) Py_RETURN_NONE;
                PyObject *cfg = item(cfgs.p, g);
                Met &slot = met[(reinterpret_cast<uintptr_t>(cfg) >> 4) & 63u];
                if (slot.cfg != cfg) {
                    Py_XDECREF(slot.cfg);
                    slot.cfg = Py_NewRef(cfg);
                    PyObject *known = PyDict_GetItemWithError(index, cfg);
                    if (!known && PyErr_Occurred()) return nullptr;
                    Ref id(known ? Py_NewRef(known) : PyObject_CallOneArg(config_id, cfg));
                    if (!id.p) return nullptr;
                    if (!int32_of(id.p, &slot.id)) Py_RETURN_NONE;
                }
                cfg_ids.push_back(slot.id);
                if (g >= length(models.p)) Py_RETURN_NONE;
                PyObject *row = item(models.p, g);
                if (!is_row(row)) Py_RETURN_NONE;
                const Py_ssize_t hosts = length(row);
                sizes.push_back((int64_t)hosts);
                const size_t at = ids.size();
                ids.resize(at + (size_t)hosts);
                for (Py_ssize_t k = 0; k < hosts; ++k)
                    if (!int32_of(item(row, k), &ids[at + (size_t)k])) Py_RETURN_NONE;
            }
            if (length(models.p) != n) Py_RETURN_NONE;
        }
        int32_t most = 1;
        for (const int32_t n : groups) most = std::max(most, n);
        std::vector<int32_t> group_cfg(groups.size() * (size_t)most, 0);
        std::vector<int64_t> gm_off;
        gm_off.reserve(groups.size() * ((size_t)most + 1));
        size_t group = 0;
        int64_t first = 0;
        for (size_t b = 0; b < groups.size(); ++b) {
            gm_off.push_back(first);
            for (int32_t g = 0; g < most; ++g) {
                if (g < groups[b]) {
                    group_cfg[b * (size_t)most + (size_t)g] = cfg_ids[group];
                    first += sizes[group++];
                }
                gm_off.push_back(first);
            }
        }
        Ref n(PyLong_FromLong(most)), a(bytes_of(groups)), c(bytes_of(group_cfg)), o(bytes_of(gm_off)), i(bytes_of(ids));
        if (!n.p || !a.p || !c.p || !o.p || !i.p) return nullptr;
        return PyTuple_Pack(5, n.p, a.p, c.p, o.p, i.p);
    } catch (const std::exception &) {  // (vectors throw nothing else than that there is no memory for them)
        return PyErr_NoMemory();
    }
}

// count_models(sols) -> models of each placement, over its groups, i64, or None
PyObject *count_models(PyObject *, PyObject *sols) {
    if (!is_row(sols)) Py_RETURN_NONE;
    try {
        std::vector<int64_t> counts;
        for (Py_ssize_t b = 0; b < length(sols); ++b) {
            Ref sol(Py_NewRef(item(sols, b)));
            Ref models(PyObject_GetAttr(sol.p, g_models));
            if (!models.p) return nullptr;
            if (!is_row(models.p)) Py_RETURN_NONE;
            int64_t n = 0;
            for (Py_ssize_t g = 0; g < length(models.p); ++g) {
                PyObject *row = item(models.p, g);
                if (!is_row(row)) Py_RETURN_NONE;
                n += (int64_t)length(row);
            }
            counts.push_back(n);
        }
        return bytes_of(counts);
    } catch (const std::exception &) {  // (vectors throw nothing else than that there is no memory for them)
        return PyErr_NoMemory();
    }
}

// request_arrays(requests, name2id) -> (model ids i32, -1: not one of them; latency objectives f32), or None
PyObject *request_arrays(PyObject *, PyObject *args) {
    PyObject *requests, *name2id;
    if (!PyArg_ParseTuple(args, "OO!", &requests, &PyDict_Type, &name2id)) return nullptr;
    if (!is_row(requests)) Py_RETURN_NONE;
    try {
        std::vector<int32_t> ids;
        std::vector<float> slos;
        for (Py_ssize_t k = 0; k < length(requests); ++k) {
            Ref req(Py_NewRef(item(requests, k)));
            Ref name(PyObject_GetAttr(req.p, g_model_name));
            if (!name.p) return nullptr;
            Ref slo(PyObject_GetAttr(req.p, g_slo));
            if (!slo.p) return nullptr;
            if (!PyFloat_CheckExact(slo.p)) Py_RETURN_NONE;
            const double d = PyFloat_AS_DOUBLE(slo.p);
            const float f = (float)d;
            if (std::isinf(f) && !std::isinf(d)) Py_RETURN_NONE;  // (numpy has a warning for it)
            PyObject *id = PyDict_GetItemWithError(name2id, name.p);
            if (!id && PyErr_Occurred()) return nullptr;
            int32_t m = -1;
            if (id && !int32_of(id, &m)) Py_RETURN_NONE;
            ids.push_back(m);
            slos.push_back(f);
        }
        Ref a(bytes_of(ids)), b(bytes_of(slos));
        if (!a.p || !b.p) return nullptr;
        return PyTuple_Pack(2, a.p, b.p);
    } catch (const std::exception &) {  // (vectors throw nothing else than that there is no memory for them)
        return PyErr_NoMemory();
    }
}

PyMethodDef methods[] = {{"pack", pack, METH_VARARGS, nullptr},
                         {"count_models", count_models, METH_O, nullptr},
                         {"request_arrays", request_arrays, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_objects", "Python objects into flat arrays.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__objects(void) {
    if (!(g_configs = PyUnicode_InternFromString("group_configs")) || !(g_models = PyUnicode_InternFromString("group_models")) ||
        !(g_model_name = PyUnicode_InternFromString("model_name")) || !(g_slo = PyUnicode_InternFromString("slo")))
        return nullptr;
    return PyModule_Create(&module);
}
