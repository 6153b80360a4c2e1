// The host side of a call, natively: `Plan` is what a wrapped function keeps per signature of its arguments. Calling it with
// the arguments walks their containers once, compares every leaf with the signature, finds the leaves that have to be copied,
// evaluates the recorded sequence and builds the result. A call it does not recognise in every respect - other containers,
// shapes, element types or layouts - is answered with NotImplemented before anything has changed, and takes the general path
// (Function.__call__), whose results are the same.
//
// For a network of 268 parameter arrays the general path spends 290 us on this (flattening, signature, which arrays to copy,
// restoring the results' containers), for one of a single layer 16. Calls, before and after: affine layer on 8 samples 42.7 -> 25.8 us,
// MLP on 256 samples 101 -> 71, ResNet-50 on one image 911 -> 610, on 64 images 5.4 -> 4.8 ms.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#define NPY_NO_DEPRECATED_API NPY_1_7_API_VERSION
#include <numpy/arrayobject.h>
#include <cstdint>
#include <memory>
#include <new>
#include <vector>

namespace {

typedef int (*EvalFn)(uint64_t seq, void* const* host_ptrs, int nslots, uint32_t flags);

struct Node {
    enum Kind { LEAF, NONE, TUPLE, LIST, DICT } kind = NONE;
    std::vector<Node> children;
    std::vector<PyObject*> keys;                    // DICT, owned by the plan's specification
    // LEAF
    std::vector<npy_intp> shape;
    int type = 0, slot = -1;                        // slot -1: nothing reads this argument
    Py_ssize_t number = 0;                          // of the leaf, in the order of the arguments
};

struct Plan {
    PyObject_HEAD
    PyObject *interpreter, *resident, *specification;
    std::vector<Node>* arguments;
    Node* result;
    std::vector<PyObject*>* numbers;                // the leaves' numbers as Python integers (keys of `resident`)
    EvalFn eval;
    unsigned long long sequence;
    int nslots, nresults;
    unsigned flags;
};

// ('a', shape, 'f' | 'i' | 'u', slot) | ('n',) | ('t' | 'l', [children]) | ('d', [keys], [children])
bool parse(PyObject* spec, Node& node, Py_ssize_t& leaves) {
    PyObject* tag = PyTuple_Check(spec) && PyTuple_GET_SIZE(spec) > 0 ? PyTuple_GET_ITEM(spec, 0) : nullptr;
    const char* t = tag ? PyUnicode_AsUTF8(tag) : nullptr;
    if (!t) { if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "Plan: bad specification"); return false; }
    if (t[0] == 'a') {
        PyObject* shape = nullptr;
        const char* type = nullptr;
        const char* ignored = nullptr;
        if (!PyArg_ParseTuple(spec, "sO!si", &ignored, &PyTuple_Type, &shape, &type, &node.slot)) return false;
        node.kind = Node::LEAF;
        node.type = type[0] == 'f' ? NPY_FLOAT32 : type[0] == 'i' ? NPY_INT32 : NPY_UINT32;
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(shape); i++) node.shape.push_back((npy_intp)PyLong_AsSsize_t(PyTuple_GET_ITEM(shape, i)));
        node.number = leaves++;
        return !PyErr_Occurred() && node.shape.size() <= NPY_MAXDIMS;
    }
    if (t[0] == 'n') { node.kind = Node::NONE; return true; }
    PyObject *keys = nullptr, *children = nullptr;
    const char* ignored = nullptr;
    if (t[0] == 'd') {
        if (!PyArg_ParseTuple(spec, "sO!O!", &ignored, &PyList_Type, &keys, &PyList_Type, &children)) return false;
        for (Py_ssize_t i = 0; i < PyList_GET_SIZE(keys); i++) node.keys.push_back(PyList_GET_ITEM(keys, i));
        if (PyList_GET_SIZE(keys) != PyList_GET_SIZE(children)) { PyErr_SetString(PyExc_TypeError, "Plan: bad specification"); return false; }
    } else if (!PyArg_ParseTuple(spec, "sO!", &ignored, &PyList_Type, &children)) {
        return false;
    }
    node.kind = t[0] == 'd' ? Node::DICT : t[0] == 'l' ? Node::LIST : Node::TUPLE;
    node.children.resize((size_t)PyList_GET_SIZE(children));
    for (size_t i = 0; i < node.children.size(); i++)
        if (!parse(PyList_GET_ITEM(children, (Py_ssize_t)i), node.children[i], leaves)) return false;
    return true;
}

struct Held {                                       // references that go when the call ends, whichever way
    std::vector<PyObject*> objects;
    ~Held() { for (PyObject* o : objects) Py_XDECREF(o); }
};

// Whether x is what the signature says; its leaves are added to `found`, with a reference each: what runs between here and the
// evaluation (the end of an array that was held, the cycle collector, another thread) may take them out of their containers.
// Exact types only: anything else may mean something else to the general path. -1: an exception is set.
int match(const Node& node, PyObject* x, Held& found) {
    switch (node.kind) {
    case Node::LEAF: {
        if (!PyArray_CheckExact(x)) return 0;
        PyArrayObject* a = (PyArrayObject*)x;
        if (PyArray_TYPE(a) != node.type || PyArray_ISBYTESWAPPED(a) || PyArray_NDIM(a) != (int)node.shape.size()) return 0;
        for (size_t d = 0; d < node.shape.size(); d++) if (PyArray_DIM(a, (int)d) != node.shape[d]) return 0;
        if (node.slot >= 0 && !PyArray_IS_C_CONTIGUOUS(a)) return 0;
        found.objects.push_back(x);
        Py_INCREF(x);
        return 1;
    }
    case Node::NONE:
        return x == Py_None;
    case Node::TUPLE:
        if (!PyTuple_CheckExact(x) || PyTuple_GET_SIZE(x) != (Py_ssize_t)node.children.size()) return 0;
        for (size_t i = 0; i < node.children.size(); i++) {
            const int r = match(node.children[i], PyTuple_GET_ITEM(x, (Py_ssize_t)i), found);
            if (r != 1) return r;
        }
        return 1;
    case Node::LIST:
        if (!PyList_CheckExact(x) || PyList_GET_SIZE(x) != (Py_ssize_t)node.children.size()) return 0;
        for (size_t i = 0; i < node.children.size(); i++) {
            const int r = match(node.children[i], PyList_GET_ITEM(x, (Py_ssize_t)i), found);
            if (r != 1) return r;
        }
        return 1;
    default:
        if (!PyDict_CheckExact(x) || PyDict_GET_SIZE(x) != (Py_ssize_t)node.children.size()) return 0;
        for (size_t i = 0; i < node.children.size(); i++) {
            PyObject* value = PyDict_GetItemWithError(x, node.keys[i]);
            if (!value) return PyErr_Occurred() ? -1 : 0;
            const int r = match(node.children[i], value, found);
            if (r != 1) return r;
        }
        return 1;
    }
}

// True for an array whose values cannot change while the caller holds it: not writeable, nor a view of anything but such an
// array or a bytes object (jaxpr_interpreter._is_immutable).
bool immutable(PyObject* x) {
    while (x && PyArray_CheckExact(x)) {
        if (PyArray_ISWRITEABLE((PyArrayObject*)x)) return false;
        x = PyArray_BASE((PyArrayObject*)x);
    }
    return !x || x == Py_None || PyBytes_CheckExact(x);
}

bool new_results(const Node& node, std::vector<PyObject*>& arrays) {
    if (node.kind == Node::LEAF) {
        PyObject* a = PyArray_SimpleNew((int)node.shape.size(), const_cast<npy_intp*>(node.shape.data()), node.type);
        if (!a) return false;
        arrays.push_back(a);
        return true;
    }
    for (const Node& c : node.children) if (!new_results(c, arrays)) return false;
    return true;
}

// The results in their containers; takes the arrays over (entries that have gone into a container are set to null).
PyObject* build(const Node& node, std::vector<PyObject*>& arrays, size_t& next) {
    if (node.kind == Node::LEAF) { PyObject* a = arrays[next]; arrays[next++] = nullptr; return a; }
    if (node.kind == Node::NONE) Py_RETURN_NONE;
    const Py_ssize_t n = (Py_ssize_t)node.children.size();
    PyObject* out = node.kind == Node::DICT ? PyDict_New() : node.kind == Node::LIST ? PyList_New(n) : PyTuple_New(n);
    for (Py_ssize_t i = 0; out && i < n; i++) {
        PyObject* c = build(node.children[(size_t)i], arrays, next);
        if (!c) { Py_CLEAR(out); break; }
        if (node.kind == Node::LIST) PyList_SET_ITEM(out, i, c);
        else if (node.kind == Node::TUPLE) PyTuple_SET_ITEM(out, i, c);
        else {
            const int r = PyDict_SetItem(out, node.keys[(size_t)i], c);
            Py_DECREF(c);
            if (r) Py_CLEAR(out);
        }
    }
    return out;
}

void result_pointers(const Node& node, const std::vector<PyObject*>& arrays, size_t& next, std::vector<void*>& host) {
    if (node.kind == Node::LEAF) { host[(size_t)node.slot] = PyArray_DATA((PyArrayObject*)arrays[next++]); return; }
    for (const Node& c : node.children) result_pointers(c, arrays, next, host);
}

void leaf_slots(const Node& node, std::vector<int>& slots) {
    if (node.kind == Node::LEAF) slots.push_back(node.slot);
    for (const Node& c : node.children) leaf_slots(c, slots);
}

PyObject* run(Plan* plan, PyObject* args) {
    if (!PyTuple_CheckExact(args) || PyTuple_GET_SIZE(args) != (Py_ssize_t)plan->arguments->size()) Py_RETURN_NOTIMPLEMENTED;
    Held found;
    found.objects.reserve(plan->numbers->size());
    for (size_t i = 0; i < plan->arguments->size(); i++) {
        const int r = match((*plan->arguments)[i], PyTuple_GET_ITEM(args, (Py_ssize_t)i), found);
        if (r < 0) return nullptr;
        if (r == 0) Py_RETURN_NOTIMPLEMENTED;
    }
    std::vector<int> slots;
    slots.reserve(found.objects.size());
    for (const Node& n : *plan->arguments) leaf_slots(n, slots);
    std::vector<void*> host((size_t)plan->nslots, nullptr);
    Held results;
    results.objects.reserve((size_t)plan->nresults);
    if (!new_results(*plan->result, results.objects)) return nullptr;
    size_t next = 0;
    result_pointers(*plan->result, results.objects, next, host);
    // Which leaves have to be copied: all that may have changed, and those that are not what their buffers hold. From here on
    // the evaluation follows at once, so what is noted as held is held.
    for (size_t k = 0; k < found.objects.size(); k++) {
        if (slots[k] < 0) continue;
        PyObject* leaf = found.objects[k];
        if (immutable(leaf)) {
            PyObject* key  = (*plan->numbers)[k];
            PyObject* held = PyDict_GetItemWithError(plan->resident, key);
            if (!held && PyErr_Occurred()) { PyDict_Clear(plan->resident); return nullptr; }
            if (held && PyTuple_CheckExact(held) && PyTuple_GET_SIZE(held) == 2 && PyTuple_GET_ITEM(held, 0) == leaf && PyTuple_GET_ITEM(held, 1) == Py_None) continue;
            PyObject* note = PyTuple_Pack(2, leaf, Py_None);
            if (!note || PyDict_SetItem(plan->resident, key, note)) { Py_XDECREF(note); PyDict_Clear(plan->resident); return nullptr; }
            Py_DECREF(note);
        } else if (PyDict_GET_SIZE(plan->resident)) {   // takes the place of what its buffer held
            const int noted = PyDict_Contains(plan->resident, (*plan->numbers)[k]);
            if (noted < 0 || (noted && PyDict_DelItem(plan->resident, (*plan->numbers)[k]))) { PyDict_Clear(plan->resident); return nullptr; }
        }
        host[(size_t)slots[k]] = PyArray_DATA((PyArrayObject*)leaf);
    }
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = plan->eval(plan->sequence, host.data(), plan->nslots, plan->flags);
    Py_END_ALLOW_THREADS
    PyObject* ended = PyObject_CallMethod(plan->interpreter, "_evaluated", "i", status);      // counts it; raises where it failed
    if (!ended) return nullptr;
    Py_DECREF(ended);
    next = 0;
    return build(*plan->result, results.objects, next);
}

PyObject* plan_call(PyObject* self, PyObject* args, PyObject* kwargs) {
    PyObject* arguments = nullptr;
    if ((kwargs && PyDict_GET_SIZE(kwargs)) || !PyArg_ParseTuple(args, "O!", &PyTuple_Type, &arguments)) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "Plan takes the tuple of arguments");
        return nullptr;
    }
    try { return run((Plan*)self, arguments); } catch (const std::bad_alloc&) { return PyErr_NoMemory(); }
}

// Plan(interpreter, resident, eval address, sequence handle, slots, flags, [argument specifications], result specification)
PyObject* plan_new(PyTypeObject* type, PyObject* args, PyObject*) {
    PyObject *interpreter, *resident, *arguments, *result;
    unsigned long long address, sequence;
    int nslots;
    unsigned flags;
    if (!PyArg_ParseTuple(args, "OO!KKiIO!O!", &interpreter, &PyDict_Type, &resident, &address, &sequence, &nslots, &flags, &PyList_Type, &arguments,
                          &PyTuple_Type, &result)) return nullptr;
    Plan* plan = (Plan*)type->tp_alloc(type, 0);
    if (!plan) return nullptr;
    Py_INCREF(interpreter); plan->interpreter = interpreter;
    Py_INCREF(resident); plan->resident = resident;
    plan->specification = PyTuple_Pack(2, arguments, result);               // (owns the keys of the containers)
    plan->eval = (EvalFn)(uintptr_t)address;
    plan->sequence = sequence; plan->nslots = nslots; plan->flags = flags;
    bool ok = plan->specification != nullptr;
    try {
        plan->arguments = new std::vector<Node>((size_t)PyList_GET_SIZE(arguments));
        plan->result    = new Node();
        plan->numbers   = new std::vector<PyObject*>();
        Py_ssize_t leaves = 0, results = 0;
        for (size_t i = 0; ok && i < plan->arguments->size(); i++) ok = parse(PyList_GET_ITEM(arguments, (Py_ssize_t)i), (*plan->arguments)[i], leaves);
        ok = ok && parse(result, *plan->result, results);
        plan->nresults = (int)results;
        std::vector<int> slots;
        if (ok) { for (const Node& n : *plan->arguments) leaf_slots(n, slots); leaf_slots(*plan->result, slots); }
        for (size_t k = 0; ok && k < slots.size(); k++)
            if (slots[k] >= nslots || (slots[k] < 0 && k >= (size_t)leaves)) { PyErr_SetString(PyExc_ValueError, "Plan: slot out of range"); ok = false; }
        for (Py_ssize_t k = 0; ok && k < leaves; k++) {
            PyObject* n = PyLong_FromSsize_t(k);
            if (!n) ok = false; else plan->numbers->push_back(n);
        }
    } catch (const std::bad_alloc&) { PyErr_NoMemory(); ok = false; }
    if (!ok) { Py_DECREF(plan); return nullptr; }
    return (PyObject*)plan;
}

void plan_dealloc(PyObject* self) {
    Plan* plan = (Plan*)self;
    if (plan->numbers) for (PyObject* n : *plan->numbers) Py_XDECREF(n);
    delete plan->arguments; delete plan->result; delete plan->numbers;
    Py_XDECREF(plan->interpreter); Py_XDECREF(plan->resident); Py_XDECREF(plan->specification);
    Py_TYPE(self)->tp_free(self);
}

PyTypeObject PlanType = [] {
    PyTypeObject t = {PyVarObject_HEAD_INIT(nullptr, 0)};
    t.tp_name = "vkjax_amd.lib.vkjax_call.Plan";
    t.tp_basicsize = sizeof(Plan);
    t.tp_flags = Py_TPFLAGS_DEFAULT;
    t.tp_new = plan_new;
    t.tp_dealloc = plan_dealloc;
    t.tp_call = plan_call;
    return t;
}();

PyModuleDef module = {PyModuleDef_HEAD_INIT, "vkjax_call", "Calls of wrapped functions, natively.", -1, nullptr, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_vkjax_call(void) {
    import_array();
    if (PyType_Ready(&PlanType) < 0) return nullptr;
    PyObject* m = PyModule_Create(&module);
    if (!m) return nullptr;
    Py_INCREF(&PlanType);
    if (PyModule_AddObject(m, "Plan", (PyObject*)&PlanType) < 0) { Py_DECREF(&PlanType); Py_DECREF(m); return nullptr; }
    return m;
}
