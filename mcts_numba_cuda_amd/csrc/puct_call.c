/* Host side of a PUCT launch from Python, for the usual case: a dictionary of contiguous torch tensors on the GPU whose
 * shapes and types fit.  What mcts_numba_cuda_amd/puct.py does attribute by attribute and then through ctypes (longer than
 * a small selection takes on the GPU), in one call into C: the same checks, the addresses, the launcher.
 * Whatever does not fit -- another kind of array, a wrong shape, a missing name -- is left to the Python code, which
 * handles it or says what is wrong. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>
#ifdef PUCT_CALL_DLPACK        /* the DLPack header that torch ships, where it has the exchange interface */
#include PUCT_CALL_DLPACK
#endif

static PyObject *tensor_type, *int32_type, *float32_type;   /* torch.Tensor, torch.int32, torch.float32 */
static PyObject *current_device, *current_stream;            /* () -> device, (device) -> stream handle */
static PyObject *s_shape, *s_dtype, *s_is_cuda, *s_is_contiguous, *s_data_ptr, *s_edge_child, *s_out_path;

enum { MOST_DIMS = 3, MOST_ARRAYS = 11 };
enum { TREES, NODES, EDGES, WALKS, PATHS };

/* sizes (trees, nodes, edges, warps, path_depth) that make up the shape of an array of each kind */
static const int dims_of[5] = {1, 2, 3, 2, 3};
static const int sizes_of[5][MOST_DIMS] = {{0}, {0, 1}, {0, 1, 2}, {0, 3}, {0, 3, 4}};

#ifdef PUCT_CALL_DLPACK
/* Torch's own answer to all of a tensor's questions in one call into C, through the table it publishes with its tensor type
 * (__dlpack_c_exchange_api__; NULL where there is none).  Five attributes each of a dozen arrays were 3 of the 6.8 us of a
 * call, as long as the launch itself: 3.9 us now, a selection and its backup of 16 trees 13.9 -> 10.5 us. */
static int (*tensor_of)(void *, DLTensor *);

/* 1: t has the answers in *out; 0: it is left to the attributes */
static int read_tensor(PyObject *t, DLTensor *out) {
    if (!tensor_of || (PyObject *)Py_TYPE(t) != tensor_type) return 0;
    if (tensor_of(t, out) == 0 && out->data) return 1;   /* (no address, or an error: the attributes say why) */
    PyErr_Clear();
    return 0;
}

/* 1: a contiguous GPU tensor of that type and shape; 0: not */
static int tensor_fits(const DLTensor *t, int is_float, int kind, const int64_t *sizes) {
    if ((t->device.device_type != kDLROCM && t->device.device_type != kDLCUDA) || t->ndim != dims_of[kind] || t->dtype.bits != 32 || t->dtype.lanes != 1 ||
        t->dtype.code != (is_float ? kDLFloat : kDLInt)) return 0;
    int64_t stride = 1;
    int dense = 1, empty = 0;
    for (int i = t->ndim - 1; i >= 0; i--) {
        if (t->shape[i] != sizes[sizes_of[kind][i]]) return 0;
        if (t->shape[i] == 0) empty = 1;
        if (t->strides && t->shape[i] != 1 && t->strides[i] != stride) dense = 0;
        stride *= t->shape[i];
    }
    return dense || empty;
}
#endif

/* 1: the shape of t was read into dim[0..want); 0: it has another number of dimensions; -1: an error is set */
static int read_shape(PyObject *t, Py_ssize_t want, int64_t *dim) {
#ifdef PUCT_CALL_DLPACK
    DLTensor as;
    if (read_tensor(t, &as)) {
        for (Py_ssize_t i = 0; as.ndim == want && i < want; i++) dim[i] = as.shape[i];
        return as.ndim == want;
    }
#endif
    PyObject *shape = PyObject_GetAttr(t, s_shape);
    if (!shape) return -1;
    int ok = PyTuple_Check(shape) && PyTuple_GET_SIZE(shape) == want;
    for (Py_ssize_t i = 0; ok && i < want; i++) {
        dim[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(shape, i));
        if (dim[i] == -1 && PyErr_Occurred()) ok = -1;
    }
    Py_DECREF(shape);
    return ok;
}

/* 1: t is a contiguous GPU tensor of that type and shape, *address is its address; 0: it is not; -1: an error is set */
static int read_array(PyObject *t, PyObject *type, int kind, const int64_t *sizes, void **address) {
    int64_t dim[MOST_DIMS];
    if ((PyObject *)Py_TYPE(t) != tensor_type) return 0;
#ifdef PUCT_CALL_DLPACK
    DLTensor as;
    if (read_tensor(t, &as)) {
        if (!tensor_fits(&as, type == float32_type, kind, sizes)) return 0;
        *address = (char *)as.data + as.byte_offset;
        return 1;
    }
#endif
    int ok = read_shape(t, dims_of[kind], dim);
    if (ok <= 0) return ok;
    for (int i = 0; i < dims_of[kind]; i++) if (dim[i] != sizes[sizes_of[kind][i]]) return 0;
    PyObject *v = PyObject_GetAttr(t, s_dtype);
    if (!v) return -1;
    ok = v == type;
    Py_DECREF(v);
    if (!ok) return 0;
    if (!(v = PyObject_GetAttr(t, s_is_cuda))) return -1;
    ok = v == Py_True;
    Py_DECREF(v);
    if (!ok) return 0;
    if (!(v = PyObject_CallMethodNoArgs(t, s_is_contiguous))) return -1;
    ok = v == Py_True;
    Py_DECREF(v);
    if (!ok) return 0;
    if (!(v = PyObject_CallMethodNoArgs(t, s_data_ptr))) return -1;
    *address = (void *)(uintptr_t)PyLong_AsUnsignedLongLong(v);
    Py_DECREF(v);
    return PyErr_Occurred() ? -1 : 1;
}

typedef int (*EdgeSelect)(float, float, float, int, void *, void *, void *, void *, void *, void *, void *, void *, void *, void *, void *, int, int, int, int, int, void *);
typedef int (*NodeSelect)(float, float, float, void *, void *, void *, void *, void *, void *, void *, void *, void *, void *, void *, int, int, int, int, int, void *);
typedef int (*EdgeBackup)(int, void *, void *, void *, void *, void *, void *, void *, void *, void *, int, int, int, int, int, void *);
typedef int (*NodeBackup)(int, void *, void *, void *, void *, void *, void *, void *, void *, void *, void *, int, int, int, int, int, void *);
enum { EDGE_SELECT, NODE_SELECT, EDGE_BACKUP, NODE_BACKUP };
static const int arrays_of[4] = {11, 11, 8, 9};

/* launch(what, address of the launcher, arrays, d, values, whole, a, b, c): arrays = ((name, 1 for float32 or 0, kind), ...)
 * in the launcher's order, then others of d that only have to have the right shape.  The launcher's answer, or None. */
static PyObject *launch(PyObject *self, PyObject *const *arg, Py_ssize_t n_args) {
    (void)self;
    if (n_args != 9 || !tensor_type) { PyErr_SetString(PyExc_TypeError, "launch: not set up, or not 9 arguments"); return NULL; }
    const long what = PyLong_AsLong(arg[0]);
    const uintptr_t entry = (uintptr_t)PyLong_AsUnsignedLongLong(arg[1]);
    PyObject *const arrays = arg[2], *const d = arg[3], *const values = arg[4];
    const int whole = (int)PyLong_AsLong(arg[5]);
    const float a = (float)PyFloat_AsDouble(arg[6]), b = (float)PyFloat_AsDouble(arg[7]), c = (float)PyFloat_AsDouble(arg[8]);
    if (PyErr_Occurred()) return NULL;
    if (what < 0 || what > NODE_BACKUP || !PyTuple_Check(arrays) || !PyDict_CheckExact(d)) Py_RETURN_NONE;
    const int n = arrays_of[what];
    PyObject *child = PyDict_GetItemWithError(d, s_edge_child), *path = child ? PyDict_GetItemWithError(d, s_out_path) : NULL;
    if (!path) { if (PyErr_Occurred()) return NULL; Py_RETURN_NONE; }
    if ((PyObject *)Py_TYPE(child) != tensor_type || (PyObject *)Py_TYPE(path) != tensor_type) Py_RETURN_NONE;
    int64_t size[5], p3[3];
    Py_INCREF(child);
    Py_INCREF(path);
    int ok = read_shape(child, 3, size);
    if (ok > 0) ok = read_shape(path, 3, p3);
    Py_DECREF(child);
    Py_DECREF(path);
    if (ok < 0) return NULL;
    if (!ok || size[0] != p3[0]) Py_RETURN_NONE;
    size[3] = p3[1]; size[4] = p3[2];
    for (int i = 0; i < 5; i++) if (size[i] > INT32_MAX) Py_RETURN_NONE;
    void *at[MOST_ARRAYS], *of_values = NULL;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(arrays); i++) {
        PyObject *const field = PyTuple_GET_ITEM(arrays, i);
        PyObject *const t = PyDict_GetItemWithError(d, PyTuple_GET_ITEM(field, 0));
        if (!t) { if (PyErr_Occurred()) return NULL; if (i < n) Py_RETURN_NONE; continue; }
        PyObject *const type = PyLong_AsLong(PyTuple_GET_ITEM(field, 1)) ? float32_type : int32_type;
        const int kind = (int)PyLong_AsLong(PyTuple_GET_ITEM(field, 2));
        void *unused;
        /* (an array that the launcher does not take: anything amiss with more than its shape is no matter, so Python looks) */
        Py_INCREF(t);
        ok = read_array(t, type, kind, size, i < n ? &at[i] : &unused);
        Py_DECREF(t);
        if (ok < 0) return NULL;
        if (!ok) Py_RETURN_NONE;
    }
    if (values != Py_None) {
        ok = read_array(values, float32_type, PATHS, size, &of_values);
        if (ok < 0) return NULL;
        if (!ok) Py_RETURN_NONE;
    }
    PyObject *device = PyObject_CallNoArgs(current_device);
    if (!device) return NULL;
    PyObject *stream = PyObject_CallOneArg(current_stream, device);
    Py_DECREF(device);
    if (!stream) return NULL;
    void *const on = (void *)(uintptr_t)PyLong_AsUnsignedLongLong(stream);
    Py_DECREF(stream);
    if (PyErr_Occurred()) return NULL;
    const int trees = (int)size[0], nodes = (int)size[1], edges = (int)size[2], warps = (int)size[3], depth = (int)size[4];
    int code = 0;
    Py_BEGIN_ALLOW_THREADS
    switch (what) {
    case EDGE_SELECT:
        code = ((EdgeSelect)entry)(a, b, c, whole, at[0], at[1], at[2], at[3], at[4], at[5], at[6], at[7], at[8], at[9], at[10], trees, nodes, edges, warps, depth, on);
        break;
    case NODE_SELECT:
        code = ((NodeSelect)entry)(a, b, c, at[0], at[1], at[2], at[3], at[4], at[5], at[6], at[7], at[8], at[9], at[10], trees, nodes, edges, warps, depth, on);
        break;
    case EDGE_BACKUP:
        code = ((EdgeBackup)entry)(whole, at[0], at[1], at[2], at[3], at[4], at[5], at[6], at[7], of_values, trees, nodes, edges, warps, depth, on);
        break;
    default:
        code = ((NodeBackup)entry)(whole, at[0], at[1], at[2], at[3], at[4], at[5], at[6], at[7], at[8], of_values, trees, nodes, edges, warps, depth, on);
    }
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(code);
}

/* setup(Tensor, int32, float32, current_device, current_stream) */
static PyObject *setup(PyObject *self, PyObject *args) {
    (void)self;
    PyObject *t, *i, *f, *d, *s;
    if (!PyArg_ParseTuple(args, "OOOOO", &t, &i, &f, &d, &s)) return NULL;
    PyObject **const keep[5] = {&tensor_type, &int32_type, &float32_type, &current_device, &current_stream};
    PyObject *const given[5] = {t, i, f, d, s};
    for (int k = 4; k >= 0; k--) { Py_INCREF(given[k]); Py_XSETREF(*keep[k], given[k]); }
#ifdef PUCT_CALL_DLPACK
    PyObject *table = PyObject_GetAttrString(t, "__dlpack_c_exchange_api__");
    const DLPackExchangeAPI *api = table ? PyCapsule_GetPointer(table, "dlpack_exchange_api") : NULL;
    Py_XDECREF(table);   /* (what it points to is the framework's, for good) */
    PyErr_Clear();
    tensor_of = api && api->header.version.major == DLPACK_MAJOR_VERSION ? api->dltensor_from_py_object_no_sync : NULL;
#endif
    Py_RETURN_NONE;
}

static PyMethodDef methods[] = {{"launch", (PyCFunction)(void (*)(void))launch, METH_FASTCALL, NULL}, {"setup", setup, METH_VARARGS, NULL}, {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_puct_call", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__puct_call(void) {
    PyObject **const names[7] = {&s_shape, &s_dtype, &s_is_cuda, &s_is_contiguous, &s_data_ptr, &s_edge_child, &s_out_path};
    static const char *const text[7] = {"shape", "dtype", "is_cuda", "is_contiguous", "data_ptr", "edge_child", "out_path"};
    for (int i = 0; i < 7; i++) if (!(*names[i] = PyUnicode_InternFromString(text[i]))) return NULL;
    return PyModule_Create(&module);
}
