/* ops_fast.c: the size checks and the call of attn.Ops.decode / prompt / pre_store in one step of native code.
 *
 * A short context's step is a few microseconds of GPU work, and the wrappers' checks and ctypes' conversion of 18 - 28 arguments
 * took longer than a launch: a token's two calls 15.2 us, of them 10 for three launches. Each function here takes the addresses
 * of the library's entry points, the GPU's handle and the wrapper's own arguments. It returns False and has called nothing
 * where a check fails or an argument is not the plain kind (int, float, a buffer of int ptr and len): the wrapper then goes the
 * general way, which says what is wrong. Else it makes the call, once, and returns True or, where that failed, the library's number:
 * a call may fail behind launches it has made, so the wrapper raises and makes no second one. */
#define Py_LIMITED_API 0x030A0000
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#include "ns_attn.h"
#include "ns_pre.h"

static PyObject *s_ptr, *s_len;

typedef struct {
    void *ptr;
    int64_t len;
} buf_t;

/* what a function returns for a call it has made */
static PyObject *made(int rc) {
    if (rc == 0) Py_RETURN_TRUE;
    return PyLong_FromLong(rc);
}

/* sizes up to 2^31: the products below then fit 128 bits */
static int get_size(PyObject *o, int64_t *v) {
    if (!PyLong_Check(o)) return 0;
    *v = PyLong_AsLongLong(o);
    if (*v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return 0;
    }
    return *v >= 0 && *v <= (int64_t) 1 << 31;
}
static int get_float(PyObject *o, float *v) {
    if (!PyFloat_Check(o) && !PyLong_Check(o)) return 0;
    const double d = PyFloat_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) {
        PyErr_Clear();
        return 0;
    }
    *v = (float) d;
    return 1;
}
static int get_address(PyObject *o, void **v) {
    if (!PyLong_Check(o)) return 0;
    *v = PyLong_AsVoidPtr(o);
    if (!*v) PyErr_Clear();
    return *v != NULL;
}
static int get_buf(PyObject *o, buf_t *b) {
    PyObject *p = PyObject_GetAttr(o, s_ptr), *n = p ? PyObject_GetAttr(o, s_len) : NULL;
    int ok = 0;
    if (p && n && get_address(p, &b->ptr) && PyLong_Check(n)) {
        b->len = PyLong_AsLongLong(n);
        ok = !(b->len == -1 && PyErr_Occurred());
    }
    Py_XDECREF(p);
    Py_XDECREF(n);
    if (!ok) PyErr_Clear();
    return ok;
}

static int64_t elt(int64_t qt) { return qt == 0 ? 4 : qt <= 2 ? 2 : -1; }
static int64_t row_bytes(int64_t kt, int64_t D) { return kt == 1 ? D + D / 32 * 2 : kt == 2 ? D / 2 + D / 32 * 2 : kt == 0 || kt == 3 ? 2 * D : -1; }
/* whether b holds (rows - 1) stride + last elements of e bytes, or n elements */
static int holds(const buf_t *b, int64_t rows, int64_t stride, int64_t last, int64_t e) {
    return (__int128) b->len >= ((__int128) (rows - 1) * stride + last) * e;
}
static int holds3(const buf_t *b, int64_t x, int64_t y, int64_t z) { return (__int128) b->len >= (__int128) x * y * z; }

/* what decode and prompt share: (.., handle, qt, kt, q, qs, kc, vc, T, Hq, Hkv, D, cap, p0, out, ..) */
typedef struct {
    void *g;
    int64_t qt, kt, qs, T, Hq, Hkv, D, cap, p0;
    buf_t q, kc, vc, out;
} pass_t;
static int get_pass(PyObject *const *a, pass_t *p) {
    if (!get_address(a[0], &p->g) || !get_size(a[1], &p->qt) || !get_size(a[2], &p->kt) || !get_buf(a[3], &p->q) || !get_size(a[4], &p->qs) ||
        !get_buf(a[5], &p->kc) || !get_buf(a[6], &p->vc) || !get_size(a[7], &p->T) || !get_size(a[8], &p->Hq) || !get_size(a[9], &p->Hkv) ||
        !get_size(a[10], &p->D) || !get_size(a[11], &p->cap) || !get_size(a[12], &p->p0) || !get_buf(a[13], &p->out))
        return 0;
    const int64_t e = elt(p->qt), rb = row_bytes(p->kt, p->D);
    return e > 0 && rb >= 0 && p->T > 0 && holds(&p->q, p->T, p->qs, p->Hq * p->D, e) && holds3(&p->out, p->T * e, p->Hq, p->D) &&
           holds3(&p->kc, p->Hkv, p->cap, rb) && holds3(&p->vc, p->Hkv, p->cap, rb);
}

/* decode(scratch entry, entry, handle, qt, kt, q, qs, kc, vc, T, Hq, Hkv, D, cap, p0, out, scratch, win, pm, scale) */
static PyObject *fast_decode(PyObject *self, PyObject *const *a, Py_ssize_t n) {
    void *fs, *fd;
    pass_t p;
    buf_t sc;
    int64_t win;
    float scale;
    if (n == 20 && get_address(a[0], &fs) && get_address(a[1], &fd) && get_pass(a + 2, &p) && get_buf(a[16], &sc) && get_size(a[17], &win) &&
        PyBool_Check(a[18]) && get_float(a[19], &scale)) {
        __typeof__(&ns_attn_decode_scratch) scratch = (__typeof__(&ns_attn_decode_scratch)) fs;
        __typeof__(&ns_attn_decode_t) decode = (__typeof__(&ns_attn_decode_t)) fd;
        int rc = 0, fits;
        Py_BEGIN_ALLOW_THREADS
        fits = (__int128) sc.len >= (__int128) scratch(p.T, p.Hq, p.Hkv, p.D, p.p0, win) * 4;
        if (fits)
            rc = decode((ns_gpu *) p.g, (int) p.qt, (int) p.kt, a[18] == Py_True, p.q.ptr, p.qs, p.kc.ptr, p.vc.ptr, p.T, p.Hq, p.Hkv, p.D, p.cap, p.p0, win,
                        scale, p.out.ptr, (float *) sc.ptr);
        Py_END_ALLOW_THREADS
        if (fits) return made(rc);
    }
    Py_RETURN_FALSE;
}

/* prompt(entry, handle, qt, kt, q, qs, kc, vc, T, Hq, Hkv, D, cap, p0, out, win, pm, scale) */
static PyObject *fast_prompt(PyObject *self, PyObject *const *a, Py_ssize_t n) {
    void *f;
    pass_t p;
    int64_t win;
    float scale;
    if (n == 18 && get_address(a[0], &f) && get_pass(a + 1, &p) && get_size(a[15], &win) && PyBool_Check(a[16]) && get_float(a[17], &scale)) {
        __typeof__(&ns_attn_prompt_t) prompt = (__typeof__(&ns_attn_prompt_t)) f;
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = prompt((ns_gpu *) p.g, (int) p.qt, (int) p.kt, a[16] == Py_True, p.q.ptr, p.qs, p.kc.ptr, p.vc.ptr, p.T, p.Hq, p.Hkv, p.D, p.cap, p.p0, win, scale,
                    p.out.ptr);
        Py_END_ALLOW_THREADS
        return made(rc);
    }
    Py_RETURN_FALSE;
}

/* pre_store(entry, handle, rope, qt, kt, ring, q, qss, qhs, qo, qos, k, kss, khs, v, vss, qw, kw, eps, n_rot, theta, T, Hq, Hkv, D, cap, p0, kc, vc) */
static PyObject *fast_pre_store(PyObject *self, PyObject *const *a, Py_ssize_t n) {
    void *f, *g;
    buf_t q, qo, k, v, qw, kw, kc, vc;
    int64_t rope, qt, kt, qss, qhs, qos, kss, khs, vss, n_rot, T, Hq, Hkv, D, cap, p0;
    float eps, theta;
    if (n == 29 && get_address(a[0], &f) && get_address(a[1], &g) && get_size(a[2], &rope) && get_size(a[3], &qt) && get_size(a[4], &kt) && PyBool_Check(a[5]) &&
        get_buf(a[6], &q) && get_size(a[7], &qss) && get_size(a[8], &qhs) && get_buf(a[9], &qo) && get_size(a[10], &qos) && get_buf(a[11], &k) &&
        get_size(a[12], &kss) && get_size(a[13], &khs) && get_buf(a[14], &v) && get_size(a[15], &vss) && get_buf(a[16], &qw) && get_buf(a[17], &kw) &&
        get_float(a[18], &eps) && get_size(a[19], &n_rot) && get_float(a[20], &theta) && get_size(a[21], &T) && get_size(a[22], &Hq) &&
        get_size(a[23], &Hkv) && get_size(a[24], &D) && get_size(a[25], &cap) && get_size(a[26], &p0) && get_buf(a[27], &kc) && get_buf(a[28], &vc)) {
        const int64_t e = elt(qt), rb = row_bytes(kt, D);
        if (e > 0 && rb >= 0 && T > 0 && Hq > 0 && Hkv > 0 && holds(&q, T, qss, (Hq - 1) * qhs + D, 4) && holds(&qo, T, qos, Hq * D, e) &&
            holds(&k, T, kss, (Hkv - 1) * khs + D, 4) && holds(&v, T, vss, Hkv * D, 4) && qw.len >= D * 4 && kw.len >= D * 4 &&
            holds3(&kc, Hkv, cap, rb) && holds3(&vc, Hkv, cap, rb)) {
            __typeof__(&ns_attn_pre_store) pre = (__typeof__(&ns_attn_pre_store)) f;
            int rc;
            Py_BEGIN_ALLOW_THREADS
            rc = pre((ns_gpu *) g, (int) rope, (int) qt, (int) kt, a[5] == Py_True, (const float *) q.ptr, qss, qhs, qo.ptr, qos, (const float *) k.ptr, kss, khs,
                     (const float *) v.ptr, vss, (const float *) qw.ptr, (const float *) kw.ptr, eps, n_rot, theta, T, Hq, Hkv, D, cap, p0, kc.ptr, vc.ptr);
            Py_END_ALLOW_THREADS
            return made(rc);
        }
    }
    Py_RETURN_FALSE;
}

static PyMethodDef methods[] = {{"decode", (PyCFunction) (void (*)(void)) fast_decode, METH_FASTCALL, "attn.Ops.decode's checks and call"},
                                {"prompt", (PyCFunction) (void (*)(void)) fast_prompt, METH_FASTCALL, "attn.Ops.prompt's checks and call"},
                                {"pre_store", (PyCFunction) (void (*)(void)) fast_pre_store, METH_FASTCALL, "attn.Ops.pre_store's checks and call"},
                                {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ops_fast", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__ops_fast(void) {
    s_ptr = PyUnicode_InternFromString("ptr");
    s_len = PyUnicode_InternFromString("len");
    return s_ptr && s_len ? PyModule_Create(&module) : NULL;
}
