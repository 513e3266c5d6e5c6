// Plan objects <-> arrays: the parts of a predict_time_breakdown call that walk Python objects (module superscaler_amd._ace_objects).
//
//   encode(...)  AcesoConfig-like objects -> code rows and headers (PlanBatch.from_configs)
//   fill(...), fill_all(...)    stage records -> the lists that predict_time_breakdown leaves on a plan object (CostModel._fill_breakdown)
//
// They handle what a search hands over -- lists of small ints -- and leave everything else (other types, other lengths,
// values outside the profile database, divisions by zero) to the Python code, which raises what it always raised: encode
// and fill_all return the index of the first plan they did not take, fill returns False.  The floating-point operations of fill are
// those of the Python code, one IEEE operation each in the same order (the file is compiled with contraction off), and
// sums of lists go through builtins.sum.
// Getting or setting an attribute may run code that changes the lists at hand: a plan or stage is held while it is read, and a
// list's length is looked at again before the next item is taken.
//
// Per plan of 134 ops: encode 19 -> 2 us, fill 8 -> 3 us.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>
#include <string.h>

namespace {

constexpr int kMaxStages = 16, kRec = 18;
// stage record fields (ACE_R_*)
enum { R_FWD, R_BWD, R_IN_COMM, R_OUT_COMM, R_RECOMP, R_WEIGHTS, R_INPUTS, R_ACT, R_SAVED, R_PEAK, R_RESERVED, R_IDEAL_FWD, R_IDEAL_BWD,
       R_IDEAL_IN, R_IDEAL_OUT };

#define NAMES(X)                                                                                                               \
    X(num_stages) X(micro_bs) X(global_bs) X(stages) X(ops) X(tp_size) X(dp_size) X(algo) X(recompute_ops) X(num_gpus)          \
    X(num_stages_behind) X(time_list) X(memory_list) X(compute_time_list) X(total_gpu_time) X(breakdown_ideal_time_per_gpu)    \
    X(breakdown_eff_loss_time_per_gpu) X(breakdown_recomp_time_per_gpu) X(efficient_time_list)
#define DECLARE(n) PyObject *s_##n;
NAMES(DECLARE)
PyObject *g_sum;

struct Ref {
    PyObject *p;
    explicit Ref(PyObject *o) : p(o) {}
    ~Ref() { Py_XDECREF(p); }
    Ref(const Ref &) = delete;
    Ref &operator=(const Ref &) = delete;
    explicit operator bool() const { return p != nullptr; }
};
inline PyObject *held(PyObject *o) {
    Py_INCREF(o);
    return o;
}

// a small int (bools too); false for anything else
inline bool as_int(PyObject *o, long *v) {
    if (!PyLong_Check(o)) return false;
    int over = 0;
    *v = PyLong_AsLongAndOverflow(o, &over);
    return !over;
}
inline bool int_attr(PyObject *o, PyObject *name, long *v) {
    Ref a(PyObject_GetAttr(o, name));
    return a && as_int(a.p, v);
}

struct EncodeArgs {
    int N, A, gpus_per_node, intra_node, n_mbs, n_lut;
    const int32_t *mbs;
    const uint8_t *tp_lut;
};

inline int mbs_index(const EncodeArgs &a, long m) {
    for (int k = 0; k < a.n_mbs; ++k)
        if (a.mbs[k] == m) return k;
    return -1;
}

// One plan; false: not taken (an exception may be set).
bool encode_one(PyObject *cfg, const EncodeArgs &a, uint8_t *row, uint32_t *hdr) {
    long S, micro;
    if (!int_attr(cfg, s_num_stages, &S) || S < 1 || S > kMaxStages || !int_attr(cfg, s_micro_bs, &micro)) return false;
    const int bidx = mbs_index(a, micro);
    if (bidx < 0) return false;
    Ref stages(PyObject_GetAttr(cfg, s_stages));
    if (!stages || !PyList_Check(stages.p) || PyList_GET_SIZE(stages.p) != S) return false;
    int at = 0;
    uint64_t sizes = 0;
    uint32_t cross = 0;
    long long till = 0;
    for (long s = 0; s < S; ++s) {
        if (s >= PyList_GET_SIZE(stages.p)) return false;
        Ref st(held(PyList_GET_ITEM(stages.p, s)));
        Ref ops(PyObject_GetAttr(st.p, s_ops)), tp(PyObject_GetAttr(st.p, s_tp_size)), dp(PyObject_GetAttr(st.p, s_dp_size)),
            al(PyObject_GetAttr(st.p, s_algo)), rc(PyObject_GetAttr(st.p, s_recompute_ops));
        if (!ops || !tp || !dp || !al || !rc || !PyList_Check(ops.p) || !PyList_Check(tp.p) || !PyList_Check(dp.p) || !PyList_Check(al.p) ||
            !PyList_Check(rc.p))
            return false;
        const Py_ssize_t n = PyList_GET_SIZE(ops.p);
        if (n < 1 || n > a.N - at || PyList_GET_SIZE(tp.p) != n || PyList_GET_SIZE(dp.p) != n || PyList_GET_SIZE(al.p) != n ||
            PyList_GET_SIZE(rc.p) != n)
            return false;
        long g = 0, last_dp = -1;
        for (Py_ssize_t i = 0; i < n; ++i) {
            long t, d, x, r;
            if (!as_int(PyList_GET_ITEM(tp.p, i), &t) || !as_int(PyList_GET_ITEM(dp.p, i), &d) || !as_int(PyList_GET_ITEM(al.p, i), &x) ||
                !as_int(PyList_GET_ITEM(rc.p, i), &r))
                return false;
            if (t < 0 || t >= a.n_lut || a.tp_lut[t] == 0xff || d < 1 || d > 0xffff || x < 0 || x >= a.A) return false;
            if (d != last_dp) {
                if (mbs_index(a, micro / d) < 0) return false;
                last_dp = d;
            }
            if (i == 0) {
                g = t * d;
                if (g < 1 || (g & (g - 1)) || g > (1l << 15)) return false;
            } else if (t * d != g)
                return false;
            row[at + i] = (uint8_t)((a.tp_lut[t] * a.A + x) | (r == 1 ? 8 : 0));
        }
        row[at] |= 16;
        at += (int)n;
        sizes |= (uint64_t)__builtin_ctzl((unsigned long)g) << (4 * s);
        if (till % a.gpus_per_node == 0 && till > 0) cross |= 1u << s;
        till += g;
        if (till % a.gpus_per_node == 0) cross |= 1u << (16 + s);
    }
    if (at != a.N) return false;
    hdr[0] = (uint32_t)S | ((uint32_t)bidx << 8);
    hdr[1] = (uint32_t)sizes;
    hdr[2] = (uint32_t)(sizes >> 32);
    hdr[3] = a.intra_node ? 0u : cross;
    return true;
}

// encode(configs, start, num_ops, n_algo, gpus_per_node, intra_node, mbs (int32 buffer), tp_lut (uint8 buffer), codes, hdr)
PyObject *encode(PyObject *, PyObject *args) {
    PyObject *configs;
    Py_ssize_t start;
    EncodeArgs a;
    Py_buffer mbs, lut, codes, hdr;
    if (!PyArg_ParseTuple(args, "Oniiipy*y*w*w*", &configs, &start, &a.N, &a.A, &a.gpus_per_node, &a.intra_node, &mbs, &lut, &codes, &hdr))
        return nullptr;
    a.mbs = static_cast<const int32_t *>(mbs.buf);
    a.n_mbs = (int)(mbs.len / 4);
    a.tp_lut = static_cast<const uint8_t *>(lut.buf);
    a.n_lut = (int)lut.len;
    Ref seq(PySequence_Fast(configs, "a sequence of plans"));
    Py_ssize_t p = start;
    if (seq) {
        const Py_ssize_t P = PySequence_Fast_GET_SIZE(seq.p);
        if (a.gpus_per_node > 0 && a.N > 0 && codes.len >= P * a.N && hdr.len >= P * 16)
            for (; p < P && p < PySequence_Fast_GET_SIZE(seq.p); ++p) {
                Ref cfg(held(PySequence_Fast_GET_ITEM(seq.p, p)));
                if (!encode_one(cfg.p, a, static_cast<uint8_t *>(codes.buf) + p * a.N, static_cast<uint32_t *>(hdr.buf) + 4 * p)) break;
            }
        if (PyErr_Occurred()) PyErr_Clear();
    }
    PyBuffer_Release(&mbs);
    PyBuffer_Release(&lut);
    PyBuffer_Release(&codes);
    PyBuffer_Release(&hdr);
    return seq ? PyLong_FromSsize_t(p) : nullptr;
}

PyObject *float_list(const double *v, long n) {
    PyObject *l = PyList_New(n);
    for (long i = 0; l && i < n; ++i) {
        PyObject *f = PyFloat_FromDouble(v[i]);
        if (!f) {
            Py_DECREF(l);
            return nullptr;
        }
        PyList_SET_ITEM(l, i, f);
    }
    return l;
}
bool set_list(PyObject *cfg, PyObject *name, const double *v, long n) {
    Ref l(float_list(v, n));
    return l && PyObject_SetAttr(cfg, name, l.p) == 0;
}
bool list_sum(const double *v, long n, double *out) {
    Ref l(float_list(v, n));
    if (!l) return false;
    Ref r(PyObject_CallFunctionObjArgs(g_sum, l.p, nullptr));
    if (!r) return false;
    *out = PyFloat_AsDouble(r.p);
    return !PyErr_Occurred();
}

// One plan from its records: 1, 0 (left to the Python code) or -1 (an exception is set).
int fill_one(PyObject *cfg, const double (*rec)[kRec], double max_mem, double main_params, double optimizer, int reserved_on) {
    long S = 0, global = 0, micro = 0;
    bool ok = int_attr(cfg, s_num_stages, &S) && S >= 1 && S <= kMaxStages && int_attr(cfg, s_global_bs, &global) &&
              int_attr(cfg, s_micro_bs, &micro) && micro > 0 && global >= 0;
    Ref stages(ok ? PyObject_GetAttr(cfg, s_stages) : nullptr);
    ok = ok && stages && PyList_Check(stages.p) && PyList_GET_SIZE(stages.p) >= S;
    double t[kMaxStages], mem[kMaxStages], comp[kMaxStages], gpu[kMaxStages], eff[kMaxStages], ideal[kMaxStages], loss[kMaxStages],
        recomp_l[kMaxStages], gpus[kMaxStages];
    bool recomputes[kMaxStages];
    for (long i = 0; ok && i < S; ++i) {
        const double *r = rec[i];
        if (i >= PyList_GET_SIZE(stages.p)) { ok = false; break; }
        Ref st(held(PyList_GET_ITEM(stages.p, i)));
        long n_gpus, nsb;
        ok = int_attr(st.p, s_num_gpus, &n_gpus) && n_gpus > 0 && n_gpus < (1l << 31) && int_attr(st.p, s_num_stages_behind, &nsb) && nsb >= 0 && nsb < (1l << 31);
        Ref rc(ok ? PyObject_GetAttr(st.p, s_recompute_ops) : nullptr);
        ok = ok && rc && PyList_Check(rc.p);
        if (!ok) break;
        long total = 0;
        for (Py_ssize_t k = 0; k < PyList_GET_SIZE(rc.p) && ok; ++k) {
            long v;
            ok = as_int(PyList_GET_ITEM(rc.p, k), &v) && v >= 0 && v < (1l << 31);
            total += v;
        }
        if (!ok) break;
        recomputes[i] = total > 0;
        const double num_gpus = (double)n_gpus;
        gpus[i] = num_gpus;
        const double fwd = r[R_FWD], bwd = r[R_BWD], in_comm = r[R_IN_COMM], out_comm = r[R_OUT_COMM], recomp = r[R_RECOMP];
        const double sum_time = ((((fwd + bwd) + in_comm) + out_comm) + recomp) / 1000;
        t[i] = sum_time;
        comp[i] = ((fwd + bwd) + recomp) / 1000;
        gpu[i] = sum_time * num_gpus;
        const double f1 = r[R_IDEAL_FWD], b1 = r[R_IDEAL_BWD];
        const double ideal_time = (((f1 + b1) + r[R_IDEAL_IN]) + r[R_IDEAL_OUT]) / 1000;
        const double per = (f1 + b1) / num_gpus;
        loss[i] = ((fwd + bwd) - per) / 1000;
        ideal[i] = per / 1000;
        recomp_l[i] = recomp / 1000;
        const double w = r[R_WEIGHTS], main_p = w * main_params, opt = w * optimizer;
        const double x = (r[R_INPUTS] + r[R_ACT]) - r[R_SAVED];
        const double act = x * (double)nsb, peak = x + r[R_PEAK], wts = w + main_p;
        mem[i] = ((((wts + w) + opt) + act) + peak) + (reserved_on ? r[R_RESERVED] : 0.0);
        const double denom = sum_time * num_gpus;
        ok = denom != 0.0 && mem[i] != 0.0;
        eff[i] = ok ? ideal_time / denom : 0.0;
    }
    double sum_stage = 0.0, sum_gpu = 0.0;
    ok = ok && list_sum(t, S, &sum_stage) && list_sum(gpu, S, &sum_gpu);
    if (!ok) {
        if (PyErr_Occurred()) PyErr_Clear();
        return 0;
    }
    const double nb1 = (double)(global / micro - 1);
    double times[kMaxStages], idle[kMaxStages];
    for (long i = 0; i < S; ++i) times[i] = t[i] * nb1 + sum_stage;
    double max_time = times[0];
    for (long i = 1; i < S; ++i)
        if (times[i] > max_time) max_time = times[i];
    for (long i = 0; i < S; ++i) {
        double v;
        if (recomputes[i]) v = (max_time - times[i]) / 2;
        else {
            const double under_time = max_time - times[i];
            const double under_memory = ((max_mem - mem[i]) / mem[i]) * times[i];
            v = under_memory > under_time ? under_time : under_memory + (under_time - under_memory) / 2;
        }
        idle[i] = v * gpus[i] * eff[i];
    }
    Ref total(PyFloat_FromDouble(sum_gpu * nb1));
    if (!total || !set_list(cfg, s_time_list, times, S) || !set_list(cfg, s_memory_list, mem, S) || !set_list(cfg, s_compute_time_list, comp, S) ||
        PyObject_SetAttr(cfg, s_total_gpu_time, total.p) != 0 || !set_list(cfg, s_breakdown_ideal_time_per_gpu, ideal, S) ||
        !set_list(cfg, s_breakdown_eff_loss_time_per_gpu, loss, S) || !set_list(cfg, s_breakdown_recomp_time_per_gpu, recomp_l, S) ||
        !set_list(cfg, s_efficient_time_list, idle, S))
        return -1;
    return 1;
}

// fill(config, records (double[16][18] buffer), memory_limit, main_params, optimizer, consider_reserved): whether it did
PyObject *fill(PyObject *, PyObject *args) {
    PyObject *cfg;
    Py_buffer buf;
    double max_mem, main_params, optimizer;
    int reserved_on;
    if (!PyArg_ParseTuple(args, "Oy*dddp", &cfg, &buf, &max_mem, &main_params, &optimizer, &reserved_on)) return nullptr;
    double rec[kMaxStages][kRec];
    const bool have = buf.len >= (Py_ssize_t)sizeof(rec);
    if (have) memcpy(rec, buf.buf, sizeof(rec));
    PyBuffer_Release(&buf);
    const int rc = have ? fill_one(cfg, rec, max_mem, main_params, optimizer, reserved_on) : 0;
    if (rc < 0) return nullptr;
    return PyBool_FromLong(rc);
}

// fill_all(configs (a sequence), records (double[n][16][18] buffer), start, memory_limit, main_params, optimizer, consider_reserved):
// the plans from `start` on; returns the index of the first one not taken (all of them: their number)
PyObject *fill_all(PyObject *, PyObject *args) {
    PyObject *configs;
    Py_buffer buf;
    Py_ssize_t p;
    double max_mem, main_params, optimizer;
    int reserved_on;
    if (!PyArg_ParseTuple(args, "Oy*ndddp", &configs, &buf, &p, &max_mem, &main_params, &optimizer, &reserved_on)) return nullptr;
    Ref seq(PySequence_Fast(configs, "fill_all: a sequence of plans"));
    const Py_ssize_t have = buf.len / (Py_ssize_t)(sizeof(double) * kMaxStages * kRec);
    int rc = seq && p >= 0 ? 1 : -1;
    for (; rc == 1 && p < PySequence_Fast_GET_SIZE(seq.p); ++p) {
        double rec[kMaxStages][kRec];                        // (a copy: the buffer need not be aligned)
        rc = p < have;
        if (!rc) break;
        memcpy(rec, static_cast<const char *>(buf.buf) + (size_t)p * sizeof(rec), sizeof(rec));
        Ref cfg(held(PySequence_Fast_GET_ITEM(seq.p, p)));
        rc = fill_one(cfg.p, rec, max_mem, main_params, optimizer, reserved_on);
        if (rc != 1) break;
    }
    PyBuffer_Release(&buf);
    if (rc < 0) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "fill_all: start");
        return nullptr;
    }
    return PyLong_FromSsize_t(p);
}

PyMethodDef methods[] = {{"encode", encode, METH_VARARGS, "plan objects -> code rows and headers; the index of the first plan not taken"},
                         {"fill", fill, METH_VARARGS, "stage records -> the lists of predict_time_breakdown; whether it did"},
                         {"fill_all", fill_all, METH_VARARGS, "the same for a list of plans; the index of the first plan not taken"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ace_objects", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ace_objects(void) {
#define INTERN(n) \
    if (!(s_##n = PyUnicode_InternFromString(#n))) return nullptr;
    NAMES(INTERN)
    Ref builtins(PyImport_ImportModule("builtins"));
    if (!builtins || !(g_sum = PyObject_GetAttrString(builtins.p, "sum"))) return nullptr;
    return PyModule_Create(&module);
}
