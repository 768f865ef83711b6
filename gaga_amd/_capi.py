"""ctypes binding of libgaga_amd.so (declarations in include/gaga_amd.h)."""
import ctypes
import os

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.environ.get("XCS_LIB_PATH", os.path.join(_HERE, "libgaga_amd.so"))

# every symbol include/gaga_amd.h declares
EXPORTS = (
    "xcs_options_default", "xcs_cs_generate", "xcs_cs_gen", "xcs_cs_smv", "xcs_cs_dct",
    "xcs_plan_create", "xcs_plan_solve", "xcs_plan_results", "xcs_plan_trace", "xcs_plan_timings",
    "xcs_plan_times", "xcs_results_timing_text", "xcs_results_timing_append",
    "xcs_plan_destroy", "xcs_plan_bytes", "xcs_plan_apply_timed", "xcs_plan_geometry",
    "xcs_batch_create", "xcs_batch_bytes", "xcs_batch_apply_timed", "xcs_batch_solve",
    "xcs_batch_results", "xcs_batch_configure", "xcs_batch_tune",
    "xcs_batch_x", "xcs_batch_info", "xcs_batch_destroy", "xcs_batch_phase_ticks",
    "xcs_find_support_set", "xcs_apply", "xcs_generate_gen", "xcs_generate_smv", "xcs_gemm_tn",
    "xcs_mrhs_create", "xcs_mrhs_solve", "xcs_mrhs_results", "xcs_mrhs_x",
    "xcs_mrhs_gemm_timed", "xcs_mrhs_phase_ms", "xcs_mrhs_fp32_solve", "xcs_mrhs_configure",
    "xcs_mrhs_samples", "xcs_mrhs_gemm_tile", "xcs_mlp_create", "xcs_mlp_destroy", "xcs_mlp_param_count",
    "xcs_mlp_get_params", "xcs_mlp_set_params", "xcs_mlp_grad", "xcs_mlp_scores",
    "xcs_mlp_set_data", "xcs_mlp_train", "xcs_plan_solve_warm", "xcs_mlp_features", "xcs_stream_copy", "xcs_mrhs_destroy",
    "xcs_last_error", "xcs_version", "xcs_results_line", "xcs_results_append",
    "xcs_cs_gen_noalloc", "xcs_batch_schedule", "xcs_batch_phase_counts", "xcs_stream_read",
    "xcs_batch_schedule_mode", "xcs_batch_exact", "xcs_batch_ran", "xcs_plan_form",
    "xcs_mrhs_row_blocks",
)


class GagaError(RuntimeError):
    """A non-zero status from the C ABI."""

    def __init__(self, code, msg):
        super().__init__("xcs error %d: %s" % (code, msg))
        self.code = code


class Options(ctypes.Structure):
    _fields_ = [
        ("tol", ctypes.c_float), ("tol_reference_default", ctypes.c_int),
        ("maxiter", ctypes.c_int), ("num_bins", ctypes.c_int), ("restart", ctypes.c_int),
        ("seed", ctypes.c_uint), ("instance", ctypes.c_uint),
        ("vec_distribution", ctypes.c_int), ("matrix_ensemble", ctypes.c_int),
        ("gpu_number", ctypes.c_int), ("mode", ctypes.c_int), ("team_size", ctypes.c_int),
        ("block_size", ctypes.c_int), ("proj_frac_tol", ctypes.c_float),
        ("timing", ctypes.c_int), ("supp_flag", ctypes.c_int), ("alpha", ctypes.c_float),
        ("barrier_spin_limit", ctypes.c_long),
    ]


_lib = None
_P = ctypes.c_void_p
_I = ctypes.c_int
_F = ctypes.c_float
_C = ctypes.c_char_p


def load():
    """Load libgaga_amd.so (raises if it has not been built)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise OSError("libgaga_amd.so not built: run `make -C gaga_amd` (or __graft_entry__.build())")
        L = ctypes.CDLL(LIB_PATH)
        L.xcs_options_default.argtypes = [_C, _C, _I, _P]
        L.xcs_cs_generate.argtypes = [_C, _C, _I, _I, _I, _I, _P, _P, _P, _P, _P, _P, _P, _P]
        L.xcs_cs_gen.argtypes = [_C, _P, _P, _I, _I, _I, _P, _P, _P, _P]
        L.xcs_cs_smv.argtypes = [_C, _P, _P, _P, _P, _I, _I, _I, _I, _P, _P, _P, _P]
        L.xcs_cs_dct.argtypes = [_C, _P, _P, _I, _I, _I, _P, _P, _P, _P]
        L.xcs_cs_gen_noalloc.argtypes = [_C, _P, _P, _I, _I, _I, _I, _P, _P, _P, _P, _P]
        L.xcs_results_line.argtypes = [ctypes.c_char_p, ctypes.c_size_t, _C, _C, _I, _I, _I, _I, _I,
                                       _I, _P, _P, _I, ctypes.c_float, _P, ctypes.c_uint]
        L.xcs_results_append.argtypes = [_C, _C, _C, _I, _I, _I, _I, _I, _I, _P, _P, _I,
                                         ctypes.c_float, _P, ctypes.c_uint]
        L.xcs_plan_create.argtypes = [_C, _C, _I, _I, _I, _I, _P, _P]
        L.xcs_plan_solve.argtypes = [_P, _P]
        L.xcs_plan_results.argtypes = [_P, _P, _P, _P, _P, _P, _P, _P]
        L.xcs_plan_trace.argtypes = [_P, _P, _P, _I]
        L.xcs_plan_timings.argtypes = [_P, _P, _P, _P, _P, _I]
        L.xcs_plan_times.argtypes = [_P, _P]
        _tline = [_I, _I, _I, _I, _I, _I, _P, _P, _I, ctypes.c_float, _P, ctypes.c_uint,
                  ctypes.c_float, _I, _P, _P, _P, _P]
        L.xcs_results_timing_text.argtypes = [_P, ctypes.c_size_t, _P, _P] + _tline
        L.xcs_results_timing_append.argtypes = [_P, _P, _P] + _tline
        L.xcs_plan_destroy.argtypes = [_P]
        L.xcs_plan_destroy.restype = None
        L.xcs_plan_bytes.argtypes = [_P, _P]
        L.xcs_plan_geometry.argtypes = [_P, _P, _P]
        L.xcs_plan_form.argtypes = [_P, _P, _P, _P, _P]
        L.xcs_plan_apply_timed.argtypes = [_P, _I, _I, _P, _P]
        L.xcs_batch_bytes.argtypes = [_P, _P]
        L.xcs_batch_apply_timed.argtypes = [_P, _I, _P, _P]
        L.xcs_batch_create.argtypes = [_C, _I, _P, _P, _P, _P, _P, _P, _P, _P]
        L.xcs_batch_solve.argtypes = [_P, _P]
        L.xcs_batch_configure.argtypes = [_P, _I, _I, _I]
        L.xcs_batch_schedule.argtypes = [_P, _I, _P, _P]
        L.xcs_batch_phase_counts.argtypes = [_P, _P, _I]
        L.xcs_batch_schedule_mode.argtypes = [_P, _I, _I]
        L.xcs_gemm_tn.argtypes = [_C, _I, _I, _I, _P, _P, _P, _P, _P]
        L.xcs_mrhs_create.argtypes = [_I, _I, _I, _I, _C, _P, _P]
        L.xcs_mrhs_solve.argtypes = [_P, _P, _P]
        L.xcs_mrhs_results.argtypes = [_P, _P, _P, _P]
        L.xcs_mrhs_x.argtypes = [_P, _I, _P, _P, _P]
        L.xcs_mrhs_gemm_timed.argtypes = [_P, _I, _C, _I, _P, _P]
        L.xcs_mrhs_phase_ms.argtypes = [_P, _P]
        L.xcs_mrhs_samples.argtypes = [_P, _I, ctypes.c_uint, _P, _P]
        L.xcs_mrhs_row_blocks.argtypes = [_P, _I]
        L.xcs_mrhs_gemm_tile.argtypes = [_P, _I]
        L.xcs_mlp_create.argtypes = [ctypes.c_uint, _P]
        L.xcs_mlp_destroy.argtypes = [_P]
        L.xcs_mlp_destroy.restype = None
        L.xcs_mlp_param_count.argtypes = []
        L.xcs_mlp_get_params.argtypes = [_P, _P]
        L.xcs_mlp_set_params.argtypes = [_P, _P]
        L.xcs_mlp_grad.argtypes = [_P, _P, _P, _I, ctypes.c_float, _P, _P]
        L.xcs_mlp_scores.argtypes = [_P, _P, _I, _P]
        L.xcs_mlp_set_data.argtypes = [_P, _P, _P, ctypes.c_long]
        L.xcs_mlp_train.argtypes = [_P, _I, _I, ctypes.c_float, ctypes.c_float, _P, _P]
        L.xcs_plan_solve_warm.argtypes = [_P, _P, _I, _P, _P, _P]
        L.xcs_mlp_features.argtypes = [_P, _I, _I, _I, _P]
        L.xcs_stream_copy.argtypes = [ctypes.c_long, _I, _P]
        L.xcs_stream_read.argtypes = [ctypes.c_long, _I, _P]
        L.xcs_mrhs_configure.argtypes = [_P, ctypes.c_float, ctypes.c_float, _I, _I, _I]
        L.xcs_mrhs_fp32_solve.argtypes = [_P, _I, _I, _I, _P, _P, _P]
        L.xcs_mrhs_destroy.argtypes = [_P]
        L.xcs_mrhs_destroy.restype = None
        L.xcs_batch_tune.argtypes = [_P, _I, _C, _I, _P, _P, _P, _P]
        L.xcs_batch_results.argtypes = [_P, _P, _P, _P, _P]
        L.xcs_batch_x.argtypes = [_P, _I, _P, _P]
        L.xcs_batch_info.argtypes = [_P, _P, _P, _P, _P]
        L.xcs_batch_exact.argtypes = [_P, _I]
        L.xcs_batch_ran.argtypes = [_P, _P, _P]
        L.xcs_batch_destroy.argtypes = [_P]
        L.xcs_batch_destroy.restype = None
        L.xcs_batch_phase_ticks.argtypes = [_P, _P]
        L.xcs_find_support_set.argtypes = [_P, _I, _I, _I, _F, _F, _F, _P, _P, _P, _P, _P, _P]
        L.xcs_apply.argtypes = [_C, _I, _I, _I, _P, _P, _P, _P, _P, _P, _P]
        L.xcs_generate_gen.argtypes = [_I, _I, ctypes.c_uint, ctypes.c_uint, _P]
        L.xcs_generate_smv.argtypes = [_I, _I, _I, _I, ctypes.c_uint, ctypes.c_uint, _P, _P, _P,
                                       _P, _P, _P]
        L.xcs_last_error.restype = _C
        L.xcs_version.restype = _C
        _lib = L
    return _lib


def _ck(code):
    if code != 0:
        raise GagaError(code, load().xcs_last_error().decode())


def _p(a):
    return None if a is None else a.ctypes.data_as(ctypes.c_void_p)


def default_options(alg, ens, n):
    o = Options()
    _ck(load().xcs_options_default(alg.encode(), ens.encode(), int(n), ctypes.byref(o)))
    return o


def generate(alg, ens, k, m, n, p, o):
    norms = np.zeros(3, np.float32)
    times = np.zeros(3, np.float32)
    it = ctypes.c_int(0)
    sup = np.zeros(4, np.int32)
    rate = ctypes.c_float(0)
    x = np.zeros(n, np.float32)
    _ck(load().xcs_cs_generate(alg.encode(), ens.encode(), k, m, n, p, ctypes.byref(o), _p(norms),
                               _p(times), ctypes.byref(it), _p(sup), ctypes.byref(rate), _p(x),
                               None))
    return norms, times, it.value, sup, rate.value, x


def _line_args(alg, ens, k, m, n, p, o, norms, times, iters, sup, rate):
    norms = np.ascontiguousarray(norms, np.float32)
    times = np.ascontiguousarray(times, np.float32)
    sup = np.ascontiguousarray(sup, np.int32)
    return (alg.encode(), ens.encode(), int(k), int(m), int(n), int(p), int(o.matrix_ensemble),
            int(o.vec_distribution), _p(norms), _p(times), int(iters), float(rate), _p(sup),
            int(o.seed) & 0xFFFFFFFF), (norms, times, sup)


def results_line(alg, ens, k, m, n, p, o, norms, times, iters, sup, rate):
    """The reference's per-solve results line (File_output*, functions.cu:34-80)."""
    args, keep = _line_args(alg, ens, k, m, n, p, o, norms, times, iters, sup, rate)
    buf = ctypes.create_string_buffer(1024)
    r = load().xcs_results_line(buf, 1024, *args)
    if r < 0:
        _ck(r)
    return buf.value.decode()


def results_append(directory, alg, ens, k, m, n, p, o, norms, times, iters, sup, rate):
    """Append the results line to <directory>/gpu_data_<ens>YYYYMMDD.txt (results.cu:509-525)."""
    args, keep = _line_args(alg, ens, k, m, n, p, o, norms, times, iters, sup, rate)
    _ck(load().xcs_results_append(str(directory).encode(), *args))


def _timing_args(alg, ens, k, m, n, p, o, norms, times, iters, sup, rate, alpha, supp_flag,
                 t_iter, t_supp, cg, t_cg):
    args, keep = _line_args(alg, ens, k, m, n, p, o, norms, times, iters, sup, rate)
    arrs = [np.ascontiguousarray(t_iter, np.float32), np.ascontiguousarray(t_supp, np.float32),
            None if cg is None else np.ascontiguousarray(cg, np.int32),
            None if t_cg is None else np.ascontiguousarray(t_cg, np.float32)]
    return args[2:] + (float(alpha), int(supp_flag)) + tuple(_p(a) if a is not None else None
                                                             for a in arrs), (keep, arrs, args)


def results_timing_text(alg, ens, k, m, n, p, o, norms, times, iters, sup, rate, alpha, supp_flag,
                        t_iter, t_supp, cg=None, t_cg=None):
    """The timing variants' results text (File_output_timings*, functions.cu:82-212)."""
    rest, keep = _timing_args(alg, ens, k, m, n, p, o, norms, times, iters, sup, rate, alpha,
                              supp_flag, t_iter, t_supp, cg, t_cg)
    size = 1024 + 160 * max(int(iters), 0)
    buf = ctypes.create_string_buffer(size)
    r = load().xcs_results_timing_text(buf, size, alg.encode(), ens.encode(), *rest)
    if r < 0:
        _ck(r)
    return buf.value.decode()


def results_timing_append(directory, alg, ens, k, m, n, p, o, norms, times, iters, sup, rate,
                          alpha, supp_flag, t_iter, t_supp, cg=None, t_cg=None):
    """Append it to <directory>/gpu_timings_data_<ens>YYYYMMDD.txt (results.cu:1540-1560)."""
    rest, keep = _timing_args(alg, ens, k, m, n, p, o, norms, times, iters, sup, rate, alpha,
                              supp_flag, t_iter, t_supp, cg, t_cg)
    _ck(load().xcs_results_timing_append(str(directory).encode(), alg.encode(), ens.encode(), *rest))


def solve_gen(alg, y, A, k, o):
    m, n = A.shape
    Acm = np.asfortranarray(A, dtype=np.float32)  # column-major
    x = np.zeros(n, np.float32)
    it = ctypes.c_int(0)
    rate = ctypes.c_float(0)
    y = np.ascontiguousarray(y, np.float32)
    _ck(load().xcs_cs_gen(alg.encode(), _p(y), Acm.ctypes.data_as(ctypes.c_void_p), m, n, k,
                          ctypes.byref(o), _p(x), ctypes.byref(it), ctypes.byref(rate)))
    return x, it.value, rate.value


def solve_smv(alg, y, rows, cols, vals, m, n, k, o):
    x = np.zeros(n, np.float32)
    it = ctypes.c_int(0)
    rate = ctypes.c_float(0)
    rows = np.ascontiguousarray(rows, np.int32)
    cols = np.ascontiguousarray(cols, np.int32)
    vals = np.ascontiguousarray(vals, np.float32)
    y = np.ascontiguousarray(y, np.float32)
    _ck(load().xcs_cs_smv(alg.encode(), _p(y), _p(rows), _p(cols), _p(vals), rows.size, m, n, k,
                          ctypes.byref(o), _p(x), ctypes.byref(it), ctypes.byref(rate)))
    return x, it.value, rate.value


def solve_dct(alg, y, rows, k, m, n, o):
    x = np.zeros(n, np.float32)
    it = ctypes.c_int(0)
    rate = ctypes.c_float(0)
    rows = np.ascontiguousarray(rows, np.int32)
    y = np.ascontiguousarray(y, np.float32)
    _ck(load().xcs_cs_dct(alg.encode(), _p(y), _p(rows), k, m, n, ctypes.byref(o), _p(x),
                          ctypes.byref(it), ctypes.byref(rate)))
    return x, it.value, rate.value


def find_support_set(v, k, num_bins, slope, intercept, max_change, min_val, alpha, max_bin, k_bin):
    """Device FindSupportSet; returns (sum, bins, state) like oracle.find_support_set."""
    v = np.ascontiguousarray(v, np.float32)
    bins = np.zeros(v.size, np.int32)
    mv = ctypes.c_float(min_val)
    al = ctypes.c_float(alpha)
    mb = ctypes.c_int(max_bin)
    kb = ctypes.c_int(k_bin)
    s = ctypes.c_int(0)
    _ck(load().xcs_find_support_set(_p(v), v.size, k, num_bins, slope, intercept, max_change,
                                    ctypes.byref(mv), ctypes.byref(al), ctypes.byref(mb),
                                    ctypes.byref(kb), _p(bins), ctypes.byref(s)))
    return s.value, bins, dict(min_val=mv.value, alpha=al.value, max_bin=mb.value, k_bin=kb.value)


def apply(ens, transpose, m, n, vec, A=None, col_ptr=None, rows=None, vals=None, dct_rows=None):
    """y = A x (transpose=0) or g = A^T r (transpose=1) on the device."""
    vec = np.ascontiguousarray(vec, np.float32)
    out = np.zeros(n if transpose else m, np.float32)
    Acm = None if A is None else np.asfortranarray(A, dtype=np.float32)
    conv = lambda a, t: None if a is None else np.ascontiguousarray(a, t)  # noqa: E731
    col_ptr, rows, vals, dct_rows = (conv(col_ptr, np.int32), conv(rows, np.int32),
                                     conv(vals, np.float32), conv(dct_rows, np.int32))
    _ck(load().xcs_apply(ens.encode(), int(transpose), m, n,
                         None if Acm is None else Acm.ctypes.data_as(ctypes.c_void_p),
                         _p(col_ptr), _p(rows), _p(vals), _p(dct_rows), _p(vec), _p(out)))
    return out


def generate_gen(m, n, seed, instance):
    A = np.zeros((n, m), np.float32)  # row j = column j of A
    _ck(load().xcs_generate_gen(m, n, seed, instance, _p(A)))
    return A


def generate_smv(m, n, p, ens, seed, instance):
    """The device smv generator: (rows, vals, row_ptr, cols, rvals, empty rows repaired)."""
    nz = n * p
    rows = np.empty(nz, np.int32)
    vals = np.empty(nz, np.float32)
    row_ptr = np.empty(m + 1, np.int32)
    cols = np.empty(nz, np.int32)
    rvals = np.empty(nz, np.float32)
    empty = ctypes.c_int(0)
    _ck(load().xcs_generate_smv(m, n, p, ens, seed, instance, _p(rows), _p(vals), _p(row_ptr),
                                _p(cols), _p(rvals), ctypes.byref(empty)))
    return rows, vals, row_ptr, cols, rvals, empty.value


class Plan:
    """A generated instance kept resident in HBM (xcs_plan_*)."""

    def __init__(self, alg, ens, k, m, n, p=0, opts=None):
        self.alg, self.ens, self.k, self.m, self.n, self.p = alg, ens, k, m, n, p
        from . import _apply_options
        o = _apply_options(alg, ens, n, opts)
        self.maxiter = o.maxiter
        h = ctypes.c_void_p()
        _ck(load().xcs_plan_create(alg.encode(), ens.encode(), k, m, n, p, ctypes.byref(o),
                                   ctypes.byref(h)))
        self._h = h

    def solve(self):
        ms = ctypes.c_float(0)
        _ck(load().xcs_plan_solve(self._h, ctypes.byref(ms)))
        return ms.value

    def results(self):
        norms = np.zeros(3, np.float32)
        sup = np.zeros(4, np.int32)
        it = ctypes.c_int(0)
        rate = ctypes.c_float(0)
        reason = ctypes.c_int(0)
        x = np.empty(self.n, np.float32)  # both filled by the call
        xt = np.empty(self.n, np.float32)
        _ck(load().xcs_plan_results(self._h, _p(norms), ctypes.byref(it), _p(sup),
                                    ctypes.byref(rate), ctypes.byref(reason), _p(x), _p(xt)))
        return dict(norms=norms, iters=it.value, support=sup, conv_rate=rate.value,
                    stop_reason=reason.value, x=x, x_true=xt)

    def bytes(self):
        b = ctypes.c_double(0)
        _ck(load().xcs_plan_bytes(self._h, ctypes.byref(b)))
        return b.value

    def geometry(self):
        """(team_size, block_size) the plan runs with."""
        t, b = ctypes.c_int(0), ctypes.c_int(0)
        _ck(load().xcs_plan_geometry(self._h, ctypes.byref(t), ctypes.byref(b)))
        return t.value, b.value

    def form(self):
        """(form, support bits in LDS, workgroups with their rows' entries in LDS, with
        their columns'): form is "general", "resident" or "split"."""
        v = [ctypes.c_int(0) for _ in range(4)]
        _ck(load().xcs_plan_form(self._h, *[ctypes.byref(q) for q in v]))
        return ("general", "resident", "split")[v[0].value], bool(v[1].value), v[2].value, v[3].value

    def solve_warm(self, net=None, cg_steps=3):
        """CGIHT from the network's predicted support (net None: the k largest
        |A^T y|), plain CGIHT as fallback: (total ms, ms before the warm CGIHT,
        fallback used)."""
        ms, wms, fb = ctypes.c_float(0), ctypes.c_float(0), ctypes.c_int(0)
        _ck(load().xcs_plan_solve_warm(self._h, net._h if net is not None else None,
                                       int(cg_steps), ctypes.byref(ms), ctypes.byref(wms),
                                       ctypes.byref(fb)))
        return ms.value, wms.value, bool(fb.value)

    def apply_timed(self, transpose, reps):
        ms = ctypes.c_float(0)
        b = ctypes.c_double(0)
        _ck(load().xcs_plan_apply_timed(self._h, int(transpose), int(reps), ctypes.byref(ms),
                                        ctypes.byref(b)))
        return ms.value, b.value

    def trace(self, length):
        kb = np.zeros(length, np.int32)
        er = np.zeros(length, np.float32)
        _ck(load().xcs_plan_trace(self._h, _p(kb), _p(er), length))
        return kb, er

    def times(self):
        """(solve ms, ms per iteration, solve + generation ms) of the last solve."""
        t = np.zeros(3, np.float32)
        _ck(load().xcs_plan_times(self._h, _p(t)))
        return t

    def timings(self, length):
        """Per-iteration (iteration ms, support-set ms, CG iterations, CG ms) of the last
        solve with timing on (NIHT, HTP)."""
        it = np.zeros(length, np.float32)
        sp = np.zeros(length, np.float32)
        cg = np.zeros(length, np.int32)
        cm = np.zeros(length, np.float32)
        _ck(load().xcs_plan_timings(self._h, _p(it), _p(sp), _p(cg), _p(cm), length))
        return it, sp, cg, cm

    def close(self):
        if self._h:
            load().xcs_plan_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


ENS_CODE = {"gen": 0, "smv": 1, "dct": 2}


class Batch:
    """Many independent instances solved in one persistent launch (xcs_batch_*).

    specs: list of dicts with keys ens, k, m, n and optionally p, instance.
    """

    def __init__(self, alg, specs, opts=None):
        from . import _apply_options
        self.alg = alg
        self.count = len(specs)
        ens = np.array([ENS_CODE[s["ens"]] for s in specs], np.int32)
        k = np.array([s["k"] for s in specs], np.int32)
        m = np.array([s["m"] for s in specs], np.int32)
        n = np.array([s["n"] for s in specs], np.int32)
        p = np.array([s.get("p", 0) for s in specs], np.int32)
        inst = np.array([s.get("instance", i) for i, s in enumerate(specs)], np.uint32)
        self.n = n
        first = specs[0]["ens"]
        o = _apply_options(alg, first, int(n.max()), opts)
        if any(s["ens"] == "smv" for s in specs) and not any(
                name == "matrixEnsemble" for name, _ in (opts or [])):
            o.matrix_ensemble = 2
        h = ctypes.c_void_p()
        _ck(load().xcs_batch_create(alg.encode(), self.count, _p(ens), _p(k), _p(m), _p(n), _p(p),
                                    _p(inst), ctypes.byref(o), ctypes.byref(h)))
        self._h = h

    def solve(self):
        ms = ctypes.c_float(0)
        _ck(load().xcs_batch_solve(self._h, ctypes.byref(ms)))
        return ms.value

    def results(self):
        norms = np.zeros((self.count, 3), np.float32)
        it = np.zeros(self.count, np.int32)
        reason = np.zeros(self.count, np.int32)
        rate = np.zeros(self.count, np.float32)
        _ck(load().xcs_batch_results(self._h, _p(norms), _p(it), _p(reason), _p(rate)))
        return dict(norms=norms, iters=it, stop_reason=reason, conv_rate=rate)

    def x(self, i):
        x = np.empty(int(self.n[i]), np.float32)  # both filled by the call
        xt = np.empty(int(self.n[i]), np.float32)
        _ck(load().xcs_batch_x(self._h, i, _p(x), _p(xt)))
        return x, xt

    def bytes(self):
        b = ctypes.c_double(0)
        _ck(load().xcs_batch_bytes(self._h, ctypes.byref(b)))
        return b.value

    def apply_timed(self, reps):
        ms = ctypes.c_float(0)
        b = ctypes.c_double(0)
        _ck(load().xcs_batch_apply_timed(self._h, int(reps), ctypes.byref(ms), ctypes.byref(b)))
        return ms.value, b.value

    def schedule(self, team_sizes=(), budgets=(), adaptive=True, split=4):
        """Tail schedule (xcs_batch_schedule): phase 0 runs every instance for
        budgets[0] iterations on the configured geometry, phase p > 0 gives the
        instances still running teams of team_sizes[p] (the last phase until done).
        Empty: one launch.  adaptive (xcs_batch_schedule_mode): the phases run in
        one persistent launch with teams formed on the device, and (split >= 2) the
        last phase-0 solves are finished by teams of `split`; False: one launch
        per phase."""
        t = np.asarray(team_sizes, np.int32)
        b = np.asarray(budgets, np.int32)
        assert len(t) == len(b)
        _ck(load().xcs_batch_schedule(self._h, len(t), _p(t) if len(t) else None,
                                      _p(b) if len(b) else None))
        _ck(load().xcs_batch_schedule_mode(self._h, 1 if adaptive else 0, int(split)))

    def phase_counts(self, phases):
        out = np.zeros(phases, np.int32)
        _ck(load().xcs_batch_phase_counts(self._h, _p(out), phases))
        return out

    def configure(self, team_size, block_size, big_count=-1, exact=False):
        """team_size workgroups per instance for the big_count largest instances
        (-1: all), one workgroup for the rest.  Where the chip has room a solve takes
        larger teams, unless exact is set (ran() tells)."""
        _ck(load().xcs_batch_configure(self._h, int(team_size), int(block_size), int(big_count)))
        _ck(load().xcs_batch_exact(self._h, 1 if exact else 0))

    def ran(self):
        """(teams, team_size) of the last solve."""
        t, c = ctypes.c_int(), ctypes.c_int()
        _ck(load().xcs_batch_ran(self._h, ctypes.byref(t), ctypes.byref(c)))
        return t.value, c.value

    def tune(self, probe_iters=32, cache=None, verbose=False):
        """Pick the team geometry by timing candidates on this batch; returns
        (team_size, block_size, big_count, probe_ms)."""
        c, b, g, t = ctypes.c_int(), ctypes.c_int(), ctypes.c_int(), ctypes.c_float()
        path = cache.encode() if cache else None
        _ck(load().xcs_batch_tune(self._h, int(probe_iters), path, 1 if verbose else 0,
                                  ctypes.byref(c), ctypes.byref(b), ctypes.byref(g),
                                  ctypes.byref(t)))
        return c.value, b.value, g.value, t.value

    def info(self):
        t, c, b, g = ctypes.c_int(), ctypes.c_int(), ctypes.c_int(), ctypes.c_float()
        _ck(load().xcs_batch_info(self._h, ctypes.byref(t), ctypes.byref(c), ctypes.byref(b),
                                  ctypes.byref(g)))
        return dict(teams=t.value, team_size=c.value, block=b.value, gen_ms=g.value)

    def phase_ticks(self):
        out = np.zeros(32, np.uint64)
        _ck(load().xcs_batch_phase_ticks(self._h, _p(out)))
        return out

    def close(self):
        if self._h:
            load().xcs_batch_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def mlp_features(g, m, k):
    """Warm-start features of one instance from g = A^T y (device kernel)."""
    g = np.ascontiguousarray(g, np.float32)
    X = np.zeros((g.size, 8), np.float32)
    _ck(load().xcs_mlp_features(_p(g), g.size, int(m), int(k), _p(X)))
    return X


def gemm_tn(fmt, A, B):
    """C = q(A) q(B)^T on the MFMA GEMM; returns (C (M x N), A_q, B_q)."""
    A = np.ascontiguousarray(A, np.float32)
    B = np.ascontiguousarray(B, np.float32)
    M, K = A.shape
    N = B.shape[0]
    C = np.zeros((N, M), np.float32)
    Aq = np.zeros_like(A)
    Bq = np.zeros_like(B)
    _ck(load().xcs_gemm_tn(fmt.encode(), M, N, K, _p(A), _p(B), _p(C), _p(Aq), _p(Bq)))
    return C.T.copy(), Aq, Bq


class ManyRHS:
    """One gen A shared by `count` signals, CGIHT in lock step (xcs_mrhs_*)."""

    def __init__(self, m, n, k, count, precision="bf16", opts=None):
        from . import _apply_options
        self.m, self.n, self.k, self.count = m, n, k, count
        o = _apply_options("CGIHT", "gen", n, opts)
        h = ctypes.c_void_p()
        _ck(load().xcs_mrhs_create(m, n, k, count, precision.encode(), ctypes.byref(o),
                                   ctypes.byref(h)))
        self._h = h

    def solve(self):
        ms = ctypes.c_float(0)
        it = np.zeros(3, np.int32)
        _ck(load().xcs_mrhs_solve(self._h, ctypes.byref(ms), _p(it)))
        return ms.value, it

    def results(self):
        norms = np.zeros((self.count, 3), np.float32)
        it = np.zeros(self.count, np.int32)
        rr = np.zeros(self.count, np.float64)
        _ck(load().xcs_mrhs_results(self._h, _p(norms), _p(it), _p(rr)))
        return dict(norms=norms, iters=it, resid_rel=rr)

    def x(self, s):
        x = np.empty(self.n, np.float32)  # all filled by the call
        xt = np.empty(self.n, np.float32)
        y = np.empty(self.m, np.float32)
        _ck(load().xcs_mrhs_x(self._h, int(s), _p(x), _p(xt), _p(y)))
        return x, xt, y

    def fp32_solve(self, first, cnt, mode="device"):
        """Signals [first, first + cnt) by the FP32 one-instance-per-launch engine:
        (summed ms, norms (cnt x 3), iterations)."""
        ms = ctypes.c_float(0)
        norms = np.zeros((cnt, 3), np.float32)
        it = np.zeros(cnt, np.int32)
        _ck(load().xcs_mrhs_fp32_solve(self._h, int(first), int(cnt), 1 if mode == "plain" else 0,
                                       ctypes.byref(ms), _p(norms), _p(it)))
        return ms.value, norms, it

    def configure(self, c_bf16=2.0 ** -7, c_fp8=2.0 ** -3, corrections=6, ref_outer=2,
                  ref_inner=4):
        _ck(load().xcs_mrhs_configure(self._h, float(c_bf16), float(c_fp8), int(corrections),
                                      int(ref_outer), int(ref_inner)))

    def gemm_tile(self, tile):
        """GEMM block tile: 0 128 x 128, 1 256 x 128, 2 256 x 256 (True means 1), -1 (the
        default) each product's by its sizes."""
        _ck(load().xcs_mrhs_gemm_tile(self._h, int(tile)))

    def row_blocks(self, keep):
        """keep=False gives back the row-blocked copy of A (4 m n bytes), True makes it
        again; results do not depend on it."""
        _ck(load().xcs_mrhs_row_blocks(self._h, 1 if keep else 0))

    def samples(self, per, seed=1):
        """Training samples of every signal: (X (count*per x 8), labels)."""
        X = np.zeros((self.count * per, 8), np.float32)
        y = np.zeros(self.count * per, np.float32)
        _ck(load().xcs_mrhs_samples(self._h, int(per), int(seed), _p(X), _p(y)))
        return X, y

    def phase_ms(self):
        out = np.zeros(6, np.float32)
        _ck(load().xcs_mrhs_phase_ms(self._h, _p(out)))
        return out

    def gemm_timed(self, transpose, fmt="bf16", reps=20):
        ms = ctypes.c_float(0)
        fl = ctypes.c_double(0)
        _ck(load().xcs_mrhs_gemm_timed(self._h, int(transpose), fmt.encode(), int(reps),
                                       ctypes.byref(ms), ctypes.byref(fl)))
        return ms.value, fl.value

    def close(self):
        if self._h:
            load().xcs_mrhs_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class MLP:
    """The warm-start network (xcs_mlp_*): 8 features -> 512 -> 512 -> 1."""

    def __init__(self, seed=1):
        h = ctypes.c_void_p()
        _ck(load().xcs_mlp_create(int(seed), ctypes.byref(h)))
        self._h = h
        self.nparams = load().xcs_mlp_param_count()

    def params(self):
        out = np.zeros(self.nparams, np.float32)
        _ck(load().xcs_mlp_get_params(self._h, _p(out)))
        return out

    def set_params(self, p):
        p = np.ascontiguousarray(p, np.float32)
        assert p.size == self.nparams
        _ck(load().xcs_mlp_set_params(self._h, _p(p)))

    def grad(self, X, labels, pos_w=1.0):
        X = np.ascontiguousarray(X, np.float32)
        labels = np.ascontiguousarray(labels, np.float32)
        g = np.empty(self.nparams, np.float32)  # filled by the call
        loss = ctypes.c_float(0)
        _ck(load().xcs_mlp_grad(self._h, _p(X), _p(labels), len(labels), float(pos_w), _p(g),
                                ctypes.byref(loss)))
        return g, loss.value

    def scores(self, X):
        X = np.ascontiguousarray(X, np.float32)
        out = np.zeros(X.shape[0], np.float32)
        _ck(load().xcs_mlp_scores(self._h, _p(X), X.shape[0], _p(out)))
        return out

    def set_data(self, X, labels):
        self._X = np.ascontiguousarray(X, np.float32)
        self._y = np.ascontiguousarray(labels, np.float32)
        _ck(load().xcs_mlp_set_data(self._h, _p(self._X), _p(self._y), len(self._y)))

    def train(self, steps, batch=8192, lr=1e-3, pos_w=1.0):
        loss = ctypes.c_float(0)
        ms = ctypes.c_float(0)
        _ck(load().xcs_mlp_train(self._h, int(steps), int(batch), float(lr), float(pos_w),
                                 ctypes.byref(loss), ctypes.byref(ms)))
        return loss.value, ms.value

    def close(self):
        if self._h:
            load().xcs_mlp_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def cs_gen_noalloc(alg, d_y, d_A, lda, m, n, k, opts, d_x, stream=None, report=True):
    """xcs_cs_gen_noalloc: solve a gen problem whose y, A (column-major, leading
    dimension lda) and output x are device pointers (ints), with the library's
    fixed scratch instead of allocations.  Returns (iterations, conv_rate) when
    report is True (the call then waits for the stream), else None."""
    it = ctypes.c_int(0)
    rate = ctypes.c_float(0)
    _ck(load().xcs_cs_gen_noalloc(alg.encode(), ctypes.c_void_p(d_y), ctypes.c_void_p(d_A), lda, m,
                                  n, k, ctypes.byref(opts), ctypes.c_void_p(d_x),
                                  ctypes.byref(it) if report else None,
                                  ctypes.byref(rate) if report else None,
                                  ctypes.c_void_p(stream) if stream else None))
    return (it.value, rate.value) if report else None
