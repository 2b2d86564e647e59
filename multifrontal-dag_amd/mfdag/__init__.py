"""Python front end of libmfdag (the MI355X numeric phase of a supernodal
multifrontal Cholesky solver).

`Solver` wraps one C-ABI handle (include/mfdag.h); `hppllt` mirrors the
reference's Fortran module API (src/main/hppllt.f90:8-9) on top of it.
The GPU path has no fallback: if libmfdag.so is missing or no gfx950 device
is present, the numeric calls raise.
"""
from __future__ import annotations

import ctypes as C
import os

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(os.path.dirname(HERE), "lib", "libmfdag.so")

MFD_OK = 0
MFD_ERR_ARG = -1
MFD_ERR_STATE = -2
MFD_ERR_NODEVICE = -7
MFD_ERR_UNSUPPORTED = -8
MFD_ERR_SCRATCH = -10
FP64 = 0
FP32_IR = 1
FP16_IR = 2
BF16_IR = 3
FLAG_GRAPH = 1
FLAG_PROFILE = 2
FLAG_ORDER_ND = 4
KERNEL_CLASSES = ["assemble", "extend_add", "small_front", "potrf", "trsm", "update", "schur", "solve_fwd",
                  "solve_bwd", "refine", "front"]

_lib = None


class MfdError(RuntimeError):
    def __init__(self, code, what):
        self.code = code
        msg = lib().mfd_error_string(code).decode() if _lib is not None else str(code)
        super().__init__(f"{what}: {msg} (code {code})")


class NotPositiveDefinite(MfdError):
    pass


class MfdStats(C.Structure):
    _fields_ = [("analyze_ms", C.c_double), ("assemble_ms", C.c_double), ("factor_ms", C.c_double),
                ("solve_ms", C.c_double), ("factor_gflops", C.c_double), ("precision", C.c_int),
                ("refine_iters", C.c_int), ("backward_error", C.c_double), ("refine_residual", C.c_double),
                ("front_bytes", C.c_int64), ("device_bytes", C.c_int64), ("num_levels", C.c_int),
                ("num_launches_factor", C.c_int), ("num_launches_solve", C.c_int)]


def lib():
    """Loads libmfdag.so (raises if it has not been built)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise FileNotFoundError(f"{LIB_PATH} is missing: run multifrontal-dag_amd/build_lib.py")
        L = C.CDLL(LIB_PATH)
        P, i, i64, d = C.c_void_p, C.c_int, C.c_int64, C.c_double
        ip = C.POINTER(C.c_int)
        lp = C.POINTER(C.c_int64)
        dp = C.POINTER(C.c_double)
        sig = {
            "mfd_create": (i, [C.POINTER(P), i, i]),
            "mfd_destroy": (None, [P]),
            "mfd_analyze": (i, [P, i, ip, ip, i, ip]),
            "mfd_analyze_batch": (i, [P, i, ip, C.POINTER(ip), C.POINTER(ip), i, C.POINTER(ip)]),
            "mfd_set_structure": (i, [P, i, ip, ip, ip, ip, lp, ip]),
            "mfd_factorize": (i, [P, dp, i]),
            "mfd_factorize_device": (i, [P, C.c_void_p, i]),
            "mfd_solve": (i, [P, dp, i, i]),
            "mfd_solve_permuted": (i, [P, dp, i, i]),
            "mfd_solve_device": (i, [P, C.c_void_p, i, i]),
            "mfd_solve_device_noalloc": (i, [P, C.c_void_p, i, i]),
            "mfd_get_solve_errors": (i, [P, i, dp, dp, dp]),
            "mfd_export_tiles": (i, [P, dp, dp]),
            "mfd_export_front": (i, [P, i, dp]),
            "mfd_get_cost": (i64, [P]),
            "mfd_get_nonzero": (i64, [P]),
            "mfd_get_array_size": (i64, [P, i]),
            "mfd_get_time_info": (d, [P, i]),
            "mfd_get_dims": (i, [P, ip, ip, lp, lp]),
            "mfd_get_structure": (i, [P, ip, ip, ip, ip, ip, ip, lp, lp]),
            "mfd_get_stats": (i, [P, C.POINTER(MfdStats)]),
            "mfd_get_kernel_time": (i, [P, i, dp, ip]),
            "mfd_get_kernel_work": (i, [P, i, i, dp, dp]),
            "mfd_order_nd": (i, [i, ip, ip, ip]),
            "mfd_tree_pruning": (i, [i, ip, ip, ip, d, i, ip, ip, ip]),
            "mfd_mm_size": (i, [C.c_char_p, ip, lp]),
            "mfd_mm_read": (i, [C.c_char_p, i, i64, ip, ip, dp]),
            "mfd_set_update_period": (i, [P, i]),
            "mfd_get_update_period": (i, [P]),
            "mfd_set_front_split": (i, [P, i]),
            "mfd_set_tile_bound": (i, [P, i]),
            "mfd_set_level_rule": (i, [P, i]),
            "mfd_get_level_rule": (i, [P]),
            "mfd_get_tile_bound": (i, [P]),
            "mfd_set_solve_block": (i, [P, i]),
            "mfd_get_solve_block": (i, [P]),
            "mfd_set_front_kinds": (i, [P, ip]),
            "mfd_set_host_subtrees": (i, [P, ip, i, i]),
            "mfd_factorize_host_subtrees": (i, [P, dp]),
            "mfd_get_host_part": (i, [P, dp, ip, dp]),
            "mfd_get_front_times": (i, [P, dp]),
            "mfd_check_schedule": (i, [P, i, lp, C.c_char_p, i]),
            "mfd_mlp_predict": (i, [i, dp, dp, dp]),
            "mfd_mlp_gradient": (i, [i, dp, dp, dp, dp, dp]),
            "mfd_mlp_train": (i, [i, dp, dp, dp, i, d, dp]),
            "mfd_error_string": (C.c_char_p, [i]),
        }
        for name, (res, args) in sig.items():
            f = getattr(L, name)
            f.restype = res
            f.argtypes = args
        _lib = L
    return _lib


def _ptr(a, ct):
    return a.ctypes.data_as(C.POINTER(ct)) if a is not None else None


def _i32(a):
    return np.ascontiguousarray(np.asarray(a), dtype=np.int32)


def order_nd(ccs_col, ccs_row):
    """Graph nested dissection ordering (new -> old, 1-based) of the pattern
    of a 1-based lower CCS: the library's stand-in for METIS_NodeND."""
    col, row = _i32(ccs_col), _i32(ccs_row)
    n = len(col) - 1
    perm = np.empty(n, np.int32)
    rc = lib().mfd_order_nd(n, _ptr(col, C.c_int), _ptr(row, C.c_int), _ptr(perm, C.c_int))
    if rc != MFD_OK:
        raise MfdError(rc, "mfd_order_nd")
    return perm


def tree_pruning(c, w, parent, tol, p):
    """Subtree partition of an assembly tree (the reference's tree_pruning):
    c, w, parent per node (postordered, 1-based parents, 0 for roots).
    Returns (subtree roots, 1-based, in the reference's list order; the bin
    of each, 0-based)."""
    c, w, pa = _i32(c), _i32(w), _i32(parent)
    m = len(c)
    sub = np.empty(m, np.int32)
    bins = np.empty(m, np.int32)
    cnt = C.c_int()
    rc = lib().mfd_tree_pruning(m, _ptr(c, C.c_int), _ptr(w, C.c_int), _ptr(pa, C.c_int), float(tol), int(p),
                                _ptr(sub, C.c_int), _ptr(bins, C.c_int), C.byref(cnt))
    if rc != MFD_OK:
        raise MfdError(rc, "mfd_tree_pruning")
    return sub[:cnt.value].copy(), bins[:cnt.value].copy()


def read_matrix_market(path):
    """(n, ccs_col, ccs_row, ccs_val) of a MatrixMarket file holding the lower
    triangle of a symmetric matrix: the 1-based lower CCS, diagonal first in
    each column, that Solver.analyze / factorize take (the reference driver's
    reading, example.f90:63-145)."""
    L = lib()
    name = os.fsencode(path)
    n, nnz = C.c_int(), C.c_int64()
    rc = L.mfd_mm_size(name, C.byref(n), C.byref(nnz))
    if rc != MFD_OK:
        raise MfdError(rc, f"mfd_mm_size({path})")
    col = np.empty(n.value + 1, np.int32)
    row = np.empty(nnz.value, np.int32)
    val = np.empty(nnz.value, np.float64)
    rc = L.mfd_mm_read(name, n.value, nnz.value, _ptr(col, C.c_int), _ptr(row, C.c_int), _ptr(val, C.c_double))
    if rc != MFD_OK:
        raise MfdError(rc, f"mfd_mm_read({path})")
    return n.value, col, row, val


MLP_INPUTS, MLP_HIDDEN = 4, 32
MLP_PARAMS = MLP_HIDDEN * (MLP_INPUTS + 2) + 1


def _f64(a):
    return np.ascontiguousarray(np.asarray(a), dtype=np.float64)


def _mlp_check(rc, what):
    if rc != MFD_OK:
        raise MfdError(rc, what)


def mlp_predict(params, x):
    """The cost model's outputs for the rows of x (n x MLP_INPUTS), on the GPU."""
    x, p = _f64(x), _f64(params)
    y = np.empty(len(x))
    _mlp_check(lib().mfd_mlp_predict(len(x), _ptr(x, C.c_double), _ptr(p, C.c_double), _ptr(y, C.c_double)),
               "mfd_mlp_predict")
    return y


def mlp_gradient(params, x, t):
    """(gradient, loss) of the mean squared error at params, on the GPU."""
    x, t, p = _f64(x), _f64(t), _f64(params)
    g = np.empty(MLP_PARAMS)
    loss = C.c_double()
    _mlp_check(lib().mfd_mlp_gradient(len(x), _ptr(x, C.c_double), _ptr(t, C.c_double), _ptr(p, C.c_double),
                                      _ptr(g, C.c_double), C.byref(loss)), "mfd_mlp_gradient")
    return g, loss.value


def mlp_train(params, x, t, epochs, lr):
    """(trained params, loss before the last step): full-batch Adam on the GPU."""
    x, t = _f64(x), _f64(t)
    p = _f64(params).copy()
    loss = C.c_double()
    _mlp_check(lib().mfd_mlp_train(len(x), _ptr(x, C.c_double), _ptr(t, C.c_double), _ptr(p, C.c_double),
                                   int(epochs), float(lr), C.byref(loss)), "mfd_mlp_train")
    return p, loss.value


class Solver:
    """One analysis + factorization + solves (one C-ABI handle).

    nb is the reference's tile size, used only for the reference-layout
    views (export_tiles, array_size).  With host_only=True the handle may be
    created on a machine without a GPU (analysis and structure queries work;
    numeric calls raise)."""

    def __init__(self, nb=64, graph=False, profile=False, host_only=False, order_nd=False):
        L = lib()
        h = C.c_void_p()
        flags = (FLAG_GRAPH if graph else 0) | (FLAG_PROFILE if profile else 0) | (FLAG_ORDER_ND if order_nd else 0)
        rc = L.mfd_create(C.byref(h), int(nb), flags)
        self.h = h
        self.nb = int(nb)
        self.device = rc == MFD_OK
        if rc not in (MFD_OK, MFD_ERR_NODEVICE) or (rc == MFD_ERR_NODEVICE and not host_only):
            L.mfd_destroy(h)
            self.h = None
            raise MfdError(rc, "mfd_create")

    def close(self):
        if getattr(self, "h", None):
            lib().mfd_destroy(self.h)
            self.h = None

    __del__ = close

    def _check(self, rc, what):
        if rc > 0:
            raise NotPositiveDefinite(rc, what)
        if rc < 0:
            raise MfdError(rc, what)
        return rc

    @property
    def update_period(self):
        """In-panel update period of the large fronts (64-column steps)."""
        return lib().mfd_get_update_period(self.h)

    @update_period.setter
    def update_period(self, period):
        self._check(lib().mfd_set_update_period(self.h, int(period)), "mfd_set_update_period")

    @property
    def tile_bound(self):
        """Update rows from which a front's Schur tiles are 128 x 128 (0: never)."""
        return lib().mfd_get_tile_bound(self.h)

    @tile_bound.setter
    def tile_bound(self, min_rows):
        self._check(lib().mfd_set_tile_bound(self.h, int(min_rows)), "mfd_set_tile_bound")

    @property
    def level_rule(self):
        """1: each front one level below its parent (default); 0: one above
        its highest child."""
        return lib().mfd_get_level_rule(self.h)

    @level_rule.setter
    def level_rule(self, rule):
        self._check(lib().mfd_set_level_rule(self.h, int(rule)), "mfd_set_level_rule")

    @property
    def solve_block(self):
        """Pivot columns from which a front's forward solve steps over
        256-column superblocks (0: 64-column blocks only)."""
        return lib().mfd_get_solve_block(self.h)

    @solve_block.setter
    def solve_block(self, min_c):
        self._check(lib().mfd_set_solve_block(self.h, int(min_c)), "mfd_set_solve_block")

    def set_host_subtrees(self, roots, threads=4):
        """CPU+GPU hybrid: the subtrees rooted at roots (0-based node ids)
        are factored on the host by `threads` threads (FP64 only)."""
        r = _i32(roots)
        self._check(lib().mfd_set_host_subtrees(self.h, _ptr(r, C.c_int) if len(r) else None, len(r), int(threads)),
                    "mfd_set_host_subtrees")

    def factorize_host_subtrees(self, a):
        """The host part alone (no GPU needed): returns 0 or the failing column."""
        a = np.ascontiguousarray(a, dtype=np.float64)
        rc = lib().mfd_factorize_host_subtrees(self.h, _ptr(a, C.c_double))
        if rc < 0:
            raise MfdError(rc, "mfd_factorize_host_subtrees")
        return rc

    def host_part(self):
        """(ms, fronts, flops) of the last host part."""
        ms, fr, fl = C.c_double(), C.c_int(), C.c_double()
        self._check(lib().mfd_get_host_part(self.h, C.byref(ms), C.byref(fr), C.byref(fl)), "mfd_get_host_part")
        return ms.value, fr.value, fl.value

    def set_front_split(self, cmax):
        """Fronts of order > 64 with at most cmax pivot columns are factored
        whole by one workgroup each (0: none)."""
        self._check(lib().mfd_set_front_split(self.h, int(cmax)), "mfd_set_front_split")

    def set_front_kinds(self, kinds):
        """Per node (0-based order): 1 one workgroup, 0 64-column steps, -1 by
        the split (and, if that takes none of them, the launch for the bottom
        of the tree, fronts of order <= 128); None clears."""
        if kinds is None:
            self._check(lib().mfd_set_front_kinds(self.h, None), "mfd_set_front_kinds")
            return
        k = _i32(kinds)
        self._check(lib().mfd_set_front_kinds(self.h, _ptr(k, C.c_int)), "mfd_set_front_kinds")

    def check_schedule(self, variant=0):
        """Static check of the factorization schedule: (number of unordered
        conflicting task pairs, report of the first few)."""
        n = C.c_int64()
        buf = C.create_string_buffer(4096)
        self._check(lib().mfd_check_schedule(self.h, int(variant), C.byref(n), buf, len(buf)), "mfd_check_schedule")
        return n.value, buf.value.decode()

    def front_times(self):
        """Per node: microseconds of its workgroup in the last factorization
        (medium fronts; -1 for the others)."""
        out = np.empty(self.num_node, dtype=np.float64)
        self._check(lib().mfd_get_front_times(self.h, _ptr(out, C.c_double)), "mfd_get_front_times")
        return out

    # -------------------------------------------------------------- analysis
    def analyze(self, ccs_col, ccs_row, max_zero=0, perm=None):
        """1-based lower CCS (diagonal first); perm: new -> old, 1-based."""
        ccs_col = _i32(ccs_col)
        ccs_row = _i32(ccs_row)
        n = len(ccs_col) - 1
        p = _i32(perm) if perm is not None else None
        self._check(lib().mfd_analyze(self.h, n, _ptr(ccs_col, C.c_int), _ptr(ccs_row, C.c_int), int(max_zero),
                                      _ptr(p, C.c_int)), "mfd_analyze")
        self._dims()

    def analyze_batch(self, systems, max_zero=0, perms=None):
        """The batching form: systems = [(ccs_col, ccs_row), ...] (each like
        analyze's), perms = None or a list with one perm (or None) per system.
        Afterwards the solver holds the block-diagonal system: values and
        right-hand sides are the systems' concatenated
        (problems.batch_problem builds that system for checks)."""
        k = len(systems)
        cols = [_i32(c) for c, _ in systems]
        rows = [_i32(r) for _, r in systems]
        ns = np.array([len(c) - 1 for c in cols], np.int32)
        ip = C.POINTER(C.c_int)
        col_arr = (ip * k)(*[_ptr(c, C.c_int) for c in cols])
        row_arr = (ip * k)(*[_ptr(r, C.c_int) for r in rows])
        perm_arr = None
        keep = []
        if perms is not None:
            ps = [_i32(p) if p is not None else None for p in perms]
            keep = ps
            perm_arr = (ip * k)(*[_ptr(p, C.c_int) if p is not None else ip() for p in ps])
        self._check(lib().mfd_analyze_batch(self.h, k, _ptr(ns, C.c_int), col_arr, row_arr, int(max_zero), perm_arr),
                    "mfd_analyze_batch")
        del keep
        self._dims()

    def set_structure(self, supernode_size, work_size, parent, local_index, a_colptr, supernodal_index):
        c, w, pa = _i32(supernode_size), _i32(work_size), _i32(parent)
        li = _i32(local_index) if len(local_index) else np.zeros(1, np.int32)
        cp = np.ascontiguousarray(a_colptr, dtype=np.int64)
        sx = _i32(supernodal_index)
        self._check(lib().mfd_set_structure(self.h, len(c), _ptr(c, C.c_int), _ptr(w, C.c_int), _ptr(pa, C.c_int),
                                            _ptr(li, C.c_int), _ptr(cp, C.c_int64), _ptr(sx, C.c_int)),
                    "mfd_set_structure")
        self._dims()

    def _dims(self):
        n, m = C.c_int(), C.c_int()
        nnz, nl = C.c_int64(), C.c_int64()
        self._check(lib().mfd_get_dims(self.h, C.byref(n), C.byref(m), C.byref(nnz), C.byref(nl)), "mfd_get_dims")
        self.n, self.num_node, self.nnz, self.nlidx = n.value, m.value, nnz.value, nl.value

    def structure(self):
        m, n, nnz, nl = self.num_node, self.n, self.nnz, self.nlidx
        out = dict(supernode_size=np.zeros(m, np.int32), work_size=np.zeros(m, np.int32),
                   parent=np.zeros(m, np.int32), perm=np.zeros(n, np.int32),
                   local_index=np.zeros(max(nl, 1), np.int32), supernodal_index=np.zeros(max(nnz, 1), np.int32),
                   ccs_perm=np.zeros(max(nnz, 1), np.int64), a_colptr=np.zeros(n + 1, np.int64))
        self._check(lib().mfd_get_structure(
            self.h, *[_ptr(out[k], C.c_int) for k in ("supernode_size", "work_size", "parent", "perm",
                                                       "local_index", "supernodal_index")],
            _ptr(out["ccs_perm"], C.c_int64), _ptr(out["a_colptr"], C.c_int64)), "mfd_get_structure")
        out["local_index"] = out["local_index"][:nl]
        out["supernodal_index"] = out["supernodal_index"][:nnz]
        out["ccs_perm"] = out["ccs_perm"][:nnz]
        return out

    def cost(self):
        return lib().mfd_get_cost(self.h)

    def nonzero(self):
        return lib().mfd_get_nonzero(self.h)

    def array_size(self, which):
        return lib().mfd_get_array_size(self.h, int(which))

    # -------------------------------------------------------------- numeric
    def factorize(self, a, precision=FP64):
        a = np.ascontiguousarray(a, dtype=np.float64)
        if a.size != self.nnz:
            raise ValueError(f"expected {self.nnz} values, got {a.size}")
        return self._check(lib().mfd_factorize(self.h, _ptr(a, C.c_double), int(precision)), "mfd_factorize")

    def factorize_device(self, d_a_ptr, precision=FP64):
        return self._check(lib().mfd_factorize_device(self.h, C.c_void_p(d_a_ptr), int(precision)),
                           "mfd_factorize_device")

    def solve(self, b, permuted=False):
        """b: (n,) or (n, nrhs); returns x (a new array)."""
        x = np.array(b, dtype=np.float64, order="F", copy=True)
        one = x.ndim == 1
        if one:
            x = x.reshape(-1, 1, order="F")
        f = lib().mfd_solve_permuted if permuted else lib().mfd_solve
        self._check(f(self.h, _ptr(x, C.c_double), x.shape[1], x.shape[0]), "mfd_solve")
        return x[:, 0] if one else x

    def solve_device(self, d_b_ptr, nrhs, ldb):
        return self._check(lib().mfd_solve_device(self.h, C.c_void_p(d_b_ptr), int(nrhs), int(ldb)),
                           "mfd_solve_device")

    def solve_device_noalloc(self, d_b_ptr, nrhs, ldb):
        """mfd_solve_device with the solve buffers in the library's fixed
        device scratch (no allocation); returns the C return code."""
        return lib().mfd_solve_device_noalloc(self.h, C.c_void_p(d_b_ptr), int(nrhs), int(ldb))

    def solve_errors(self, nrhs=1, forward=True):
        """Errors of the last solve per right-hand side, computed on the GPU in
        FP64: dict of arrays eta (normwise backward error), res2 (the
        reference driver's ||b - Ax||_2/||x||_2) and, with forward=True, ferr
        (forward error estimate from one more solve with the current factor)."""
        eta, res2 = np.zeros(nrhs), np.zeros(nrhs)
        ferr = np.zeros(nrhs) if forward else None
        self._check(lib().mfd_get_solve_errors(self.h, int(nrhs), _ptr(eta, C.c_double), _ptr(res2, C.c_double),
                                               _ptr(ferr, C.c_double)), "mfd_get_solve_errors")
        out = dict(eta=eta, res2=res2)
        if forward:
            out["ferr"] = ferr
        return out

    def export_tiles(self):
        sn = np.zeros(max(self.array_size(1), 1))
        wk = np.zeros(max(self.array_size(2), 1))
        self._check(lib().mfd_export_tiles(self.h, _ptr(sn, C.c_double), _ptr(wk, C.c_double)), "mfd_export_tiles")
        return sn[: self.array_size(1)], wk[: self.array_size(2)]

    def front(self, node):
        st = self.structure()
        n = int(st["supernode_size"][node - 1] + st["work_size"][node - 1])
        out = np.zeros(n * n)
        self._check(lib().mfd_export_front(self.h, int(node), _ptr(out, C.c_double)), "mfd_export_front")
        return out.reshape(n, n, order="F")

    def stats(self):
        s = MfdStats()
        self._check(lib().mfd_get_stats(self.h, C.byref(s)), "mfd_get_stats")
        return {k: getattr(s, k) for k, _ in MfdStats._fields_}

    def kernel_times(self):
        out = {}
        for k, name in enumerate(KERNEL_CLASSES):
            ms, cnt = C.c_double(), C.c_int()
            lib().mfd_get_kernel_time(self.h, k, C.byref(ms), C.byref(cnt))
            out[name] = (ms.value, cnt.value)
        return out

    def kernel_work(self, elem_bytes=8):
        """Algorithmic (flops, bytes) per kernel class for one factorization /
        one single-RHS solve."""
        out = {}
        for k, name in enumerate(KERNEL_CLASSES):
            f, b = C.c_double(), C.c_double()
            self._check(lib().mfd_get_kernel_work(self.h, k, int(elem_bytes), C.byref(f), C.byref(b)),
                        "mfd_get_kernel_work")
            out[name] = (f.value, b.value)
        return out

    def time_info(self, i):
        return lib().mfd_get_time_info(self.h, int(i))
