"""libokq.so's own dispatch rules (okq_internal.h), called through their C++
symbols: what a call of given sizes would run.  No GPU is needed."""
import ctypes

from ocelotl_amd import okq


class GemmPlan(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in ("bm", "groups", "kwaves", "ksplit", "wide")] + \
               [(n, ctypes.c_size_t) for n in ("off_lo", "off_sums", "off_rscale", "off_part", "workspace", "reserve")]


def _rule(symbol, restype, *argtypes):
    f = getattr(okq.lib(), symbol)
    f.restype, f.argtypes = restype, argtypes
    return f


def _arr(t, v):
    return (t * len(v))(*v)


def gemm_plan(t, rows, n, k, bf16, cus):
    f = _rule("_ZN3okq9gemm_planEilllbi", GemmPlan, ctypes.c_int, *[ctypes.c_int64] * 3, ctypes.c_bool, ctypes.c_int)
    return f(t, rows, n, k, bf16, cus)


def decode_pairs(t, rows, inter, hidden, cus):
    """Whether a gated MLP's gate and up tiles go in pairs (decode batches)."""
    f = _rule("_ZN3okq17gemm_decode_pairsERKNS_8GemmPlanE", ctypes.c_bool, ctypes.POINTER(GemmPlan))
    return f(ctypes.byref(gemm_plan(t, rows, 2 * ((inter + 15) // 16 * 16), hidden, False, cus)))


def gemv_pairs(t, inter, hidden, cus):
    """Whether one row's gate and up rows go in pairs (16-byte aligned weights)."""
    f = _rule("_ZN3okq10gemv_pairsEilPKvS1_li", ctypes.c_bool, ctypes.c_int, ctypes.c_int64, ctypes.c_void_p,
              ctypes.c_void_p, ctypes.c_int64, ctypes.c_int)
    return f(t, hidden, 4096, 4096, inter, cus)


def gemv_mixes(k, types, ns, cus):
    """Whether one row's Q4_K and Q6_K matrices share a launch (aligned weights)."""
    f = _rule("_ZN3okq10gemv_mixesEliPKiPKPKvPKli", ctypes.c_bool, ctypes.c_int64, ctypes.c_int, *[ctypes.c_void_p] * 3,
              ctypes.c_int)
    return f(k, len(ns), _arr(ctypes.c_int, types), _arr(ctypes.c_void_p, [4096] * len(ns)), _arr(ctypes.c_int64, ns), cus)
