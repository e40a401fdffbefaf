"""The host-side rules that choose a kernel, a launch or a workspace, called in
libokq.so directly (no GPU): each at the sizes where it decides."""
import ctypes

import pytest

CUS = 256
Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14


@pytest.fixture(scope="module")
def lib():
    from ocelotl_amd import okq
    return okq.lib()


def _arr(t, v):
    return (t * len(v))(*v)


@pytest.mark.parametrize("k,q4,q6,mixes", [
    (4096, [4096, 1024], [1024], True),     # q, k and v of one layer
    (2048, [2048, 512], [512], True),
    (8192, [8192, 1024], [1024], True),
    (5120, [5120], [5120], True),
    (4096, [1024], [128256], False),        # many steps: each format's own launch is faster
    (2048, [32768], [2048], False),
    (1024, [28672], [1024], False),
    (5120, [32768], [1024], False),
    (14336, [1024], [32768], False),
    (4096, [4096], [], False),              # one format
    (20480, [1024], [1024], False),         # K past the streaming kernel
])
def test_one_row_of_two_formats_shares_a_launch_only_where_it_pays(lib, k, q4, q6, mixes):
    rule = getattr(lib, "_ZN3okq10gemv_mixesEliPKiPKPKvPKli")
    rule.restype = ctypes.c_bool
    rule.argtypes = [ctypes.c_int64, ctypes.c_int] + [ctypes.c_void_p] * 3 + [ctypes.c_int]
    n = q4 + q6
    got = rule(k, len(n), _arr(ctypes.c_int, [Q4_K] * len(q4) + [Q6_K] * len(q6)),
               _arr(ctypes.c_void_p, [4096] * len(n)), _arr(ctypes.c_int64, n), CUS)
    assert got == mixes


class Plan(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in ("bm", "groups", "kwaves", "ksplit", "wide")] + \
               [(n, ctypes.c_size_t) for n in ("off_lo", "off_sums", "off_rscale", "off_part", "workspace", "reserve")]


@pytest.mark.parametrize("n,k", [(4096, 14336), (8192, 28672), (28672, 8192), (4096, 4096), (1024, 4096), (96, 256),
                                 (128256, 4096)])
@pytest.mark.parametrize("t,bf16", [(Q4_K, False), (Q8_0, False), (Q6_K, False), (Q6_K, True)])
def test_a_larger_prefill_call_reserves_what_every_smaller_one_needs(lib, t, bf16, n, k):
    """The K split, and with it the partials, rises and falls with the rows
    (Q6_K 14336 -> 4096: 89 MB at 1568 rows, 197 MB of partials and planes
    at 1135 before the partials had a bound); what a call reserves does not."""
    plan = getattr(lib, "_ZN3okq9gemm_planEilllbi")
    plan.restype = Plan
    plan.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.c_bool, ctypes.c_int]
    reserved = 0
    for rows in list(range(33, 400)) + list(range(400, 4200, 7)):
        p = plan(t, rows, n, k, bf16, CUS)
        smaller = plan(t, rows, max(1, n - 300), k - 256 if k > 256 else k, bf16, CUS)
        assert p.workspace <= p.reserve and reserved <= p.reserve and smaller.workspace <= p.reserve, rows
        assert p.reserve <= max(64 << 20, p.off_part + (192 << 20)), rows
        reserved = p.reserve
