"""The host-side rules that choose a launch or a workspace (no GPU): each at
the sizes where it decides."""
import pytest

import plan_query

CUS = 256
Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14


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
def test_one_row_of_two_formats_shares_a_launch_only_where_it_pays(k, q4, q6, mixes):
    assert plan_query.gemv_mixes(k, [Q4_K] * len(q4) + [Q6_K] * len(q6), q4 + q6, CUS) == mixes


@pytest.mark.parametrize("n,k", [(4096, 14336), (8192, 28672), (28672, 8192), (4096, 4096), (1024, 4096), (96, 256),
                                 (128256, 4096)])
@pytest.mark.parametrize("t,bf16", [(Q4_K, False), (Q8_0, False), (Q6_K, False), (Q6_K, True)])
def test_a_larger_prefill_call_reserves_what_every_smaller_one_needs(t, bf16, n, k):
    """The K split, and with it the partials, rises and falls with the rows
    (Q6_K 14336 -> 4096: 93 MB unsplit at 1568 rows, 197 MB in seven slices at
    1135); what a call reserves only rises, and has a bound."""
    reserved = 0
    for rows in list(range(33, 400)) + list(range(400, 4200, 7)):
        p = plan_query.gemm_plan(t, rows, n, k, bf16, CUS)
        smaller = plan_query.gemm_plan(t, rows, max(1, n - 300), k - 256 if k > 256 else k, bf16, CUS)
        assert p.workspace <= p.reserve and reserved <= p.reserve and smaller.workspace <= p.reserve, rows
        assert p.reserve <= max(64 << 20, p.off_part + (192 << 20)), rows
        reserved = p.reserve
