"""GPU parity of prefill with f32 activations (more than 32 rows, every linear
format) and of several matrices sharing one call (needs an MI355X).

Bars: outputs against float64 on the oracle's dequantised weights; the shared
calls bit for bit against each matrix's own call.
"""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

TYPES = [O.Q4_K, O.Q5_K, O.Q6_K, O.Q8_0]


@pytest.fixture(scope="module")
def torch():
    import torch as _t
    if not _t.cuda.is_available():
        pytest.skip("no GPU")
    return _t


@pytest.fixture(scope="module")
def okq(torch):
    from ocelotl_amd import okq as _okq
    _okq.call("okq_init", 0)
    return _okq


@pytest.fixture(scope="module")
def orc():
    return O.Oracle()


def _dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _linear(torch, okq, t, xd, rows, k, wd, n, bd=None, entry="okq_linear_out_by_in_q", stream=None):
    out = torch.full((rows * n,), float("nan"), dtype=torch.float32, device="cuda")
    okq.call(entry, xd.data_ptr(), rows, k, t, wd.data_ptr(), wd.numel(), n, None if bd is None else bd.data_ptr(),
             out.data_ptr(), torch.cuda.current_stream().cuda_stream if stream is None else stream)
    return out


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("rows,k,n", [
    (33, 256, 40),      # one super-block, the 64-row tile mostly padding
    (64, 768, 255),     # a full 64-row tile, an odd number of super-blocks
    (65, 2304, 257),    # 96-row tiles, two column tiles, split K
    (96, 512, 260),     # a full 96-row tile
    (97, 512, 512), (128, 4096, 300), (129, 1280, 96), (333, 1024, 520),
    (300, 8192, 4096),  # unsplit or long slices: Q8_0's sums wait in the output or the partials
    (1100, 7424, 4100),
])
def test_f32_prefill_matches_float64(torch, okq, orc, t, rows, k, n):
    """Every product is exact but for the activations' hi + lo planes (2^-22)
    and, in Q6_K, the dropped lo * remainder (2^-22); f32 sums of up to 3 K / 16
    MFMA accumulations round at random: 2^-20 of sum |x| max |w| bounds them
    with room (one wrong product of K would be 1 / K)."""
    print(f"[gpu] f32 prefill type={t} rows={rows} K={k} N={n}", flush=True)
    wq = orc.quantize(t, orc.normal(9000 + t + k, n * k, 0.02))
    x = orc.normal(9001 + rows, rows * k, 1.0).reshape(rows, k)
    x[:, :3] *= 100.0
    x[rows // 2] *= np.float32(2.0 ** 30)
    bias = orc.normal(9002, n, 0.1)
    xd, wd, bd = _dev(torch, x), _dev(torch, wq), _dev(torch, bias)
    out = _linear(torch, okq, t, xd, rows, k, wd, n, bd)
    torch.cuda.synchronize()
    w = _dev(torch, orc.dequantize(t, wq, n * k)).view(n, k).double()
    want = xd.double() @ w.t() + bd.double()
    bound = 2.0 ** -20 * xd.double().abs().sum(1, keepdim=True) * 2 * w.abs().amax(1) + 2.0 ** -22 * want.abs()
    err = (out.view(rows, n).double() - want).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("rows,k,n", [(33, 256, 40), (64, 768, 255), (65, 2304, 257), (97, 512, 520), (128, 4096, 300),
                                      (333, 1024, 512)])
def test_bf16_q6k_prefill_on_small_grids_matches_float64(torch, okq, orc, rows, k, n):
    """bf16 activations through Q6_K grids that do not fill the 8-wave tiles:
    the one-plane form.  Every product is exact; the sums of at most 2 K / 16
    accumulations are bounded as above."""
    print(f"[gpu] bf16 Q6_K prefill rows={rows} K={k} N={n}", flush=True)
    wq = orc.quantize(O.Q6_K, orc.normal(9300 + k, n * k, 0.02))
    x = _dev(torch, orc.normal(9301 + rows, rows * k, 1.0)).view(rows, k).to(torch.bfloat16)
    x[:, :3] *= 100.0
    wd, bd = _dev(torch, wq), _dev(torch, orc.normal(9302, n, 0.1))
    out = _linear(torch, okq, O.Q6_K, x, rows, k, wd, n, bd, entry="okq_linear_out_by_in_q_bf16")
    torch.cuda.synchronize()
    w = _dev(torch, orc.dequantize(O.Q6_K, wq, n * k)).view(n, k).double()
    want = x.double() @ w.t() + bd.double()
    bound = 2.0 ** -20 * x.double().abs().sum(1, keepdim=True) * 2 * w.abs().amax(1) + 2.0 ** -22 * want.abs()
    err = (out.view(rows, n).double() - want).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("t", [O.Q4_K, O.Q5_K])
def test_bf16_prefill_on_weights_near_4_gib_matches_float64(torch, okq, orc, t):
    """bf16 activations through Q4_K and Q5_K tensors too close to 4 GiB for the
    kernels that address a padded column tile: the one-plane form, at its three
    tile heights, the last column tile and rows ragged.  The tensor repeats
    4093 rows, so that no tile sees the same columns twice; bounds as above."""
    k, base = 7168, 4093
    row = k // 256 * O.BLOCK_BYTES[t]
    n = ((1 << 32) - 1025) // row - 141
    wq = orc.quantize(t, orc.normal(9400 + t, base * k, 0.02))
    w = _dev(torch, orc.dequantize(t, wq, base * k)).view(base, k).double()
    wd = _dev(torch, wq).view(base, row).repeat((n + base - 1) // base, 1)[:n].contiguous().view(-1)
    for rows in (33, 70, 127):
        print(f"[gpu] bf16 prefill near 4 GiB type={t} rows={rows} K={k} N={n}", flush=True)
        x = _dev(torch, orc.normal(9401 + rows, rows * k, 1.0)).view(rows, k).to(torch.bfloat16)
        out = _linear(torch, okq, t, x, rows, k, wd, n, entry="okq_linear_out_by_in_q_bf16").view(rows, n)
        torch.cuda.synchronize()
        want = x.double() @ w.t()
        bound = 2.0 ** -20 * x.double().abs().sum(1, keepdim=True) * 2 * w.abs().amax(1) + 2.0 ** -22 * want.abs()
        for c in range(0, n, base):
            m = min(base, n - c)
            err = (out[:, c:c + m].double() - want[:, :m]).abs()
            assert bool((err <= bound[:, :m]).all()), (c, float((err / bound[:, :m]).max()))


@pytest.mark.parametrize("types,rows,k,ns", [
    ([O.Q4_K, O.Q4_K, O.Q6_K], 70, 4096, [1024, 256, 256]),
    ([O.Q8_0, O.Q8_0, O.Q8_0], 333, 2048, [2048, 512, 300]),
    ([O.Q5_K, O.Q6_K, O.Q5_K, O.Q8_0], 40, 768, [33, 300, 512, 17]),
])
def test_f32_prefill_matrices_share_a_call_bit_for_bit(torch, okq, orc, types, rows, k, ns):
    """okq_linear_multi_q above 32 rows: one pre-pass, one launch per format,
    one reduction; every output is its own call's, also in rows with an
    infinity or a NaN."""
    print(f"[gpu] f32 prefill shared types={types} rows={rows} K={k} N={ns}", flush=True)
    x = orc.normal(9100 + rows, rows * k, 1.0).reshape(rows, k)
    x[3, 5], x[rows - 1, 7], x[rows - 1, 9] = np.inf, np.nan, -np.inf
    xd = _dev(torch, x)
    wds = [_dev(torch, orc.quantize(t, orc.normal(9110 + i, n * k, 0.02))) for i, (t, n) in enumerate(zip(types, ns))]
    bds = [_dev(torch, orc.normal(9120 + i, n, 0.1)) if i != 1 else None for i, n in enumerate(ns)]
    outs = [torch.full((rows * n,), 7.0, dtype=torch.float32, device="cuda") for n in ns]
    arr = lambda ty, vals: (ty * len(ns))(*vals)
    args = (xd.data_ptr(), rows, k, len(ns), arr(ctypes.c_uint32, types), arr(ctypes.c_void_p, [w.data_ptr() for w in wds]),
            arr(ctypes.c_uint64, [w.numel() for w in wds]), arr(ctypes.c_int64, ns),
            arr(ctypes.c_void_p, [None if b is None else b.data_ptr() for b in bds]),
            arr(ctypes.c_void_p, [o.data_ptr() for o in outs]))
    okq.call("okq_linear_multi_q", *args, torch.cuda.current_stream().cuda_stream)
    single = [_linear(torch, okq, t, xd, rows, k, w, n, b) for t, w, n, b in zip(types, wds, ns, bds)]
    torch.cuda.synchronize()
    for o, s in zip(outs, single):
        a, b = o.cpu().numpy(), s.cpu().numpy()
        assert ((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))).all()
        assert np.isnan(a.reshape(rows, -1)[rows - 1]).all() and not np.isfinite(a.reshape(rows, -1)[3]).any()
    # under capture on a stream that has only served single calls: the same bits
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for t, w, n, b in zip(types, wds, ns, bds):
            _linear(torch, okq, t, xd, rows, k, w, n, b, stream=side.cuda_stream)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        okq.call("okq_linear_multi_q", *args, side.cuda_stream)
    for _ in range(3):
        for o in outs:
            o.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        for o, s in zip(outs, single):
            a, b = o.cpu().numpy(), s.cpu().numpy()
            assert ((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))).all()


def test_f32_prefill_near_the_static_scratch(torch, okq, orc):
    """2800 rows of 4096: the two planes take 46 of the 64 MiB of the
    allocation-free entry point, so the K split that would fill the CUs is cut
    to fit; both entry points take the same split."""
    t, rows, k, n = O.Q4_K, 2800, 4096, 512
    print(f"[gpu] f32 prefill scratch rows={rows} K={k} N={n}", flush=True)
    wd = _dev(torch, orc.quantize(t, orc.normal(9200, n * k, 0.02)))
    xd = torch.randn(rows * k, generator=torch.Generator().manual_seed(9201)).cuda()
    a = _linear(torch, okq, t, xd, rows, k, wd, n, entry="okq_linear_out_by_in_q_noalloc")
    b = _linear(torch, okq, t, xd, rows, k, wd, n)
    torch.cuda.synchronize()
    assert (a.cpu().numpy().view(np.uint32) == b.cpu().numpy().view(np.uint32)).all()


@pytest.mark.parametrize("t,rows,hidden,ns", [
    (O.Q4_K, 40, 256, [64, 17]),           # the last thread's chunks past the row
    (O.Q8_0, 333, 4096, [512, 128, 128]),
    (O.Q6_K, 34, 8192, [96]),              # four chunks per thread
    (O.Q5_K, 33, 16384, [40, 8]),          # eight
    (O.Q4_K, 33, 16640, [40]),             # longer rows: normalised by a pass of its own
])
def test_rmsnorm_in_the_prepass_matches_float64(torch, okq, orc, t, rows, hidden, ns):
    """okq_rmsnorm_linear_q_multi above 32 rows.  The normalised row carries a
    relative error of fewer than 2^-18 (a tree of under 40 roundings in the
    sum, a square root, a division, two products), the linear the bound of
    test_f32_prefill_matches_float64.  A row with an infinity is NaN
    throughout (inf * (1 / inf))."""
    print(f"[gpu] rms prepass type={t} rows={rows} hidden={hidden} N={ns}", flush=True)
    x = orc.normal(9400 + hidden, rows * hidden, 1.5).reshape(rows, hidden)
    x[1, 3] = np.inf
    g = orc.normal(9401 + hidden, hidden, 1.0)
    xd, gd = _dev(torch, x), _dev(torch, g)
    wds = [_dev(torch, orc.quantize(t, orc.normal(9410 + i, n * hidden, 0.02))) for i, n in enumerate(ns)]
    outs = [torch.full((rows * n,), 7.0, device="cuda") for n in ns]
    arr = lambda ty, vals: (ty * len(ns))(*vals)
    okq.call("okq_rmsnorm_linear_q_multi", xd.data_ptr(), rows, hidden, gd.data_ptr(), 1e-6, t, len(ns),
             arr(ctypes.c_void_p, [w.data_ptr() for w in wds]), arr(ctypes.c_uint64, [w.numel() for w in wds]),
             arr(ctypes.c_int64, ns), None, arr(ctypes.c_void_p, [o.data_ptr() for o in outs]),
             torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    x64 = xd.double()
    xn = x64 / torch.sqrt((x64 * x64).mean(1, keepdim=True) + float(np.float32(1e-6))) * gd.double()
    keep = torch.arange(rows, device="cuda") != 1
    for n, w, o in zip(ns, wds, outs):
        got = o.view(rows, n).double()
        wm = _dev(torch, orc.dequantize(t, w.cpu().numpy(), n * hidden)).view(n, hidden).double()
        want = xn[keep] @ wm.t()
        mag = xn[keep].abs().sum(1, keepdim=True) * wm.abs().amax(1)
        assert bool(((got[keep] - want).abs() <= (2.0 ** -19 + 2.0 ** -18) * mag).all())
        assert bool(torch.isnan(got[1]).all())


@pytest.mark.parametrize("t,td,rows,hidden,inter", [
    (O.Q4_K, O.Q6_K, 40, 1024, 2816), (O.Q8_0, O.Q4_K, 130, 512, 8192), (O.Q6_K, O.Q8_0, 33, 768, 16640),
])
def test_swiglu_in_the_prepass_leaves_its_rows(torch, okq, orc, t, td, rows, hidden, inter):
    """okq_mlp_gated_silu_q above 32 rows: gate_buf holds silu(g) * u of the
    grouped projections (up to the rounding of exp), up_buf their u bit for
    bit, and out is okq_linear_out_by_in_q on gate_buf bit for bit -- also in a
    row with an infinity, and captured on a stream without workspaces of this
    size but those of the single calls."""
    print(f"[gpu] swiglu prepass types={t},{td} rows={rows} hidden={hidden} inter={inter}", flush=True)
    x = orc.normal(9500 + rows, rows * hidden, 1.0).reshape(rows, hidden)
    x[2, 1] = -np.inf
    xd = _dev(torch, x)
    gd, ud, dd = (_dev(torch, orc.quantize(ty, orc.normal(9501 + i, n * k, 0.02)))
                  for i, (ty, n, k) in enumerate([(t, inter, hidden), (t, inter, hidden), (td, hidden, inter)]))
    gb, ub, out = (torch.full((rows * n,), 7.0, device="cuda") for n in (inter, inter, hidden))
    s = torch.cuda.current_stream().cuda_stream
    args = (xd.data_ptr(), rows, hidden, inter, t, gd.data_ptr(), gd.numel(), t, ud.data_ptr(), ud.numel(), td,
            dd.data_ptr(), dd.numel(), gb.data_ptr(), ub.data_ptr(), out.data_ptr())
    okq.call("okq_mlp_gated_silu_q", *args, s)
    g = _linear(torch, okq, t, xd, rows, hidden, gd, inter).cpu().numpy()
    u = _linear(torch, okq, t, xd, rows, hidden, ud, inter).cpu().numpy()
    down = _linear(torch, okq, td, gb, rows, inter, dd, hidden)
    torch.cuda.synchronize()
    same = lambda a, b: ((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))).all()
    h, got = gb.cpu().numpy(), out.cpu().numpy()
    assert same(ub.cpu().numpy(), u) and same(got, down.cpu().numpy())
    with np.errstate(all="ignore"):
        want = (g * (np.float32(1.0) / (np.float32(1.0) + np.exp(-g)))) * u
        fine = np.isfinite(want)
        assert np.all(np.abs(h[fine] - want[fine]) <= 8 * np.spacing(np.abs(want[fine])))
    assert (np.isfinite(h) == fine).all()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    _linear(torch, okq, t, xd, rows, hidden, gd, inter, stream=side.cuda_stream)
    _linear(torch, okq, td, gb, rows, inter, dd, hidden, stream=side.cuda_stream)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        okq.call("okq_mlp_gated_silu_q", *args, side.cuda_stream)
    for _ in range(3):
        gb.fill_(7.0)
        out.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert same(gb.cpu().numpy(), h) and same(out.cpu().numpy(), got)
