"""mm_t's one-launch GEMM for fp32 activations on the 4-wavefront tiles (32x128, 64x128, 64x64, split and
unsplit; x streamed through fp32 LDS stages, rows rescaled as they leave fp16's range, each K slice by
itself) against the two-launch sequence (rowscale cast, GEMM on the same plan) and fp64: ragged M, N
and K, one to a few K steps, fp32 and fp16 outputs, rows past fp16's range early, late and several
times, infinities and NaN; repeat calls bitwise equal and the split counters left zero."""
from __future__ import annotations

import pytest
import torch

import oracle
from _inputs import outlier_rows, randn
from _plan import tile as planned_tile

pytestmark = pytest.mark.gpu

# (M, K, N, tile on 256 CUs, planned split): every tile of the route, ragged edges, 1 to 8 slices
ROUTES = [
    (64, 1024, 1024, (32, 128), 4),
    (33, 3072, 768, (32, 128), 8),
    (24, 5000, 1000, (32, 128), 8),      # ragged M, N, K; a last slice shorter than the others
    (100, 1000, 264, (32, 128), 3),
    (9, 14336, 512, (32, 128), 8),
    (20, 1288, 32768, (32, 128), 1),     # unsplit past the resident route's K
    (64, 1024, 11008, (64, 128), 2),
    (48, 2056, 14336, (64, 128), 2),
    (900, 1000, 1096, (64, 128), 1),
    (128, 6144, 8192, (64, 128), 2),
    (1024, 264, 1024, (64, 64), 1),
    (513, 8, 512, (64, 64), 1),          # one K step of 8
    (72, 3072, 264, (64, 64), 8),
    (160, 11008, 1536, (64, 64), 3),
]
KINDS = ["within", "outliers", "special", "late"]


def _x(M, K, kind, out16):
    x = randn((M, K), seed=M + K)
    if kind == "outliers":
        x = outlier_rows(x, 0.1, 2e3, 8e3 if out16 else 2e5, seed=3)
    elif kind == "special":
        for r, k, v in ((0, K - 1, "inf"), (M // 2, 0, "-inf"), (M - 2, K // 2, "nan"), (M - 1, K - 1, "nan")):
            x[r, k] = float(v)
        x[1, 0] = 5e3 if out16 else 3e5
    elif kind == "late" and not out16:
        x[3, K - 1] = 70000.0
        x[M - 1, K - 1] = -3e6
        for i, k in enumerate(range(0, K, 64)):
            x[5, k] = 7e4 * 3.0 ** min(i, 20)
    return x


def _two(lib, x, w, b, out16, cus):
    M, K = x.shape
    N = w.shape[1]
    dev = x.device
    st = torch.cuda.current_stream(dev).cuda_stream
    y = torch.empty(M, K, dtype=torch.float16, device=dev)
    s = torch.empty(M, device=dev)
    out = torch.empty(M, N, dtype=torch.float16 if out16 else torch.float32, device=dev)
    assert lib.g16_rowscale_f32(x.data_ptr(), y.data_ptr(), s.data_ptr(), M, K, 1024.0, st) == 0
    ks = lib.g16_hgemm_plan(M, N, K, cus)
    ws = torch.empty(max(16, lib.g16_hgemm_splitk_workspace_bytes(M, N, K, ks, cus)), dtype=torch.uint8, device=dev)
    cnt = torch.zeros(max(16, lib.g16_hgemm_splitk_counter_bytes(M, N, K, ks, cus)), dtype=torch.uint8, device=dev)
    assert lib.g16_hgemm_splitk(y.data_ptr(), w.data_ptr(), out.data_ptr(), int(out16), b.data_ptr(), s.data_ptr(), M, N, K,
                                ks, cus, ws.data_ptr(), ws.numel(), cnt.data_ptr(), cnt.numel(), st) == 0
    return out


@pytest.mark.parametrize("M,K,N,tile,ks", ROUTES)
@pytest.mark.parametrize("kind", KINDS)
def test_stream_equals_the_two_launch_sequence(cuda, M, K, N, tile, ks, kind):
    import gtx16_fp16 as g
    from gtx16_fp16 import _clib, kernels

    lib = _clib.load()
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    if cus != 256:
        pytest.skip(f"the route table is for 256 CUs (this device has {cus})")
    assert planned_tile(lib, M, N, K, cus) == tile and lib.g16_hgemm_plan(M, N, K, cus) == ks
    w = randn((K, N), seed=1, scale=0.02, dtype=torch.float16)
    bias = randn((N,), seed=2, scale=0.02)
    wd, b = w.to(cuda), bias.to(cuda)
    for out16 in (False, True):
        x = _x(M, K, kind, out16)
        xd = x.to(cuda)
        odt, bits = (torch.float16, torch.int16) if out16 else (torch.float32, torch.int32)
        two = _two(lib, xd, wd, b, out16, cus)
        outs = [g.mm_t(xd, wd, b, odt) for _ in range(4)]
        torch.cuda.synchronize()
        y = outs[0]
        for o in outs[1:]:
            assert torch.equal(o.view(bits), y.view(bits))
        assert all(int(c.count_nonzero()) == 0 for c in kernels._counters.values())
        assert torch.equal(torch.isnan(y), torch.isnan(two))
        fin = ~torch.isnan(two)
        if kind == "within" or out16:
            assert torch.equal(y[fin], two[fin])  # no value is scaled below fp16's normal range
        xd64, ok = xd.double(), torch.isfinite(xd).all(1)
        ref = (xd64 @ wd.double() + b.double())[ok]
        err, err2 = ((o.double()[ok] - ref).norm(dim=1) / ref.norm(dim=1) for o in (y, two))
        # fp16 rounding of the activations (and of an fp16 output): 2^-11 per value each
        assert (err <= 2.0 ** -10).all() and (err <= err2 * 1.001 + 1e-7).all(), (kind, out16, err.max(), err2.max())
        want = oracle.mm_t(x[:16].numpy(), w.numpy(), bias.numpy(), "float16" if out16 else "float32") if M >= 16 else None
        if want is not None:
            assert torch.equal(torch.isnan(y[:16]).cpu(), torch.isnan(torch.from_numpy(want)))


def test_stream_replays_in_a_graph(cuda):
    import gtx16_fp16 as g

    shapes = [(64, 1024, 1024), (160, 4104, 1536), (1024, 264, 1024), (64, 1024, 11008)]
    xs = [outlier_rows(randn((M, K), seed=M), 0.05, 2e3, 2e5, seed=6).to(cuda) for M, K, _ in shapes]
    ws = [randn((K, N), seed=7, scale=0.02, dtype=torch.float16).to(cuda) for _, K, N in shapes]
    eager = [g.mm_t(x, w) for x, w in zip(xs, ws)]
    s = torch.cuda.Stream(cuda)
    s.wait_stream(torch.cuda.current_stream(cuda))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        for x, w in zip(xs, ws):
            g.mm_t(x, w)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=s):
            outs = [g.mm_t(x, w) for x, w in zip(xs, ws)]
    for _ in range(3):
        for o in outs:
            o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for o, e, x, w in zip(outs, eager, xs, ws):
            assert torch.equal(o, e) and torch.equal(g.mm_t(x, w), e)


@pytest.mark.parametrize("shape,K,N", [((64,), 1024, 1024), ((3, 37), 1000, 264), ((2, 2, 40), 768, 3072)])
@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("bias", [True, False])
def test_fast_linear_small_batches_are_mm_t(cuda, shape, K, N, dt, bias):
    # FastLinear's short path for M > 8 gives mm_t's bits; what it does not take (views, another bias
    # dtype, a replaced weight) still goes through the general path
    import torch.nn as nn

    import gtx16_fp16 as g

    torch.manual_seed(0)
    fl = g.FastLinear.from_linear(nn.Linear(K, N, bias=bias).to(cuda))
    x = torch.randn(*shape, K, device=cuda).to(dt)
    want = g.mm_t(x.reshape(-1, K), fl.weight_t, fl.bias, dt).reshape(*shape, N)
    if dt == torch.float32:
        assert fl._small_gemm(x, x.numel() // K) is not None
    y = fl(x)
    assert y.shape == want.shape and y.dtype == dt and torch.equal(y, want)
    strided = torch.randn(*shape, 2 * K, device=cuda).to(dt)[..., ::2]
    assert torch.equal(fl(strided), fl(strided.contiguous()))
    fl.weight_t = (fl.weight_t * 2).contiguous()
    want = g.mm_t(x.reshape(-1, K), fl.weight_t, fl.bias, dt).reshape(*shape, N)
    assert torch.equal(fl(x), want)
    if bias:
        fl.bias = fl.bias.half()
        if dt == torch.float32:
            assert fl._small_gemm(x, x.numel() // K) is None
        assert torch.equal(fl(x), g.mm_t(x.reshape(-1, K), fl.weight_t, fl.bias.float(), dt).reshape(*shape, N))


@pytest.mark.parametrize("thresh", [1.0, 2.0, 4.0, 1024.0, 2.0 ** 15])
def test_gemm_call_takes_any_threshold(cuda, thresh):
    # a row of 2^127 has the largest exponents: for thresholds below 4 a direct launch's factor would
    # not be a normal number (two launches there); past 2^15 the scaled value itself is no fp16 number
    from gtx16_fp16 import _clib

    lib = _clib.load()
    M, K, N = 64, 1024, 1024
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    x = randn((M, K), seed=11)
    x[5, 100] = 2.0 ** 127
    w = randn((K, N), seed=12, scale=0.02, dtype=torch.float16)
    xd, wd = x.to(cuda), w.to(cuda)
    out = torch.empty(M, N, device=cuda)
    ks = lib.g16_hgemm_plan(M, N, K, cus)
    bufs = [torch.zeros(max(16, n), dtype=torch.uint8, device=cuda)
            for n in (lib.g16_mm_t_scratch_bytes(M, N, K, cus), lib.g16_hgemm_splitk_workspace_bytes(M, N, K, ks, cus),
                      lib.g16_hgemm_splitk_counter_bytes(M, N, K, ks, cus))]
    st = torch.cuda.current_stream(cuda).cuda_stream
    assert lib.g16_mm_t_gemm(xd.data_ptr(), 1, wd.data_ptr(), out.data_ptr(), 0, None, thresh, M, N, K, cus,
                             *(v for b in bufs for v in (b.data_ptr(), b.numel())), st) == 0
    ref = x.double() @ w.double()
    err = (out.cpu().double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert (err <= 2.0 ** -10).all(), err.max()  # fp16 rounding of the activations: 2^-11 per value


# splits of 2 to 8 slices on each tile of the route
@pytest.mark.parametrize("M,K,N,tile,ks", [r for r in ROUTES if r[4] > 1])
def test_slices_past_fp32_range_cancel(cuda, M, K, N, tile, ks):
    # partial sums near 1e40 in the first and the last slice cancel; what is left is finite, as it is
    # where one pass over the row scales it (sums in scaled units until the epilogue)
    import gtx16_fp16 as g

    x = randn((M, K), seed=M + K)
    w = randn((K, N), seed=1, scale=0.02, dtype=torch.float16)
    x[:, :40] = x[:, K - 40:] = 0.0  # (the other rows do not meet the weights of 1)
    rows = [0, M // 2, M - 1]
    for i, r in enumerate(rows):
        x[r] = 0.0
        x[r, :40], x[r, K - 40:] = 3e38, -3e38
        x[r, K // 2] = (-2.0) ** (127 - i)
    w[:40] = w[K - 40:] = 1.0
    for odt in (torch.float32, torch.float16):
        y = g.mm_t(x.to(cuda), w.to(cuda), None, odt)
        torch.cuda.synchronize()
        ref = x.double() @ w.double()
        if odt == torch.float16:
            assert not torch.isnan(y[rows]).any()  # (past fp16's range)
            y, ref = (torch.stack([t[r] for r in range(M) if r not in rows]) for t in (y, ref))
        err = (y.cpu().double() - ref).norm(dim=1) / ref.norm(dim=1)
        # fp16 rounding of the activations (and of an fp16 output): 2^-11 per value each
        assert (err <= 2.0 ** -10).all(), err.max()


# (M, K, N, slices, streamed): above 64 rows and past K = 4096 only 3 slices and more, or up to 6 tile
# columns, are streamed
@pytest.mark.parametrize("M,K,N,ks,streamed", [
    (333, 4104, 4096, 1, False), (700, 4352, 1024, 1, False), (128, 6144, 4096, 2, False), (160, 11008, 1536, 3, True),
    (142, 8192, 1856, 5, True), (333, 4096, 4096, 1, False), (64, 4096, 11008, 2, True), (1024, 1024, 1024, 1, True),
    (3193, 6600, 432, 1, True), (2318, 6304, 264, 1, True), (2527, 6232, 264, 2, True), (1554, 5320, 432, 1, False)])
def test_route_by_its_rounding(cuda, M, K, N, ks, streamed):
    # a row with |max| 2000 is halved by the rowscale cast, and 3 * 2^-24 with it (to 2 * 2^-24, a tie to
    # even); the streamed tiles scale only rows that leave fp16's range
    import gtx16_fp16 as g
    from gtx16_fp16 import _clib

    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    if cus != 256:
        pytest.skip(f"the route table is for 256 CUs (this device has {cus})")
    assert _clib.load().g16_hgemm_plan(M, N, K, cus) == ks
    x = torch.zeros(M, K)
    x[M - 1, 0], x[M - 1, K - 1] = 2000.0, 3 * 2.0 ** -24
    w = torch.zeros(K, N, dtype=torch.float16)
    w[K - 1] = 1.0
    y = g.mm_t(x.to(cuda), w.to(cuda)).cpu()
    assert (y[M - 1] == (3 if streamed else 4) * 2.0 ** -24).all() and not y[:-1].any()
