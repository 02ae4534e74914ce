"""The raw GEMM route (g16_mm_t_raw: fp16 activations multiplied as they are on the unsplit 256x256 tile)
against the two-launch sequence (rowscale cast, packed GEMM) and fp64: ragged M, N and K (a last tile of
one row, K tails of 8 and 24, one K step), one round of tiles and persistent grids, fp32 and fp16
outputs, both weight layouts, rows past the threshold, infinities and NaN in x, an infinite weight."""
from __future__ import annotations

import pytest
import torch

import oracle
from _inputs import outlier_rows, randn

pytestmark = pytest.mark.gpu

SHAPES = [(2304, 256, 4096), (49153, 8, 256), (16640, 1048, 768), (4000, 1000, 5000), (65536, 152, 264)]
KINDS = ["within", "outliers", "special"]


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("kind", KINDS)
def test_raw_equals_the_two_launch_sequence(cuda, M, K, N, kind):
    import gtx16_fp16 as g
    from gtx16_fp16 import _clib, ops

    lib = _clib.load()
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    if cus != 256:
        pytest.skip(f"the shapes are for 256 CUs (this device has {cus})")
    assert lib.g16_mm_t_raw_route(M, N, K, cus) == 1
    x = randn((M, K), seed=M + K)
    w = randn((K, N), seed=1, scale=0.02, dtype=torch.float16)
    bias = randn((N,), seed=2, scale=0.02)
    if kind == "outliers":
        x = outlier_rows(x, 0.05, 2e3, 8e3, seed=3)
    elif kind == "special":
        for r, k, v in ((0, K - 1, "inf"), (255, 0, "-inf"), (256, K // 2, "nan"), (M - 1, K - 1, "-inf")):
            x[r, k] = float(v)
        w[K - 1, N - 3] = float("inf")  # an infinite sum that no infinite activation makes
        w[0, 1] = 0.0
    xd, wd, b = x.half().to(cuda), w.to(cuda), bias.to(cuda)
    wp = ops.pack_weight(wd)
    st = torch.cuda.current_stream(cuda).cuda_stream
    xp = torch.empty(lib.g16_packed_a_bytes(M, K) // 2, dtype=torch.float16, device=cuda)
    s = torch.empty(M, device=cuda)
    assert lib.g16_rowscale_pack_f16(xd.data_ptr(), xp.data_ptr(), s.data_ptr(), M, K, 1024.0, st) == 0
    for odt, bits in ((torch.float32, torch.int32), (torch.float16, torch.int16)):
        two = torch.empty(M, N, dtype=odt, device=cuda)
        fn = lib.g16_hgemm_packed_ab_f16out if odt == torch.float16 else lib.g16_hgemm_packed_ab_f32out
        assert fn(xp.data_ptr(), wp.data_ptr(), two.data_ptr(), b.data_ptr(), s.data_ptr(), M, N, K, st) == 0
        outs = [g.mm_t(xd, wd, b, odt), ops.mm_t_prepacked(xd, wd, wp, b, odt), g.mm_t(xd, wd, b, odt)]
        torch.cuda.synchronize()
        y = outs[0]
        for o in outs[1:]:
            assert torch.equal(o.view(bits), y.view(bits))
        assert torch.equal(torch.isnan(y), torch.isnan(two)) and torch.equal(torch.isinf(y), torch.isinf(two))
        if kind == "within":
            assert torch.equal(y.view(bits), two.view(bits))
        if kind == "special":
            assert torch.isnan(y[[0, 255, 256, M - 1]]).all() and torch.isinf(y[1, N - 3])
            fin = torch.isfinite(two)
            assert torch.equal(y[fin], two[fin])  # no finite row is scaled
            continue
        rows = list(range(64)) + [255, 256, M // 2, M - 1]
        ref = xd[rows].double() @ wd.double() + b.double()
        err, err2 = ((o[rows].double() - ref).norm(dim=1) / ref.norm(dim=1) for o in (y, two))
        # exact products, fp32 sums, one rounding of an fp16 output (2^-11 per value)
        assert (err <= (2.0 ** -10 if odt == torch.float16 else 1e-5)).all(), err.max()
        assert (err <= err2 * 1.001 + 1e-7).all(), (err.max(), err2.max())
        want = oracle.mm_t(xd[rows].cpu().numpy(), w.numpy(), bias.numpy(), str(odt).split(".")[1])
        assert oracle.rel_err(y[rows].cpu().numpy(), want) <= 1e-3


@pytest.mark.parametrize("M,K,N", [(777, 1096, 8192), (513, 1048, 10248), (1280, 2048, 4096)])
@pytest.mark.parametrize("kind", KINDS)
def test_medium_batches_with_and_without_scratch(cuda, M, K, N, kind):
    # 256x128 tiles in one round: mm_t and FastLinear cast and pack x, a C caller without scratch gets
    # the raw launch; the two-launch sequence's bits where no row is scaled, NaN rows alike
    import torch.nn as nn

    import gtx16_fp16 as g
    from gtx16_fp16 import _clib

    lib = _clib.load()
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    if cus != 256:
        pytest.skip(f"the shapes are for 256 CUs (this device has {cus})")
    x = randn((M, K), seed=M + K)
    if kind == "outliers":
        x = outlier_rows(x, 0.05, 2e3, 8e3, seed=3)
    elif kind == "special":
        x[0, K - 1], x[M - 1, 0], x[5, 7] = float("inf"), -float("inf"), float("nan")
    w, bias = randn((K, N), seed=1, scale=0.02, dtype=torch.float16), randn((N,), seed=2, scale=0.02)
    wd, b = w.to(cuda), bias.to(cuda)
    fl = g.FastLinear(K, N, device=cuda)
    fl.weight_t, fl.bias = wd, b
    st = torch.cuda.current_stream(cuda).cuda_stream
    for dt in (torch.float16, torch.float32):
        xd = x.to(dt).to(cuda)
        y = g.mm_t(xd, wd, b, dt)
        assert torch.equal(fl(xd).nan_to_num(1.0), y.nan_to_num(1.0)) and fl._wp is None
        fin = torch.isfinite(xd).all(1)
        assert torch.isnan(y[~fin]).all() and torch.isfinite(y[fin]).all()
        ref = xd[fin].double() @ wd.double() + b.double()
        err = (y[fin].double() - ref).norm(dim=1) / ref.norm(dim=1)
        # fp16 rounding of the activations and of an fp16 output: 2^-11 per value each
        assert (err <= 2.0 ** -10).all(), err.max()
        out = torch.empty_like(y)
        rc = lib.g16_mm_t_gemm(xd.data_ptr(), int(dt == torch.float32), wd.data_ptr(), out.data_ptr(),
                               int(dt == torch.float16), b.data_ptr(), 1024.0, M, N, K, cus, None, 0, None, 0, None, 0, st)
        assert rc == (-3 if dt == torch.float32 else 0)  # fp32 x needs its scratch, as on other tiles
        if rc == 0:
            assert torch.equal(torch.isnan(out), torch.isnan(y))
            err = (out[fin].double() - ref).norm(dim=1) / ref.norm(dim=1)
            assert (err <= 2.0 ** -10).all(), err.max()
            if kind != "outliers":
                assert torch.equal(out[fin], y[fin])


@pytest.mark.parametrize("M,K,N,raw", [(4096, 4104, 4096, False), (4096, 4128, 4096, True), (5000, 1048, 4096, True),
                                       (16384, 4104, 1024, True)])
@pytest.mark.parametrize("share", [False, True])
def test_raw_route_by_its_rounding(cuda, M, K, N, raw, share):
    # a row with |max| 2000 is halved by the rowscale cast, and 3 * 2^-24 with it (to 2 * 2^-24, a tie to
    # even); the raw launch rounds nothing. mm_t, the layer on its prepacked weight and, on every such
    # shape, the raw entry point itself
    import torch.nn as nn

    import gtx16_fp16 as g
    from gtx16_fp16 import _clib

    if torch.cuda.get_device_properties(cuda).multi_processor_count != 256:
        pytest.skip("the shapes are for 256 CUs")
    x = torch.zeros(M, K, dtype=torch.float16, device=cuda)
    x[M - 1, 0], x[M - 1, K - 1] = 2000.0, 3 * 2.0 ** -24
    fl = g.FastLinear.from_linear(nn.Linear(K, N, bias=False).to(cuda))
    fl.share_cast = share
    fl.weight_t.zero_()
    fl.weight_t[K - 1] = 1.0
    for y in (g.mm_t(x, fl.weight_t), fl(x)):
        assert (y[M - 1] == (3 if raw else 4) * 2.0 ** -24).all() and not y[:-1].any()
    assert fl._wp is not None
    y = torch.full((M, N), 7.0, device=cuda)
    st = torch.cuda.current_stream(cuda).cuda_stream
    assert _clib.load().g16_mm_t_raw(x.data_ptr(), fl.weight_t.data_ptr(), 0, y.data_ptr(), 0, None, M, N, K, 256, st) == 0
    assert (y[M - 1] == 3 * 2.0 ** -24).all() and not y[:-1].any()
