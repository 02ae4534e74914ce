"""The direct GEMM route (g16_mm_t_direct: fp32 activations read and cast by the 256x256 GEMM itself,
rows rescaled as they leave fp16's range) against the two-launch sequence (rowscale cast, packed
GEMM) and the fp64 oracle: ragged M, N and K (K tails of 8 and 24), one K step, fp32 and fp16 outputs,
both weight layouts, rows past fp16's range from the first or the last K step on and several times
over, infinities and NaN."""
from __future__ import annotations

import pytest
import torch

import oracle
from _inputs import outlier_rows, randn

pytestmark = pytest.mark.gpu

# (M, K, N), each with 192 or more tiles of 256x256 on at most 4 tile columns
SHAPES = [(12500, 768, 1000), (49153, 8, 256), (16640, 1048, 768), (24600, 96, 520), (65536, 152, 264)]
KINDS = ["within", "outliers", "special", "late"]


@pytest.fixture(scope="module")
def lib(cuda):
    from gtx16_fp16 import _clib

    return _clib.load()


def _x(M, K, kind, out16):
    x = randn((M, K), seed=M + K)
    if kind == "outliers":
        x = outlier_rows(x, 0.01, 2e3, 1e4 if out16 else 2e5, seed=3)
    elif kind == "special":
        for r, k, v in ((0, K - 1, "inf"), (255, 0, "-inf"), (256, K // 2, "nan"), (M - 1, K - 1, "nan")):
            x[r, k] = float(v)
        x[M - 1, 0] = 1e38 if not out16 else 2.0
    elif kind == "late" and not out16:
        # the last value of a row, and one row raised by step after step
        x[7, K - 1] = 70000.0
        x[M - 1, K - 1] = -3e6
        for i, k in enumerate(range(0, K, 32)):
            x[300, k] = 7e4 * 3.0 ** min(i, 20)
    return x


def _two(lib, x, wp, b, out16):
    M, K, N = x.shape[0], x.shape[1], b.numel()
    st = torch.cuda.current_stream(x.device).cuda_stream
    xp = torch.empty(lib.g16_packed_a_bytes(M, K) // 2, dtype=torch.float16, device=x.device)
    s = torch.empty(M, device=x.device)
    out = torch.empty(M, N, dtype=torch.float16 if out16 else torch.float32, device=x.device)
    assert lib.g16_rowscale_pack_f32(x.data_ptr(), xp.data_ptr(), s.data_ptr(), M, K, 1024.0, st) == 0
    fn = lib.g16_hgemm_packed_ab_f16out if out16 else lib.g16_hgemm_packed_ab_f32out
    assert fn(xp.data_ptr(), wp.data_ptr(), out.data_ptr(), b.data_ptr(), s.data_ptr(), M, N, K, st) == 0
    return out


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("kind", KINDS)
def test_direct_equals_the_two_launch_sequence(lib, cuda, M, K, N, kind):
    import gtx16_fp16 as g
    from gtx16_fp16 import ops

    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    if cus != 256:
        pytest.skip(f"the shapes are for 256 CUs (this device has {cus})")
    assert lib.g16_mm_t_direct_route(M, N, K, cus) == 1
    w = randn((K, N), seed=1, scale=0.02, dtype=torch.float16)
    bias = randn((N,), seed=2, scale=0.02)
    wd, b = w.to(cuda), bias.to(cuda)
    wp = ops.pack_weight(wd)
    for out16 in (False, True):
        x = _x(M, K, kind, out16)
        xd = x.to(cuda)
        odt = torch.float16 if out16 else torch.float32
        bits = torch.int16 if out16 else torch.int32
        two = _two(lib, xd, wp, b, out16)
        plain = g.mm_t(xd, wd, b, odt)
        packed = ops.mm_t_prepacked(xd, wd, wp, b, odt)
        again = g.mm_t(xd, wd, b, odt)
        torch.cuda.synchronize()
        assert torch.equal(plain.view(bits), packed.view(bits)) and torch.equal(plain.view(bits), again.view(bits))
        assert torch.equal(torch.isnan(plain), torch.isnan(two))
        if kind in ("within", "special") or out16:
            # no finite value is scaled below fp16's normal range: the same bits
            fin = ~torch.isnan(two)
            assert torch.equal(plain[fin], two[fin])
        # against fp64, the two-launch result too (more than 8 rows, so that the oracle takes the GEMM's path)
        rows = sorted({0, 7, 255, 256, 300, M // 2, M - 1} | set(range(400, 408)))
        if kind == "outliers":
            rows = sorted(set(rows) | set(x.abs().amax(1).topk(8).indices.tolist()))
        ref = x[rows].double() @ w.double() + bias.double()
        fin = torch.isfinite(x[rows]).all(1)
        err, err2 = ((o[rows].cpu().double() - ref)[fin].norm(dim=1) / ref[fin].norm(dim=1) for o in (plain, two))
        # fp16 rounding of the activations (and of an fp16 output): 2^-11 per value each
        assert (err <= 2.0 ** -10).all(), (kind, out16, err.max())
        assert (err <= err2 * 1.001 + 1e-7).all(), (kind, out16, err, err2)
        want = oracle.mm_t(x[rows].numpy(), w.numpy(), bias.numpy(), "float16" if out16 else "float32")
        assert torch.equal(torch.isnan(plain[rows]).cpu(), torch.isnan(torch.from_numpy(want)))


def test_direct_replays_in_a_graph(cuda):
    import gtx16_fp16 as g

    M, K, N = 12500, 136, 1000
    x = outlier_rows(randn((M, K), seed=5), 0.01, 2e3, 2e5, seed=6).to(cuda)
    w = randn((K, N), seed=7, scale=0.02, dtype=torch.float16).to(cuda)
    eager = g.mm_t(x, w)
    s = torch.cuda.Stream(cuda)
    s.wait_stream(torch.cuda.current_stream(cuda))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        g.mm_t(x, w)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=s):
            out = g.mm_t(x, w)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager) and torch.equal(g.mm_t(x, w), eager)


# the 256x256 tile and, in their own loop, the 4-wavefront ones
@pytest.mark.parametrize("M,K,N", [(24600, 96, 520), (49153, 8, 256), (128, 1024, 1024), (1024, 264, 1024), (128, 6144, 8192)])
@pytest.mark.parametrize("pos", range(4))
def test_signaling_nan_beside_a_row_past_fp16_range(cuda, M, K, N, pos):
    # rows 8 apart share a lane of the cast: a signaling NaN in one of them, at any place of its 4 values,
    # leaves the others' exponents alone (a CPU copy keeps its bits)
    import gtx16_fp16 as g

    x = randn((M, K), seed=pos)
    base = (K // 8 // 2) * 8  # a chunk of 4 values past the first K steps
    huge, nan = [], []
    for blk in range(4):  # rows 32 blk + {0, 8, 16, 24}: one NaN row after, between and before huge ones
        rows = [32 * blk + 1 + 8 * i for i in range(4)]
        for i, r in enumerate(rows):
            if i == blk:
                x[r].view(torch.int32)[base + pos] = 0x7F800001 + 0x1000 * pos
                nan.append(r)
            else:
                x[r, base + (pos + i) % 4] = 1e5 * (i + 1)
                huge.append(r)
    assert torch.isnan(x[nan]).any(1).all()
    w = randn((K, N), seed=1, scale=0.02, dtype=torch.float16)
    y = g.mm_t(x.to(cuda), w.to(cuda)).cpu()
    assert torch.isnan(y[nan]).all()
    ref = x[huge].double() @ w.double()
    err = (y[huge].double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert (err <= 2.0 ** -10).all(), err  # fp16 rounding of the activations: 2^-11 per value


@pytest.mark.parametrize("thresh", [2.0, 1024.0, 2.0 ** 15])
def test_a_changed_threshold_reaches_every_route(cuda, monkeypatch, thresh):
    # ops.ROW_SCALE_THRESHOLD is read by each call: the direct route and the prepacked weight (two launches
    # for thresholds the direct kernel does not take), the streamed tiles and FastLinear's short path
    import torch.nn as nn

    import gtx16_fp16 as g
    from gtx16_fp16 import ops

    monkeypatch.setattr(ops, "ROW_SCALE_THRESHOLD", thresh)
    for M, K, N in ((24600, 96, 520), (64, 1024, 1024)):
        fl = g.FastLinear.from_linear(nn.Linear(K, N, bias=False).to(cuda))
        # 3 * 2^-24 rounds to 4 * 2^-24 wherever its row, whose largest value is 3, is halved (threshold 2,
        # two launches) and is itself elsewhere
        x = torch.zeros(M, K, device=cuda)
        x[M - 1, 0], x[M - 1, K - 1] = 3.0, 3 * 2.0 ** -24
        fl.weight_t.zero_()
        fl.weight_t[K - 1] = 1.0
        want = (4 if thresh == 2.0 else 3) * 2.0 ** -24
        outs = [g.mm_t(x, fl.weight_t), fl(x), ops.mm_t_prepacked(x, fl.weight_t, ops.pack_weight(fl.weight_t))]
        for y in outs:
            assert (y[M - 1] == want).all() and not y[:-1].any()
