"""The skinny kernels with fp16 activations and fp16 outputs (M <= 8): wavefronts whose K rows start at
even and at odd rows (fp16 activations come in pairs), both strip widths, partial batches, every M;
an fp16 output is the fp32 output rounded once; FastLinear's fp16 token-by-token path on the split
kernel and on the decode layout, eager and in a graph."""
from __future__ import annotations

import pytest
import torch
import torch.nn as nn

import oracle
from _inputs import randn

pytestmark = pytest.mark.gpu


# (K, N): 1000 and 1096 give odd rows per wavefront on 256-column strips at some M, 4096 even ones;
# (264, 8712) is on 512-column strips
@pytest.mark.parametrize("M", range(1, 9))
@pytest.mark.parametrize("K,N", [(8, 8), (1000, 264), (1096, 1032), (4096, 512), (264, 8712), (1000, 8712)])
def test_skinny_fp16_activations_and_outputs(cuda, M, K, N):
    import gtx16_fp16 as g

    w = randn((K, N), seed=K, scale=0.02, dtype=torch.float16)
    b = randn((N,), seed=N, scale=0.02)
    for dt in (torch.float16, torch.float32):
        x = randn((M, K), seed=M, dtype=dt)
        for bias in (b, None):
            bd = None if bias is None else bias.to(cuda)
            y = g.mm_t(x.to(cuda), w.to(cuda), bd, torch.float32)
            h = g.mm_t(x.to(cuda), w.to(cuda), bd, torch.float16)
            torch.cuda.synchronize()
            assert h.dtype == torch.float16
            assert torch.equal(h.view(torch.int16), y.half().view(torch.int16))
            ref = oracle.skinny(x.numpy(), w.numpy(), None if bias is None else bias.numpy())
            assert oracle.rel_err(y.cpu().numpy(), ref) <= 1e-5


@pytest.mark.parametrize("ksplit", [1, 3, 7])
@pytest.mark.parametrize("M", [1, 4, 8])
def test_skinny_fp16_odd_slice_starts(cuda, M, ksplit):
    # explicit splits of K = 1000: 125, 42 and 18 rows per wavefront, so wavefronts start at odd rows;
    # +-inf at a slice's first and last row reach the outputs as the oracle's
    from gtx16_fp16 import _clib

    lib = _clib.load()
    K, N = 1000, 264
    x = randn((M, K), seed=3, dtype=torch.float16)
    x[0, 125] = float("inf")
    x[M - 1, 124] = float("-inf")
    w = randn((K, N), seed=4, scale=0.02, dtype=torch.float16)
    xd, wd = x.to(cuda), w.to(cuda)
    y = torch.empty(M, N, device=cuda)
    ws = torch.empty(max(16, lib.g16_skinny_workspace_bytes(M, N, K, ksplit)), dtype=torch.uint8, device=cuda)
    cnt = torch.zeros(max(16, lib.g16_skinny_counter_bytes(M, N, K, ksplit)), dtype=torch.uint8, device=cuda)
    st = torch.cuda.current_stream(cuda).cuda_stream
    assert lib.g16_skinny(xd.data_ptr(), 0, wd.data_ptr(), y.data_ptr(), 0, None, M, N, K, ksplit, ws.data_ptr(),
                          ws.numel(), cnt.data_ptr(), cnt.numel(), st) == 0
    torch.cuda.synchronize()
    want = torch.from_numpy(oracle.skinny(x.numpy(), w.numpy(), None))
    got = y.cpu().double()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got) * got.sign(), torch.isinf(want) * want.sign())
    fin = torch.isfinite(want)
    if fin.any():
        assert (got[fin] - want[fin]).norm() <= 1e-5 * want[fin].norm()


@pytest.mark.parametrize("decode_copy", [False, True])
@pytest.mark.parametrize("M", [1, 3, 4, 8])
def test_fast_linear_fp16_decode(cuda, M, decode_copy):
    import gtx16_fp16 as g
    from gtx16_fp16 import ops

    torch.manual_seed(M)
    K, N = 1096, 520
    fl = g.FastLinear.from_linear(nn.Linear(K, N).to(cuda))
    fl.prepack_decode = decode_copy
    x = torch.randn(2, M, K, device=cuda).half() if M <= 4 else torch.randn(M, K, device=cuda).half()
    rows = x.numel() // K
    y = fl(x)
    assert y.dtype == torch.float16 and y.shape == (*x.shape[:-1], N)
    strips = decode_copy and rows <= 4
    assert (fl._wd is not None) == strips
    x2 = x.reshape(-1, K)
    want = ops.skinny_strips(x2, fl._wd, fl.bias) if strips else g.mm_t(x2, fl.weight_t, fl.bias, torch.float32)
    assert torch.equal(y.reshape(-1, N).view(torch.int16), want.half().view(torch.int16))
    assert fl(x.float()).dtype == torch.float32
    s = torch.cuda.Stream(cuda)
    s.wait_stream(torch.cuda.current_stream(cuda))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        fl(x)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=s):
            out = fl(x)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, y) and torch.equal(fl(x), y)


# (M, K, N): what fp16 activations take on the matrix cores (6 x 14336 x 4096: 112 rows per wavefront),
# and shapes on 512-column strips or with short wavefronts, where they and fp32 ones take the FMA loop;
# rising values, infinities and NaN
@pytest.mark.parametrize("M,K,N", [(8, 8192, 9216), (7, 7000, 8200), (7, 4096, 11008), (6, 14336, 4096), (5, 11008, 520),
                                   (8, 4104, 8712), (7, 512, 9000)])
@pytest.mark.parametrize("kind", ["plain", "rising", "inf"])
@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
def test_skinny_matrix_core_groups(cuda, M, K, N, kind, dt):
    import gtx16_fp16 as g

    x = randn((M, K), seed=K + M)
    if kind == "rising":
        # later rows of K hold larger values (and the first ones of row 1 only zeros)
        x *= torch.linspace(-8, 8, K).exp2()
        x[1, : K // 2] = 0.0
    x = x.to(dt)
    w = randn((K, N), seed=N, scale=0.02, dtype=torch.float16)
    if kind == "inf":
        x[0, K - 1] = float("inf")
        x[M - 1, K // 2] = float("nan")
        w[K // 3, 5] = float("-inf")
        w[0, N - 1] = float("inf")
    y = g.mm_t(x.to(cuda), w.to(cuda)).cpu()
    again = g.mm_t(x.to(cuda), w.to(cuda)).cpu()
    assert torch.equal(y.view(torch.int32), again.view(torch.int32))
    want = torch.from_numpy(oracle.skinny(x.numpy(), w.numpy(), None))
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    assert torch.equal(torch.isposinf(y), torch.isposinf(want)) and torch.equal(torch.isneginf(y), torch.isneginf(want))
    fin = torch.isfinite(want)
    assert (y.double()[fin] - want[fin]).norm() <= 1e-5 * want[fin].norm()


# shapes whose wavefronts hold enough K rows for the matrix cores, and one on 512-column strips; fp32
# activations take them at M = 8 with 32 to 128 rows only, which none of these is
@pytest.mark.parametrize("M,K,N", [(5, 11008, 4096), (6, 14336, 4096), (7, 11008, 4096), (7, 4096, 11008), (8, 20480, 8192),
                                   (8, 4104, 8712)])
@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
def test_skinny_multiplies_every_bit_of_the_activations(cuda, M, K, N, dt):
    import gtx16_fp16 as g

    w = randn((K, N), seed=N, scale=0.02, dtype=torch.float16)
    x = randn((M, K), seed=K + M)
    x[1] = 0.0
    x[1, K // 3] = 1.0 + 2.0 ** -23       # one-hot, all 24 bits (fp16: rounds to 1)
    x[2] = 0.0
    x[2, 0], x[2, 7] = 3e4, 1e-3 / 3       # a large value that meets a zero weight, in one wavefront
    w[0] = 0.0
    x = x.to(dt)
    y = g.mm_t(x.to(cuda), w.to(cuda)).cpu().double()
    # a single product, rounded once to fp32 (2^-24) and added to zeros; the product itself is exact
    for row, k in ((1, K // 3), (2, 7)):
        want = x[row, k].double() * w[k].double()
        assert ((y[row] - want).abs() <= 2.0 ** -24 * want.abs()).all(), (row, (y[row] - want).abs().max())
    # every output: at most n roundings of 2^-24 each along its chain of sums, n < 512 here (the rows
    # of a wavefront, two parts, eight wavefronts, the slices), on sum |x w|
    x64, w64 = x.to(cuda).double(), w.to(cuda).double()
    bound = (512 * 2.0 ** -24 * (x64.abs() @ w64.abs())).cpu()
    assert ((y - (x64 @ w64).cpu()).abs() <= bound).all()


def test_fast_linear_fp16_sees_other_operands_at_the_same_address(cuda):
    # a bias or a weight replaced by a view of its memory: another type is used as what it is, another
    # shape is refused, after calls that had the layer's own tensors
    import gtx16_fp16 as g

    torch.manual_seed(0)
    K, N = 1024, 256
    x = torch.randn(4, K, device=cuda).half()
    fl = g.FastLinear.from_linear(nn.Linear(K, N).to(cuda))
    first = fl(x)
    bias = fl.bias.clone()
    fl.bias = fl.bias.view(torch.float16)[:N]
    fl.bias.copy_(torch.arange(N))
    want = g.mm_t(x, fl.weight_t, fl.bias.float(), torch.float16)
    assert torch.equal(fl(x), want) and torch.equal(fl(x), want)
    fl.bias = bias
    assert torch.equal(fl(x), first)
    whole = fl.weight_t
    fl.weight_t = whole[: K // 2]
    with pytest.raises(RuntimeError):
        fl(x)
    fl.weight_t = whole
    assert torch.equal(fl(x), first)
    # a scalar is still a batch of one for a layer of one feature
    one = g.FastLinear(1, 8, bias=False, device=cuda)
    one.weight_t.fill_(2.0)
    assert torch.equal(one(torch.tensor(3.0, dtype=torch.float16, device=cuda)), torch.full((8,), 6.0, device=cuda).half())
