"""The rowscale cast's workgroup-per-row form (up to 512 rows, and K > 4096): bit-exact against the
oracle at the edges of its register cache (K = 4096, 16384) and of the rule (512 and 513 rows), row-major
and packed, with rescaled rows, NaN, infinities and zeros."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from _inputs import outlier_rows, randn
from _packing import pack_a

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K", [(1, 8), (9, 4096), (9, 4104), (300, 264), (512, 1032), (513, 1032), (513, 4104),
                                 (12, 16384), (10, 16392), (17, 40000)])
@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
def test_rowscale_wide_bitexact(cuda, M, K, dt):
    from gtx16_fp16 import _clib

    lib = _clib.load()
    x = outlier_rows(randn((M, K), seed=M + K), 0.3, 2e3, 6e4 if dt == torch.float16 else 2e5, seed=3)
    if M > 8:
        x[1] = 0.0
        x[2, K - 1] = float("nan")
        x[3, K // 2] = float("-inf")
        x[4, K - 1] = 3e4  # the row's only large value, in its last chunk
    x = x.to(dt)
    xd = x.to(cuda)
    st = torch.cuda.current_stream(cuda).cuda_stream
    name = "f32" if dt == torch.float32 else "f16"
    want, S, _ = oracle.rowscale(x.numpy())
    y = torch.empty(M, K, dtype=torch.float16, device=cuda)
    s = torch.empty(M, device=cuda)
    assert getattr(lib, f"g16_rowscale_{name}")(xd.data_ptr(), y.data_ptr(), s.data_ptr(), M, K, 1024.0, st) == 0
    yp = torch.full((lib.g16_packed_a_bytes(M, K) // 2,), 7.0, dtype=torch.float16, device=cuda)
    sp = torch.empty(M, device=cuda)
    assert getattr(lib, f"g16_rowscale_pack_{name}")(xd.data_ptr(), yp.data_ptr(), sp.data_ptr(), M, K, 1024.0, st) == 0
    torch.cuda.synchronize()
    got, gp = y.cpu().numpy(), yp.cpu().numpy()
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got.view(np.uint16)[~nan], want.view(np.uint16)[~nan])
    pw = pack_a(want).reshape(gp.shape)
    pn = np.isnan(pw)
    assert np.array_equal(np.isnan(gp), pn) and np.array_equal(gp.view(np.uint16)[~pn], pw.view(np.uint16)[~pn])
    for t in (s, sp):
        assert np.array_equal(t.cpu().numpy().view(np.uint32), S.astype(np.float32).view(np.uint32))


def test_rowscale_of_more_rows_than_one_launch_holds(cuda):
    # 2^24 + 3 rows of 4104 fp16 values (138 GB, cast onto themselves: each value is read before it is
    # written): a workgroup of 256 threads per row is past the 2^32 threads of a launch
    from gtx16_fp16 import _clib

    M, K = (1 << 24) + 3, 4104
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info(cuda)[0] < 150 * 10 ** 9:
        pytest.skip("needs 150 GB of free GPU memory")
    x = torch.zeros(M, K, dtype=torch.float16, device=cuda)
    s = torch.zeros(M, device=cuda)
    rows = [0, (1 << 23) - 1, 1 << 23, (1 << 24) - 1, 1 << 24, M - 1]
    for i, r in enumerate(rows):
        x[r, K - 1 - i] = 2048.0 * (i + 1)
    want, S, _ = oracle.rowscale(x[rows].cpu().numpy())
    st = torch.cuda.current_stream(cuda).cuda_stream
    assert _clib.load().g16_rowscale_f16(x.data_ptr(), x.data_ptr(), s.data_ptr(), M, K, 1024.0, st) == 0
    got, gs = x[rows].cpu().numpy(), s[rows].cpu().numpy()
    ones = int((s == 1.0).sum())
    del x, s
    torch.cuda.empty_cache()
    assert np.array_equal(got.view(np.uint16), want.view(np.uint16)) and np.array_equal(gs, S.astype(np.float32))
    assert ones == M - len(rows)


@pytest.mark.parametrize("packed", [False, True])
def test_rowscale_of_short_rows_past_one_launch(cuda, packed):
    # 2^26 + 5 rows of 8: four rows to a workgroup, past the 2^32 threads as well
    from gtx16_fp16 import _clib

    lib = _clib.load()
    M, K = (1 << 26) + 5, 8
    if torch.cuda.mem_get_info(cuda)[0] < 8 * 10 ** 9:
        pytest.skip("needs 8 GB of free GPU memory")
    x = torch.zeros(M, K, dtype=torch.float16, device=cuda)
    rows = [0, (1 << 23) - 1, 1 << 23, (1 << 26) - 1, 1 << 26, M - 1]
    for i, r in enumerate(rows):
        x[r, i] = 2048.0 * (i + 1)
    want, S, _ = oracle.rowscale(x[rows].cpu().numpy())
    s = torch.zeros(M, device=cuda)
    y = torch.full((lib.g16_packed_a_bytes(M, K) // 2 if packed else M * K,), 7.0, dtype=torch.float16, device=cuda)
    st = torch.cuda.current_stream(cuda).cuda_stream
    fn = lib.g16_rowscale_pack_f16 if packed else lib.g16_rowscale_f16
    assert fn(x.data_ptr(), y.data_ptr(), s.data_ptr(), M, K, 1024.0, st) == 0
    if packed:  # row r's 8 values, one chunk of its 256-row block (a single block of 32 columns wide)
        blocks = y.view(-1, 16, 64, 8)
        sw = [(r % 256 >> 1) & 3 for r in rows]
        got = torch.stack([blocks[r // 256, r % 256 // 16, r % 16 * 4 + w] for r, w in zip(rows, sw)])
    else:
        got = y.view(M, K)[rows]
    assert np.array_equal(got.cpu().numpy().view(np.uint16), want.view(np.uint16))
    assert np.array_equal(s[rows].cpu().numpy(), S.astype(np.float32))
    assert int((s == 1.0).sum()) == M - len(rows) and int((y != 0).sum()) == len(rows)


@pytest.mark.parametrize("M,K,dt", [(2048, 4104, torch.float32), (2053, 5120, torch.float32), (2053, 5128, torch.float32),
                                    (4096, 4104, torch.float16), (4100, 6400, torch.float16), (4100, 6408, torch.float16)])
def test_packed_rows_a_little_past_4096(cuda, M, K, dt):
    # a wavefront per row with a remainder past its registers, and a workgroup per row just beyond the rule:
    # bit-exact against the oracle on a few rows, and the packed bytes those of the row-major cast
    from gtx16_fp16 import _clib

    lib = _clib.load()
    x = randn((M, K), seed=M + K)
    x[5] *= 5000.0 if dt == torch.float32 else 500.0
    x[7, K - 1], x[M - 1, 4100] = 6e4, 3e4  # a row's only large value, past the registers
    x[9] = 0.0
    x = x.to(dt)
    xd = x.to(cuda)
    st = torch.cuda.current_stream(cuda).cuda_stream
    name = "f32" if dt == torch.float32 else "f16"
    y = torch.empty(M, K, dtype=torch.float16, device=cuda)
    s, sp = torch.empty(M, device=cuda), torch.empty(M, device=cuda)
    yp = torch.full((lib.g16_packed_a_bytes(M, K) // 2,), 7.0, dtype=torch.float16, device=cuda)
    assert getattr(lib, f"g16_rowscale_{name}")(xd.data_ptr(), y.data_ptr(), s.data_ptr(), M, K, 1024.0, st) == 0
    assert getattr(lib, f"g16_rowscale_pack_{name}")(xd.data_ptr(), yp.data_ptr(), sp.data_ptr(), M, K, 1024.0, st) == 0
    torch.cuda.synchronize()
    rows = [0, 5, 7, 9, 255, 256, M - 1]
    want, S, _ = oracle.rowscale(x[rows].numpy())
    assert np.array_equal(y[rows].cpu().numpy().view(np.uint16), want.view(np.uint16))
    assert np.array_equal(sp[rows].cpu().numpy(), S.astype(np.float32)) and torch.equal(s, sp)
    pw = pack_a(y.cpu().numpy()).reshape(-1)
    assert np.array_equal(yp.cpu().numpy().view(np.uint16), pw.view(np.uint16))
