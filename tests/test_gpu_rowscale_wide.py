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
