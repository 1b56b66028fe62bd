"""init_quantized_state's one-pass row kernel (ck_quantize_rows_init) at the edges
of its tiles: K around a lane's elements, the lane counts and the longest row, row
counts that leave waves partly empty, rows off 16-byte alignment, every residual
layout written over dirty memory. Bit for bit against the oracle's in-dtype
restatement."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from carrykernel_amd import _native
from carrykernel_amd.vllm_integration import quantized_packed_decode as qpd

pytestmark = pytest.mark.gpu

NAMES = {torch.float32: "float32", torch.bfloat16: "bfloat16", torch.float16: "float16", torch.float64: "float64"}


def _dirty(n):
    """Leave n bytes of 0x55 in the caching allocator's free blocks."""
    for size in (n, n // 2, 4096, 512):
        t = torch.full((max(size, 1),), 0x55, dtype=torch.uint8, device="cuda")
        del t


@pytest.mark.parametrize("dtype", list(NAMES))
@pytest.mark.parametrize("K", [1, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 64, 100, 128, 129, 255, 256, 257, 511, 512, 513])
def test_every_k(K, dtype, S=3, HV=2, V=7):
    g = torch.Generator().manual_seed(K)
    h0 = (torch.randn(S, HV, V, K, generator=g) * 0.2).to(dtype)
    h0[1, 0, 2] = 0.0
    host = h0.double().numpy() if dtype == torch.float64 else h0.float().numpy()
    c_ref, s_ref = oracle.quantize_rows_in_dtype(host, NAMES[dtype], 127.0)
    for fmt, per_head in ((qpd.RESID_INT8, False), (qpd.RESID_INT4, True), (qpd.RESID_INT8, True)):
        if fmt == qpd.RESID_INT4 and K % 2:
            continue
        _dirty(S * HV * V * K)
        sc, ss, rc, rs = qpd.init_quantized_state(S, HV, V, K, "cuda", h0=h0.cuda(), resid_fmt=fmt,
                                                  per_head_resid_scale=per_head)
        np.testing.assert_array_equal(sc.cpu().numpy(), c_ref)
        np.testing.assert_array_equal(ss.cpu().numpy(), s_ref)
        assert not rc.any() and not rs.any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("rows", [1, 5, 333])
def test_codes_and_scales_only(rows, K, dtype):
    """ck_quantize_rows on aligned rows of a power of two, strided and with zero
    rows; nothing past its outputs is written."""
    g = torch.Generator().manual_seed(rows + K)
    x = torch.zeros(rows, K + 16, dtype=dtype)
    x[:, :K] = (torch.randn(rows, K, generator=g) * 0.2).to(dtype)
    x[rows // 2] = 0.0
    c_ref, s_ref = oracle.quantize_rows_in_dtype(x[:, :K].float().numpy(), NAMES[dtype], 127.0)
    xd, codes = x.cuda(), torch.full((rows * K + 64,), 77, dtype=torch.int8, device="cuda")
    scale = torch.full((rows + 16,), -1.0, device="cuda")
    st = _native.lib().ck_quantize_rows(xd.data_ptr(), _native.dtype_code(xd, "x"), K + 16, rows, K, 127.0,
                                        codes.data_ptr(), scale.data_ptr(), _native.stream_handle(0))
    _native.check(st, "ck_quantize_rows")
    np.testing.assert_array_equal(codes[:rows * K].view(rows, K).cpu().numpy(), c_ref)
    np.testing.assert_array_equal(scale[:rows].cpu().numpy(), s_ref)
    assert (codes[rows * K:] == 77).all() and (scale[rows:] == -1.0).all()


@pytest.mark.parametrize("K", [100, 300])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_infinities(K, dtype):
    """Rows of a ragged K: beside an infinity the finite values are 0 (scale
    inf), the other rows are not affected."""
    x = torch.randn(1, 1, 9, K, device="cuda").to(dtype)
    ref = qpd.init_quantized_state(1, 1, 9, K, "cuda", h0=x)
    x[0, 0, 4, 7] = float("inf")
    sc, ss, _, _ = qpd.init_quantized_state(1, 1, 9, K, "cuda", h0=x)
    assert ss[0, 0, 4] == float("inf") and not sc[0, 0, 4].any()
    rows = [0, 1, 2, 3, 5, 6, 7, 8]
    assert torch.equal(sc[0, 0, rows], ref[0][0, 0, rows]) and torch.equal(ss[0, 0, rows], ref[1][0, 0, rows])
