"""The column quantizer's one-pass outputs (ck_quantize_cols_init) at the edges
of its tiles: K at and between the padded sizes, V around one column group and
one tile, views off 16-byte alignment. The quotient is correctly rounded, so
everything equals torch's expression bit for bit."""

from __future__ import annotations

import pytest
import torch

from carrykernel_amd.statequant import kernel as sq

pytestmark = pytest.mark.gpu


def _expect(x, qmax):
    x = x.cpu()  # torch's GPU division by a Python number multiplies by its reciprocal
    scale = x.abs().amax(-2).clamp(min=1e-12) / qmax
    codes = torch.round(x / scale[..., None, :]).clamp(-qmax, qmax)
    return codes.to(torch.int8).cuda(), scale.cuda()


def _off_by_one(x):
    """The same values one element past a 16-byte boundary."""
    buf = torch.zeros(x.numel() + 1, device=x.device)
    buf[1:] = x.flatten()
    return buf[1:].view_as(x)


@pytest.mark.parametrize("K", [1, 15, 16, 17, 64, 100, 128, 200, 256, 300])
@pytest.mark.parametrize("V", [1, 4, 31, 128, 130, 132])
@pytest.mark.parametrize("aligned", [True, False])
def test_outputs(K, V, aligned):
    g = torch.Generator(device="cuda").manual_seed(K * 1000 + V)
    x = torch.randn(3, 2, K, V, generator=g, device="cuda") * 0.3
    x[1, 0] = 0.0  # an empty state: the scale's floor
    x = x if aligned else _off_by_one(x)
    codes, scale = _expect(x, 127.0)
    got = sq.per_v_channel_quantize(x)
    for name, a, b in zip(("codes", "scale", "deq"), got, (codes, scale, codes.float() * scale[..., None, :])):
        assert torch.equal(a, b), name
    codes6, scale6 = _expect(x, 31.0)
    for fmt in (sq.RES_FP32, sq.RES_FP16, sq.RES_FP8, sq.RES_INT8):
        c, s, e, es = sq.init_quant_state(x, bits=6, res_fmt=fmt)
        assert torch.equal(c, codes6) and torch.equal(s, scale6)
        assert e.shape == x.shape and e.dtype == sq.residual_dtype(fmt) and not e.float().any()
        assert (es is None) == (fmt != sq.RES_INT8)
        if es is not None:
            assert es.shape == s.shape and es.dtype == torch.float32 and not es.any()


@pytest.mark.parametrize("K,V", [(100, 36), (64, 33)])
def test_infinities_and_huge_values(K, V):
    """Shapes of the IEEE form: a column with an infinity has scale inf (finite
    values give 0), one near the largest float divides without its reciprocal;
    the columns beside them are not affected."""
    g = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randn(2, K, V, generator=g, device="cuda")
    ref, _ = _expect(x, 127.0)
    x[0, 3, 1] = float("inf")
    x[1, :, 2] *= 1e38 / x[1, :, 2].abs().max()
    huge, s_huge = _expect(x[1, :, 2:3], 127.0)
    codes, scale, _ = sq.per_v_channel_quantize(x)
    assert scale[0, 1] == float("inf")
    rows = [r for r in range(K) if r != 3]
    assert not codes[0, rows, 1].any()
    assert torch.equal(codes[1, :, 2:3], huge) and torch.equal(scale[1, 2:3], s_huge)
    cols = [c for c in range(V) if c not in (1, 2)]
    assert torch.equal(codes[:, :, cols], ref[:, :, cols])


@pytest.mark.parametrize("V", [(1 << 21) + 4, 1 << 28])
def test_very_wide_matrix(V, K=16):
    """Aligned, V % 4 == 0 and K a power of two (the non-IEEE arithmetic), up to
    2^32 elements: columns of both ends and the middle as torch quantizes them."""
    x = torch.empty(K, V, device="cuda").normal_(std=0.3, generator=torch.Generator(device="cuda").manual_seed(5))
    at = torch.cat([torch.arange(40), torch.arange(V // 2, V // 2 + 40), torch.arange(V - 40, V)]).cuda()
    cols = lambda t: t[..., at].contiguous()  # noqa: E731
    codes, scale = _expect(cols(x), 127.0)
    got = sq.per_v_channel_quantize(x)
    for name, a, b in zip(("codes", "scale", "deq"), got, (codes, scale, codes.float() * scale[None, :])):
        assert torch.equal(cols(a), b), name
    del got
    c, s, e, es = sq.init_quant_state(x[None, None], res_fmt=sq.RES_INT8)
    assert torch.equal(cols(c)[0, 0], codes) and torch.equal(cols(s)[0, 0], scale) and not e.any() and not es.any()


@pytest.mark.parametrize("M,K,V", [(3, 1, 256), (3, 2, 127), (4096, 4, 7), (8192, 16, 16), (8192, 16, 17),
                                   (16384, 17, 6), (16384, 32, 9), (16384, 100, 4), (16384, 256, 3), (65536, 128, 4)])
def test_many_small_matrices(M, K, V):
    """One thread per column up to a few columns, a workgroup per matrix above."""
    x = torch.randn(M, K, V, generator=torch.Generator(device="cuda").manual_seed(K + V), device="cuda")
    x[1], x[2, 0, 0] = 0.0, float("inf")
    codes, scale = _expect(x, 127.0)
    got = sq.per_v_channel_quantize(x)
    ok = torch.ones_like(scale, dtype=torch.bool)
    ok[2, 0] = False   # the infinity's column: a scale of inf, its other codes 0
    assert torch.equal(got[1], scale) and torch.equal(got[0].mT[ok], codes.mT[ok])
    assert torch.equal(got[2].mT[ok], (codes.float() * scale[:, None, :]).mT[ok]) and not got[0][2, 1:, 0].any()
    for fmt in (sq.RES_FP32, sq.RES_FP16, sq.RES_FP8, sq.RES_INT8):
        c, s, e, es = sq.init_quant_state(x, res_fmt=fmt)
        assert torch.equal(c, got[0]) and torch.equal(s, scale) and not e.float().any()
        assert (es is None) == (fmt != sq.RES_INT8) and (es is None or not es.any())
