"""The statequant step's column tiles (ck_tiles.h, TileForm): V below one
4-column group, around one group, one wave, the widest tile and two tiles, where
the last thread shares columns with its neighbour, in place and out of place, on
tensors one element off alignment. Bit for bit against the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from carrykernel_amd.hip import binding
from carrykernel_amd.statequant import kernel as sq

pytestmark = pytest.mark.gpu

FORMATS = [sq.RES_FP32, sq.RES_FP16, sq.RES_FP8, sq.RES_INT8]


def _off(t):
    """A copy one element past an allocation's start."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
    buf[1:] = t.cuda().flatten()
    return buf[1:].view(t.shape)


def _np(e, fmt):
    e = e.cpu()
    if fmt == sq.RES_FP16:
        return e.view(torch.int16).numpy().view(np.uint16)
    return e.view(torch.uint8).numpy() if fmt == sq.RES_FP8 else e.numpy()


@pytest.mark.parametrize("K", [16, 100, 128, 256])
@pytest.mark.parametrize("V", [1, 3, 4, 5, 31, 64, 96, 127, 129, 131, 160, 161, 225, 321])
def test_step(K, V):
    B, HV = 1, 2
    fmt = FORMATS[(V + K // 16) % 4]
    g = torch.Generator().manual_seed(K * 1000 + V)
    h0 = torch.randn(B, HV, K, V, generator=g) * 0.1
    codes, scale = oracle.quantize_cols(h0.numpy(), 127)
    r = torch.randn(B, HV, K, V, generator=g) * torch.from_numpy(scale)[:, :, None, :] * 0.3
    es = None
    if fmt == sq.RES_INT8:
        es = (r.abs().amax(-2) / 127).clamp(min=1e-12)
        r = torch.round(r / es[:, :, None, :]).clamp(-127, 127)
    e = r.to(sq.residual_dtype(fmt))
    q, k = torch.randn(B, HV, K, generator=g) * K ** -0.5, torch.randn(B, HV, K, generator=g) * K ** -0.5
    v, beta = torch.randn(B, HV, V, generator=g), torch.rand(B, HV, generator=g)
    alpha = torch.full((B, HV), 0.97)
    ref = oracle.quant_step_kv(codes, scale, _np(e, fmt), None if es is None else es.numpy(), q.numpy(), k.numpy(),
                               v.numpy(), alpha.numpy(), beta.numpy(), res_fmt=fmt)
    st = [_off(torch.from_numpy(codes)), _off(torch.from_numpy(scale)), _off(e),
          torch.zeros(B, HV, V, device="cuda") if es is None else _off(es)]
    x = [t.cuda() for t in (q, k, v, alpha, beta)]
    o = _off(torch.zeros(B, HV, V))

    def check(h, s, e_, es_):
        for a, b in zip((o, h, s, e_), ref):
            np.testing.assert_array_equal(_np(a, fmt) if a is e_ else a.cpu().numpy(), b)
        if fmt == sq.RES_INT8:
            np.testing.assert_array_equal(es_.cpu().numpy(), ref[4])

    new = [torch.empty_like(t) for t in st]
    ext = binding.load_extension()
    ext.gdn_quant_step(*st, *x, o, *new, 127.0, fmt, 128)
    check(*new)
    ext.gdn_quant_step(*st, *x, o, *st, 127.0, fmt, 128)  # in place
    check(*st)

    h = _off(h0)
    href, oref = oracle.fp32_step_kv(h0.numpy(), q.numpy(), k.numpy(), v.numpy(), alpha.numpy(), beta.numpy())
    ext.gdn_fp32_step(h, *x, o, h, 128)  # in place
    np.testing.assert_array_equal(h.cpu().numpy(), href)
    np.testing.assert_array_equal(o.cpu().numpy(), oref)


def test_very_wide_head():
    """A ragged head of two million columns."""
    B, HV, K, V = 1, 1, 2, (1 << 21) + 3
    g = torch.Generator().manual_seed(1)
    h0 = torch.randn(B, HV, K, V, generator=g) * 0.1
    codes, scale = oracle.quantize_cols(h0.numpy(), 127)
    e = torch.randn(B, HV, K, V, generator=g) * 1e-4
    q, k, v = torch.randn(B, HV, K, generator=g), torch.randn(B, HV, K, generator=g), torch.randn(B, HV, V, generator=g)
    alpha, beta = torch.full((B, HV), 0.9), torch.full((B, HV), 0.5)
    ref = oracle.quant_step_kv(codes, scale, e.numpy(), None, q.numpy(), k.numpy(), v.numpy(), alpha.numpy(),
                               beta.numpy(), res_fmt=sq.RES_FP32)
    got = sq.gdn_quant_step_fused(torch.from_numpy(codes).cuda(), torch.from_numpy(scale).cuda(), e.cuda(), None,
                                  *[t.cuda() for t in (q, k, v, alpha, beta)])
    for a, b in zip(got, ref):
        if a is not None:
            np.testing.assert_array_equal(a.cpu().numpy(), b)


@pytest.mark.parametrize("K,V", [(128, 6241), (256, 3969)])
def test_wide_ragged_heads(K, V):
    """Heads whose columns once left the last tile a single ragged group, in place
    and out of place."""
    test_step(K, V)


@pytest.mark.parametrize("K", [16, 128, 256])
@pytest.mark.parametrize("V", [100, 132, 164, 192, 260])
def test_full_tiles_of_a_ragged_head(K, V):
    """V a multiple of 4 whose last tile of whole groups has idle lanes."""
    test_step(K, V)


@pytest.mark.parametrize("K,V", [(256, (1 << 24) - 4), (1, (1 << 28) + 4)])
def test_offsets_around_32_bits(K, V):
    """The largest matrix with 32-bit lane offsets, and one past it (one column
    per thread): the columns at both ends as in a small head of their own."""
    g = torch.Generator(device="cuda").manual_seed(K)
    at = torch.cat([torch.arange(9), torch.arange(V // 2, V // 2 + 9), torch.arange(V - 9, V)]).cuda()
    cols = lambda t: t[..., at].contiguous()  # noqa: E731
    h = torch.randint(-127, 128, (1, 1, K, V), generator=g, device="cuda", dtype=torch.int8)
    e = torch.randint(0, 100, (1, 1, K, V), generator=g, device="cuda", dtype=torch.uint8)
    scale, v = torch.rand(1, 1, V, generator=g, device="cuda"), torch.randn(1, 1, V, generator=g, device="cuda")
    x = [torch.randn(1, 1, K, device="cuda") * K ** -0.5 for _ in range(2)]
    gates = [torch.full((1, 1), 0.9, device="cuda"), torch.full((1, 1), 0.5, device="cuda")]
    fp8 = torch.float8_e5m2
    got = sq.gdn_quant_step_fused(h, scale, e.view(fp8), None, *x, v, *gates, res_fmt=sq.RES_FP8)
    ref = sq.gdn_quant_step_fused(cols(h), cols(scale), cols(e).view(fp8), None, *x, cols(v), *gates,
                                  res_fmt=sq.RES_FP8)
    for a, b in zip(got[:4], ref[:4]):
        a, b = (t.view(torch.uint8) if t.dtype == fp8 else t for t in (a, b))
        assert torch.equal(cols(a), b)
    del got, e
    hf = h.float()
    got, o = sq.gdn_step_fused_fp32(hf, *x, v, *gates)
    ref, o_ref = sq.gdn_step_fused_fp32(cols(hf), *x, cols(v), *gates)
    assert torch.equal(cols(got), ref) and torch.equal(cols(o), o_ref)
    del got
    codes, s, _, _ = sq.init_quant_state(hf)
    c_ref, s_ref, _, _ = sq.init_quant_state(cols(hf))
    assert torch.equal(cols(codes), c_ref) and torch.equal(cols(s), s_ref)
