"""Calls whose workgroups together pass 2^32 work items, HIP's limit of one
launch: they run as launches over slices. The parts before, at and past the cut
are compared with the same call on those parts alone."""

from __future__ import annotations

import pytest
import torch

import bench
from carrykernel_amd.statequant import kernel as sq
from carrykernel_amd.vllm_integration import quantized_packed_decode as qpd

pytestmark = pytest.mark.gpu


def _parts(n, cut):
    """Indexes around the start, the cut and the end."""
    return torch.cat([torch.arange(s, min(s + 9, n)) for s in (0, cut - 4, n - 5)]).cuda()


def test_column_ingest():
    M = (1 << 26) + 5   # workgroups of 64 threads
    x = torch.randn(M, 1, 5, device="cuda")
    at = _parts(M, (1 << 26) - 1)
    for a, b in zip(sq.init_quant_state(x, res_fmt=sq.RES_INT8), sq.init_quant_state(x[at], res_fmt=sq.RES_INT8)):
        assert torch.equal(a[at], b)


def test_decode_of_many_heads():
    B, K, V = (1 << 22) + 5, 1, 128   # four workgroups of 256 threads per head
    h0, v = torch.randn(B, 1, K, V, device="cuda"), torch.randn(1, B, 1, V, device="cuda")
    q, k = torch.randn(1, B, 1, K, device="cuda"), torch.randn(1, B, 1, K, device="cuda")
    alpha, beta = torch.rand(1, B, 1, device="cuda"), torch.rand(1, B, 1, device="cuda")
    at = _parts(B, (1 << 22) - 1)
    o, *state = sq.gdn_quant_decode_fused(h0, q, k, v, alpha, beta, 1, res_fmt=sq.RES_INT8)
    ref_o, *ref = sq.gdn_quant_decode_fused(h0[at], *[t[:, at] for t in (q, k, v, alpha, beta)], 1, res_fmt=sq.RES_INT8)
    assert torch.equal(o[:, at], ref_o)
    for a, b in zip(state, ref):
        assert torch.equal(a[at], b)


def _requests(B, H, HV, K, V, live, dtype=torch.bfloat16):
    """Inputs of B requests of which only `live` have a slot (1, 2, ...)."""
    g = torch.Generator(device="cuda").manual_seed(3)
    mixed = torch.empty(B, 2 * H * K + HV * V, dtype=dtype, device="cuda")
    mixed[live] = torch.randn(len(live), mixed.shape[1], generator=g, device="cuda").to(dtype)
    a, b = (torch.randn(B, HV, generator=g, device="cuda").to(dtype) for _ in range(2))
    A_log, dt_bias = torch.randn(HV, generator=g, device="cuda"), torch.randn(HV, generator=g, device="cuda")
    ids = torch.zeros(B, dtype=torch.int32, device="cuda")
    ids[live] = torch.arange(1, len(live) + 1, dtype=torch.int32, device="cuda")
    return mixed, a, b, A_log, dt_bias, ids


@pytest.mark.parametrize("K,B,cut", [(18, (1 << 24) + 5, 1 << 24), (16, (1 << 25) + 5, 1 << 25)])
def test_packed_decode_of_many_requests(K, B, cut):
    """The masked kernel (256 threads per item) and the one-item kernel (128)."""
    H = HV = V = 1
    live = _parts(B, cut - 1)
    mixed, a, b, A_log, dt_bias, ids = _requests(B, H, HV, K, V, live)
    h0 = torch.randn(len(live) + 1, HV, V, K, device="cuda") * 0.1
    got = []
    for m, aa, bb, i in ((mixed, a, b, ids), (mixed[live], a[live], b[live], ids[live])):
        pool = qpd.init_quantized_state(len(live) + 1, HV, V, K, "cuda", h0=h0)
        out = torch.empty(len(m), 1, HV, V, device="cuda")
        qpd.quantized_gated_delta_rule_packed_decode(m, aa, bb, A_log, dt_bias, K ** -0.5, *pool, out, i)
        got.append((out, pool))
    (out, pool), (ref, ref_pool) = got
    assert torch.equal(out[live], ref) and ref.any()
    for x, y in zip(pool, ref_pool):
        assert torch.equal(x, y)
    out[live] = 0
    assert not out.any()   # requests without a slot


def test_float_state_of_many_requests():
    H = HV = V = 1
    K, B = 16, (1 << 24) + 5
    live = _parts(B, (1 << 24) - 1)
    mixed, a, b, A_log, dt_bias, ids = _requests(B, H, HV, K, V, live)
    state = torch.randn(len(live) + 1, HV, V, K, device="cuda").to(torch.bfloat16)
    st, st_ref = state.clone(), state.clone()
    out = torch.empty(B, 1, HV, V, device="cuda")
    bench.float_state_step(st, mixed, a, b, A_log, dt_bias, K ** -0.5, out, ids, True)
    ref = torch.empty(len(live), 1, HV, V, device="cuda")
    bench.float_state_step(st_ref, mixed[live], a[live], b[live], A_log, dt_bias, K ** -0.5, ref, ids[live], True)
    assert torch.equal(out[live], ref) and torch.equal(st, st_ref) and ref.any()
    out[live] = 0
    assert not out.any()
