"""The any-K decode's row ends (packed_decode_masked.h): every number of codes
past the last whole lane, so that each combination of the pieces a lane stores
occurs, heads whose rows leave waves of the workgroup empty, and pools that start
and end next to guard bytes, which have to stay as they are. Bit for bit against
the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from carrykernel_amd.vllm_integration import quantized_packed_decode as qpd
from tests._helpers import make_packed_inputs, make_pool

pytestmark = pytest.mark.gpu

GUARD = 0x5A


def _guarded(arr, lead):
    """A device copy of arr, `lead` guard bytes before it and 64 after."""
    raw = np.ascontiguousarray(arr).view(np.uint8).ravel()
    buf = torch.full((lead + raw.size + 64,), GUARD, dtype=torch.uint8, device="cuda")
    buf[lead:lead + raw.size] = torch.from_numpy(raw).cuda()
    t = buf[lead:lead + raw.size].view(torch.from_numpy(arr[:0].copy()).dtype).view(arr.shape)
    return buf, t


def _run(K, V, B, HV, resid, per_head, mode="fast", lead=0, act=torch.float32):
    H = 1
    S = B + 2
    pool = make_pool(S, HV, V, K, resid, per_head, seed=K)
    # the scales are fp32: guards of a multiple of 4 bytes
    bufs, dpool = zip(*(_guarded(x, lead if x.dtype == np.int8 else 4 * lead) for x in pool))
    idx = np.arange(1, B + 1, dtype=np.int32)
    idx[-1] = S - 1  # the pool's last row
    for t in range(2):
        mixed, a, b, A_log, dt_bias = make_packed_inputs(B, H, HV, K, V, seed=K + t, dtype=act)
        out = torch.empty(B, 1, HV, V, device="cuda")
        qpd.quantized_gated_delta_rule_packed_decode(
            mixed.cuda(), a.cuda(), b.cuda(), A_log.cuda(), dt_bias.cuda(), K ** -0.5, *dpool, out,
            torch.from_numpy(idx).cuda(), use_qk_l2norm_in_kernel=True, resid_fmt=resid, quant_mode=mode)
        ref = oracle.packed_decode(
            mixed.float().numpy(), a.float().numpy(), b.float().numpy(), A_log.float().numpy(),
            dt_bias.float().numpy(), K ** -0.5, *pool, idx, H, use_qk_l2norm=True, resid_fmt=resid,
            per_head=per_head, mode=oracle.MODE_EXACT if mode == "exact" else oracle.MODE_FAST)
        np.testing.assert_array_equal(out[:, 0].cpu().numpy(), ref)
        for name, buf, d, h in zip(("state_codes", "state_scale", "resid_codes", "resid_scale"), bufs, dpool, pool):
            np.testing.assert_array_equal(d.cpu().numpy(), h, err_msg=f"{name} at step {t}")
            n = d.numel() * d.element_size()
            g = buf.cpu().numpy()
            at = lead if h.dtype == np.int8 else 4 * lead
            assert np.all(g[:at] == GUARD) and np.all(g[at + n:] == GUARD), f"{name}: written outside"


@pytest.mark.parametrize("K", [*range(17, 32), 33, 63, 97, 127, 129, 191, 255, 257, 511, 1023])
@pytest.mark.parametrize("per_head", [False, True])
def test_int8_tails(K, per_head):
    _run(K, 19, 3, 2, qpd.RESID_INT8, per_head, lead=K % 3, act=torch.bfloat16 if K % 2 else torch.float32)


@pytest.mark.parametrize("K", [*range(18, 32, 2), 34, 62, 98, 126, 130, 254, 258, 1022])
@pytest.mark.parametrize("per_head", [False, True])
def test_int4_tails(K, per_head):
    _run(K, 19, 3, 2, qpd.RESID_INT4, per_head, mode="exact" if K % 4 else "fast", lead=K % 5,
         act=torch.float16 if K % 4 else torch.float32)


@pytest.mark.parametrize("K", [16, 32, 48, 64, 100, 128, 200, 256])
@pytest.mark.parametrize("V", [1, 33, 65, 96, 97, 127])
def test_partly_filled_workgroups(K, V):
    """Per head (waves without a row are not launched) and per row (they skip)."""
    _run(K, V, 2, 3, qpd.RESID_INT4, True, lead=1)
    _run(K, V, 2, 3, qpd.RESID_INT8, False, lead=1)


@pytest.mark.parametrize("K", range(1, 16))
@pytest.mark.parametrize("per_head", [False, True])
def test_rows_of_less_than_a_lane(K, per_head):
    """K below 16: a row is put together from its first and last bytes."""
    _run(K, 67, 3, 2, qpd.RESID_INT8, per_head, lead=K % 3, act=torch.bfloat16)
    if K % 2 == 0:
        _run(K, 67, 3, 2, qpd.RESID_INT4, per_head, mode="exact", lead=K % 5)
