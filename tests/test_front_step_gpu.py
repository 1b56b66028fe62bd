"""The statequant steps' C++ front end (csrc/front.cpp) against their Python one:
the same bits for contiguous inputs, and every other form declined there and
converted or refused by the Python checks as before."""

from __future__ import annotations

import pytest
import torch

from carrykernel_amd import _native
from carrykernel_amd.statequant import kernel as sq

pytestmark = pytest.mark.gpu


def _inputs(B, HV, K, V, fmt):
    g = torch.Generator(device="cuda").manual_seed(K + V)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    state = list(sq.init_quant_state(r(B, HV, K, V) * 0.1, res_fmt=fmt))
    return state, [r(B, HV, K) * K ** -0.5, r(B, HV, K) * K ** -0.5, r(B, HV, V), torch.rand(B, HV, device="cuda"),
                   torch.rand(B, HV, device="cuda")]


@pytest.fixture
def limited_memory():
    """limited_memory(n): from now on no more than n bytes of new GPU memory."""
    def limit(n):
        torch.cuda.empty_cache()
        total = torch.cuda.get_device_properties(0).total_memory
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + n) / total)
    yield limit
    torch.cuda.set_per_process_memory_fraction(1.0)


def _bits(ts):
    return [None if t is None else t.contiguous().view(torch.uint8).cpu() for t in ts]


def _same(a, b):
    assert type(a) is tuple and len(a) == len(b)
    for x, y in zip(_bits(a), _bits(b)):
        assert (x is None) == (y is None) and (x is None or torch.equal(x, y))


@pytest.mark.parametrize("fmt", [sq.RES_FP32, sq.RES_FP16, sq.RES_FP8, sq.RES_INT8])
@pytest.mark.parametrize("K,V", [(128, 128), (7, 3)])
def test_same_as_python(fmt, K, V, monkeypatch):
    state, x = _inputs(2, 3, K, V, fmt)
    front = _native._front
    assert front is not None
    got = sq.gdn_quant_step_fused(*state, *x, bits=6, res_fmt=fmt, quant_mode="exact")
    stream = _native.stream_handle(0)
    assert front.quant_step(*state, *x, 31.0, fmt, 1, stream) is not None
    h = torch.randn(2, 3, K, V, device="cuda")
    got32 = sq.gdn_step_fused_fp32(h, *x)
    assert front.fp32_step(h, *x, stream) is not None
    # other forms: 16-bit and strided inputs, wrong shapes, devices and formats
    xb = [t.to(torch.bfloat16) for t in x]
    strided = [t.transpose(0, 1).contiguous().transpose(0, 1) for t in x]
    cpu = [t.cpu() for t in x]
    for other in (xb, strided, [x[0][..., :-1], *x[1:]], cpu):
        assert front.quant_step(*state, *other, 127.0, fmt, 0, stream) is None
        assert front.fp32_step(h, *other, stream) is None
    assert front.quant_step(*state, *x, 127.0, (fmt + 1) % 4, 0, stream) is None
    got_b, got_s = sq.gdn_quant_step_fused(*state, *xb, res_fmt=fmt), sq.gdn_quant_step_fused(*state, *strided, res_fmt=fmt)
    with pytest.raises(ValueError):
        sq.gdn_quant_step_fused(*state, x[0][..., :-1], *x[1:], res_fmt=fmt)
    with pytest.raises(ValueError):
        sq.gdn_quant_step_fused(*state, *x, bits=9, res_fmt=fmt)
    monkeypatch.setattr(_native, "_front", None)
    _same(got, sq.gdn_quant_step_fused(*state, *x, bits=6, res_fmt=fmt, quant_mode="exact"))
    _same(got32, sq.gdn_step_fused_fp32(h, *x))
    _same(got_b, sq.gdn_quant_step_fused(*state, *[t.float() for t in xb], res_fmt=fmt))
    _same(got_s, sq.gdn_quant_step_fused(*state, *x, res_fmt=fmt))


def test_out_of_memory_is_torch_s(limited_memory):
    """An output that cannot be allocated raises torch.OutOfMemoryError."""
    state, x = _inputs(16, 16, 256, 256, sq.RES_FP32)
    assert _native._front is not None
    limited_memory(1 << 20)
    with pytest.raises(torch.OutOfMemoryError):
        sq.gdn_quant_step_fused(*state, *x)


def test_decode_without_room_for_the_converted_inputs(limited_memory):
    """bf16 inputs whose fp32 copies for all tokens do not fit run token by
    token, to the same bits (the copies take 136 MB, the outputs 2 MB)."""
    T, B, HV, K, V = 512, 8, 32, 128, 4
    g = torch.Generator(device="cuda").manual_seed(2)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    h0 = r(B, HV, K, V) * 0.1
    x = [t.to(torch.bfloat16) for t in (r(T, B, HV, K) * 0.1, r(T, B, HV, K) * 0.1, r(T, B, HV, V),
                                        torch.rand(T, B, HV, device="cuda"), torch.rand(T, B, HV, device="cuda"))]
    ref = [None if t is None else t.cpu() for t in sq.gdn_quant_decode_fused(h0, *x, T)]
    limited_memory(64 << 20)
    assert sq._decode_one_launch(h0, tuple(x), T, 8, sq.RES_FP32, "fast") is None
    got = sq.gdn_quant_decode_fused(h0, *x, T)
    _same(tuple(got), tuple(ref))
