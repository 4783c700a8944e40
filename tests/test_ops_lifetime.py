"""Contiguous copies that an op makes of its inputs live until the library call is issued (CPU: the
library is replaced by a recorder).

A copy whose only reference is the expression that takes its address is freed at once, and the caching
allocator may hand its memory to the next copy, or to another thread of the stream, before the kernels
that read it are queued."""
import weakref

import pytest
import torch

from kernelbench_harbor_amd import inputs, ops

F16 = torch.float16


def _strided(t):
    """The same values in a tensor that is not contiguous."""
    u = torch.empty(*t.shape, 2, dtype=t.dtype)[..., 0]
    u.copy_(t)
    return u


class _Recorder:
    """Stands in for the library: the size queries return 0, a compute call notes which of the
    copies made so far are still alive."""

    def __init__(self, copies):
        self.copies, self.alive = copies, None

    def __getattr__(self, name):
        if name.endswith("_bytes"):
            return lambda *a: 0

        def call(*args):
            self.alive = [r() is not None for r in self.copies]
            return 0
        return call


def _silu():
    return (torch.zeros(4, 512, dtype=F16),)


def _mxfp8():
    return (torch.zeros(4, 256, dtype=torch.uint8), torch.zeros(4, 8, dtype=torch.uint8),
            torch.zeros(128, 256, dtype=torch.uint8), torch.zeros(128, 8, dtype=torch.uint8))


def _w8a8():
    return (torch.zeros(4, 256, dtype=torch.int8), torch.zeros(256, 128, dtype=torch.int8),
            torch.ones(4, 1, dtype=F16), torch.ones(1, 128, dtype=F16))


def _moe():
    return (torch.zeros(4, 128, dtype=F16), torch.zeros(4, 128, 128, dtype=F16), torch.zeros(4, 4, dtype=F16))


CALLS = {
    "w4a16_gemm": (ops.w4a16_gemm, lambda: inputs.w4a16(4, 256, 128, 128, F16, seed=0)),
    "w8a8_gemm": (ops.w8a8_gemm, _w8a8),
    "w8a8_gemm_i32": (ops.w8a8_gemm_i32, lambda: _w8a8()[:2]),
    "fp8w_gemm": (ops.fp8w_gemm, lambda: inputs.fp8w(4, 256, 128, 128, F16, seed=0)),
    "mxfp8_gemm": (ops.mxfp8_gemm, _mxfp8),
    "qmoe": (ops.qmoe, lambda: inputs.qmoe(4, 256, 4, 128, F16, seed=0)),
    "qmoe_ffn": (ops.qmoe_ffn, lambda: inputs.qmoe_ffn(4, 256, 256, 4, group=128, dtype=F16, seed=0)),
    "silu_fp8_quant": (ops.silu_fp8_quant, _silu),
    "moe": (lambda *a: ops.moe(*a, 2), _moe),
    "moe_route_top2": (ops.moe_route_top2, lambda: (torch.zeros(4, 8),)),
    "moe_route_topk": (lambda lg: ops.moe_route_topk(lg, 3), lambda: (torch.zeros(4, 8),)),
    "lora_qgemm": (ops.lora_qgemm, lambda: inputs.lora_qgemm(4, 256, 128, 16, 2, F16, seed=0)),
}


@pytest.mark.parametrize("name", sorted(CALLS))
def test_copies_outlive_the_library_call(name, monkeypatch):
    fn, make = CALLS[name]
    args = [_strided(t) for t in make()]
    assert not any(t.is_contiguous() for t in args if t.numel() > 1)
    copies = []
    plain = torch.Tensor.contiguous

    def contiguous(t, *a, **k):
        r = plain(t, *a, **k)
        if r is not t:
            copies.append(weakref.ref(r))
        return r

    lib = _Recorder(copies)
    monkeypatch.setattr(torch.Tensor, "contiguous", contiguous)
    monkeypatch.setattr(ops, "_check_device", lambda *t: (t[0].device, 0))
    monkeypatch.setattr(ops, "_stream_ptr", lambda idx: 0)
    monkeypatch.setattr(ops._lib, "load", lambda *a: lib)
    monkeypatch.setattr(ops, "_sizes", {})
    fn(*args)
    assert lib.alive, "the op made no copy"
    assert all(lib.alive), f"{lib.alive.count(False)} of {len(lib.alive)} copies freed before the call"
