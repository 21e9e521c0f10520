"""The C++ forms of the ops (tq_torch.cpp) against the checks of ops.py: they
take the ordinary call, leave everything else to Python's checks and errors,
and launch on the caller's current stream."""
import math

import pytest
import torch

from turboquant_amd import _lib, ops
from turboquant_amd import workloads as W
from turboquant_amd.geometry import hadamard_signs


def test_cpu_tensors_are_left_to_the_checks():
    nat = ops._native()
    cache = torch.zeros((2, 1, 16, 2, 48), dtype=torch.uint8)
    k, s = torch.zeros((3, 2, 64)), torch.ones(64)
    slots = torch.arange(3, dtype=torch.int32)
    assert nat.write_cache(cache, k, k, s, slots, 64, 64) is False
    with pytest.raises(RuntimeError, match="GPU only"):
        ops.quantize_write_kv_cache(cache, k, k, s, slots, 64, 64)
    assert nat.mse_quantize(k, 64, 4, s, [0.0] * 15) is None
    with pytest.raises(RuntimeError, match="GPU only"):
        ops.mse_quantize(k, 64, 4, s, [0.0] * 15)


@pytest.mark.gpu
def test_op_errors_are_the_ones_of_the_python_checks():
    ops.register_ops()
    op = torch.ops.turboquant_write.quantize_write_kv_cache
    cache = torch.zeros((2, 1, 16, 2, 48), dtype=torch.uint8, device="cuda")
    k, s = torch.zeros((3, 2, 64), device="cuda").half(), hadamard_signs(64, "cuda")
    slots = torch.arange(3, dtype=torch.int32, device="cuda")
    with pytest.raises(RuntimeError, match="slot_mapping must be int32"):
        op(cache, k, k, s, slots.long(), 64, 64)
    with pytest.raises(RuntimeError, match="must share a float dtype"):
        op(cache, k, k.float(), s, slots, 64, 64)
    with pytest.raises(_lib.TQError, match="does not pad"):  # refused by the library
        op(cache, k, k, hadamard_signs(256, "cuda"), slots, 64, 128)
    op(cache, k[:0], k[:0], s, slots[:0], 64, 64)
    op(cache, k, k, s, slots, 64, 64)


@pytest.mark.gpu
def test_ordinary_calls_are_taken_and_others_are_not():
    nat = ops._native()
    c = W.decode_case(5, 2, [40, 9], 8, 2, 64)
    cache, pd = W.build_cache(c, "cuda:0")
    d = W.decode_inputs(c, pd, "cuda:0")
    rows = ops.balanced_rows(2, 8, 2, pd)
    o = torch.empty((2, 8, pd), dtype=torch.float16, device="cuda")
    ws = [torch.empty((rows, 8, pd), device="cuda"), torch.empty((rows, 8), device="cuda"),
          torch.zeros(4, dtype=torch.int32, device="cuda")]
    args = [d["q"], cache, d["indices"], d["indptr"], d["seq"], 2, 64, pd, 1 / math.sqrt(64),
            hadamard_signs(pd, "cuda"), o, *ws]
    assert nat.decode_balanced(*args, False)
    for i, bad in ((0, d["q"].float()), (1, cache[:, :, :, :1]), (3, d["indptr"].long()),
                   (4, d["seq"][:1]), (10, o.float()), (11, ws[0][:, :, :32]), (13, ws[2][:3])):
        assert not nat.decode_balanced(*args[:i], bad, *args[i + 1:], False), i
    x = torch.randn((6, 5, 128), device="cuda")
    s, b = hadamard_signs(128, "cuda"), [(i - 7) / 8 for i in range(15)]
    packed, norms = nat.mse_quantize(x, 128, 4, s, b)
    assert packed.shape == (6, 5, 64) and norms.shape == (6, 5)
    off = torch.empty(x.numel() + 1, device="cuda")[1:].view(x.shape).copy_(x)
    for bad in (x.half(), x.transpose(0, 1), off, x[:0]):
        assert nat.mse_quantize(bad, 128, 4, s, b) is None
    # what it leaves, Python copies and launches: the same result
    assert torch.equal(ops.mse_quantize(off, 128, 4, s, iter(b))[0], packed)
    assert torch.equal(ops.mse_quantize(x.transpose(0, 1), 128, 4, s, b)[1], norms.t())


@pytest.mark.gpu
def test_calls_run_on_the_current_stream():
    x = torch.randn((200000, 128), device="cuda")
    s, b = hadamard_signs(128, "cuda"), [(i - 7) / 64 for i in range(15)]
    want = ops.mse_quantize(x, 128, 4, s, b)[0].clone()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    for _ in range(5):
        with torch.cuda.stream(side):
            y = torch.zeros_like(x)
            y.copy_(x)  # ordered before the call only on the side stream
            got = ops.mse_quantize(y, 128, 4, s, b)[0]
        side.synchronize()
        assert torch.equal(got, want)
