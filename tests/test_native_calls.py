"""The C++ forms of the ops (tq_torch.cpp) against the checks of ops.py: they
take the ordinary call, leave everything else to Python's checks and errors,
and launch on the caller's current stream."""
import math

import pytest
import torch

from turboquant_amd import _lib, ops
from turboquant_amd import workloads as W
from turboquant_amd.geometry import entry_bytes, hadamard_signs


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


@pytest.mark.gpu
def test_strided_slots_and_signs_are_read_by_their_strides():
    """A column of a table of slots, and every other value of a longer table of
    signs, give what their packed copies give."""
    g = torch.Generator("cuda").manual_seed(5)
    hkv, hd, pd, n = 2, 96, 128, 37
    key, value = (torch.randn((n, hkv, hd), generator=g, device="cuda").half() for _ in range(2))
    table = torch.randperm(64 * 3, generator=g, device="cuda").to(torch.int32).view(64, 3)
    slots = table[:n, 1]
    signs = hadamard_signs(2 * pd, "cuda")[::2]
    assert not slots.is_contiguous() and not signs.is_contiguous()
    ops.register_ops()
    ebs = entry_bytes(hd)[2]
    caches = [torch.zeros((2, 12, 16, hkv, ebs), dtype=torch.uint8, device="cuda")
              for _ in range(3)]
    packed = (signs.contiguous(), slots.contiguous())
    ops.quantize_write_kv_cache(caches[0], key, value, *packed, hd, pd)
    ops.quantize_write_kv_cache(caches[1], key, value, signs, slots, hd, pd)
    torch.ops.turboquant_write.quantize_write_kv_cache(caches[2], key, value, signs, slots, hd, pd)
    assert torch.equal(caches[0], caches[1]) and torch.equal(caches[0], caches[2])
    outs = []
    pages = torch.arange(12, dtype=torch.int32, device="cuda")
    for s in (packed[0], signs):
        k, v = (torch.zeros((192, hkv, hd), dtype=torch.float16, device="cuda") for _ in range(2))
        ops.dequant_paged(caches[0], pages, 192, hkv, hd, pd, s, k, v)
        gk, gv = (torch.zeros((197, hkv, pd), dtype=torch.float16, device="cuda")
                  for _ in range(2))
        ops.prefill_gather(caches[0], pages[None], key, value, [(0, 192, 0, 5, 0)], hd, pd, s, gk,
                           gv)
        q = torch.randn((1, 4, pd), generator=torch.Generator("cuda").manual_seed(1),
                        device="cuda").half()
        i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device="cuda")
        o = torch.zeros_like(q)
        rows = ops.balanced_rows(1, 4, hkv, pd)
        ops.decode_paged_balanced(q, caches[0], pages, i32(0, 12), i32(192), hkv, hd, pd, 0.1, s,
                                  o, torch.empty((rows, 4, pd), device="cuda"),
                                  torch.empty((rows, 4), device="cuda"), i32(0, 0, 0))
        o2 = torch.zeros_like(q)
        ops.decode_paged_splitkv(q, caches[0], pages, i32(0, 12), i32(192), hkv, hd, pd, 0.1, s,
                                 o2, torch.empty((2, 4, pd), device="cuda"),
                                 torch.empty((2, 4), device="cuda"), 2, 96)
        outs.append((k, v, gk, gv, o, o2))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
