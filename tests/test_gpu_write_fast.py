"""The write's kernels against each other: rows in aligned 16-byte pieces take
the fast kernel (or, in small launches, vector loads of the general one), the
same rows one element off alignment the general kernel's scalar loads, which
test_gpu_write.py and test_gpu_sweep.py pin to the oracle.  Same bytes for
every type, head size and special row, on both sides of the size rule."""
import pytest
import torch

from turboquant_amd import ops
from turboquant_amd import workloads as W
from turboquant_amd.geometry import hadamard_signs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rows(n, h, hd, dtype, seed):
    g = torch.Generator(DEV).manual_seed(seed)
    x = torch.randn((n, 2 * h, hd), generator=g, device=DEV)
    x[1] = 0.0
    x[2] *= 1e-20  # squares underflow
    x[3] *= 1e25   # squares overflow on finite values (fp16: infinities)
    x[4, :, 0] = float("inf")
    x[5, :, hd - 1] = -float("inf")
    x[6] *= 1e-38  # subnormals
    x[7] *= 3e4
    if dtype != torch.float16:  # (an fp16 row of full width stores a NaN norm with either sign)
        x[0, :, 3] = float("nan")
    return x.to(dtype)


def _write(rows, h, hd, slots, nb):
    shape, pd = W.cache_bytes(nb, h, hd)
    cache = torch.full(shape, 0x5A, dtype=torch.uint8, device=DEV)
    ops.quantize_write_kv_cache(cache, rows[:, :h], rows[:, h:], hadamard_signs(pd, DEV), slots,
                                hd, pd)
    return cache


@pytest.mark.parametrize("hd", [64, 72, 80, 96, 128, 136, 192, 256])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_fast_and_general_kernels_write_the_same_bytes(hd, dtype):
    # 8192 vectors is the last small launch: 512 x 8 tokens-heads, K and V
    for n, h in ((1, 1), (9, 3), (512, 8), (513, 8), (1400, 3)):
        print(f"case: write {hd} {dtype} n={n} h={h}", flush=True)
        rows = _rows(max(n, 8), h, hd, dtype, hd + n)[:n]
        off = torch.empty(rows.numel() + 1, dtype=dtype, device=DEV)[1:].view(rows.shape)
        off.copy_(rows)
        assert off.data_ptr() % 16 != 0 and rows.data_ptr() % 16 == 0
        nb = -(-n // 16) + 1
        g = torch.Generator(DEV).manual_seed(n)
        slots = torch.randperm(nb * 16, generator=g, device=DEV)[:n].to(torch.int32)
        if n > 8:
            slots[8] = -1
        assert torch.equal(_write(rows, h, hd, slots, nb), _write(off, h, hd, slots, nb))
