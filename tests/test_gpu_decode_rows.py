"""The decode over the model's own rows (fp16 or bf16, head sizes below their
padded size) against the decode of the same rows converted and padded by
torch: the same arithmetic, so the same bits in fp16."""
import math

import pytest
import torch

from tests import gpu_cases as G
from turboquant_amd import ops
from turboquant_amd import workloads as W
from turboquant_amd.geometry import hadamard_signs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,hd", [(32, 8, 128), (6, 2, 96), (16, 4, 64), (16, 2, 256),
                                       (16, 1, 128), (16, 2, 200), (12, 1, 72)])
def test_rows_equal_padded_and_converted(hq, hkv, hd):
    print(f"case: decode rows {hq}/{hkv}/{hd}", flush=True)
    lens = [700, 0, 1, 33]
    c = W.decode_case(hd + hq, len(lens), lens, hq, hkv, hd, k_dist="t3")
    cache, pd = G.build_cache(c)
    d = G.decode_inputs(c, pd)
    signs, scale, dev = hadamard_signs(pd, G.DEV), 1.0 / math.sqrt(hd), G.DEV
    rows = ops.balanced_rows(len(lens), hq, hkv, pd)
    ws = [torch.empty((rows, hq, pd), dtype=torch.float32, device=dev),
          torch.empty((rows, hq), dtype=torch.float32, device=dev),
          torch.zeros(len(lens) + 2, dtype=torch.int32, device=dev)]
    for s in (signs, None):
        args = (cache, d["indices"], d["indptr"], d["seq"], hkv, hd, pd, scale, s)
        for dtype in (torch.float16, torch.bfloat16):
            # values that both types hold, in rows of a wider tensor
            q = d["q"][:, :, :hd].to(torch.bfloat16).to(torch.float16).to(dtype)
            wide = torch.full((len(lens), hq + 2, (hd + 15) // 8 * 8), 9.0, dtype=dtype, device=dev)
            wide[:, 1:-1, :hd] = q
            qv = wide[:, 1:-1, :hd]
            qp = torch.nn.functional.pad(q.to(torch.float16), (0, pd - hd))
            want = torch.empty((len(lens), hq, pd), dtype=torch.float16, device=dev)
            ops.decode_paged_balanced(qp, *args, want, *ws)
            half = torch.empty((len(lens), hq, hd), dtype=torch.float16, device=dev)
            ops.decode_paged_balanced_rows(qv, *args, half, *ws)
            assert torch.equal(half, want[:, :, :hd])
            out = torch.empty((len(lens), hq, hd), dtype=torch.bfloat16, device=dev)
            ops.decode_paged_balanced_rows(qv, *args, out, *ws)
            # both round the same sum: bf16 (8 significant bits) by up to 2^-8 of
            # it, fp16 by 2^-11
            err = (out.float() - half.float()).abs()
            assert bool((err <= half.float().abs() * (2.0 ** -8 + 2.0 ** -10) + 1e-7).all())
            assert (out[1] == 0).all()


def test_rows_refuse_other_types_and_shapes():
    c = W.decode_case(3, 1, [40], 4, 2, 96)
    cache, pd = G.build_cache(c)
    d = G.decode_inputs(c, pd)
    po = torch.empty((64, 4, pd), dtype=torch.float32, device=G.DEV)
    pl = torch.empty((64, 4), dtype=torch.float32, device=G.DEV)
    sp = torch.zeros(3, dtype=torch.int32, device=G.DEV)
    q = d["q"][:, :, :96].contiguous()
    for bad_q, bad_o in ((q.float(), q), (q, q.float()), (d["q"], q), (q, d["q"])):
        with pytest.raises(RuntimeError):
            ops.decode_paged_balanced_rows(bad_q, cache, d["indices"], d["indptr"], d["seq"], 2, 96,
                                           pd, 0.1, None, torch.empty_like(bad_o), po, pl, sp)
