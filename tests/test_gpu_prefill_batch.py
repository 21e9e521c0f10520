"""The prefill of several requests in one launch (tq_prefill_attention_batch)
and the assembly of their keys and values (tq_prefill_gather), at the edges of
query blocks, tiles and launches, against float64 attention, the one-sequence
read-back and torch conversions."""
import math

import pytest
import torch

from turboquant_amd import ops
from turboquant_amd import workloads as W
from turboquant_amd.geometry import hadamard_signs, padded_dim
from tests import gpu_cases as G

pytestmark = pytest.mark.gpu

MANY = [(1 + i % 5, 3 * (i % 7)) for i in range(70)]  # more requests than one launch takes


def _attention64(q, k, v, scale):
    """Causal attention of q [n, hq, d] at the end of k, v [m, hkv, d]."""
    n, m, r = q.shape[0], k.shape[0], q.shape[1] // k.shape[1]
    late = torch.arange(m)[None, :] > (torch.arange(n) + m - n)[:, None]
    out = torch.empty(q.shape, dtype=torch.float64)
    for h in range(q.shape[1]):
        s = (q[:, h].double() @ k[:, h // r].double().t()) * scale
        s.masked_fill_(late, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // r].double()
    return out


# (new, cached) of each request; heads; head size; dtype of q and o
BATCHES = [
    ([(1, 0), (127, 0), (128, 1), (129, 0), (255, 64), (256, 0), (257, 63)], 4, 2, 128, torch.float16),
    ([(5, 3000), (130, 2000)], 4, 1, 128, torch.bfloat16),       # split keys and merges
    ([(1100, 0), (1030, 17)], 64, 8, 128, torch.float16),        # 256-row blocks
    ([(700, 0), (33, 1500), (64, 64)], 4, 4, 64, torch.bfloat16),
    ([(2100, 0)] * 4, 32, 8, 64, torch.float16),                 # two row blocks per wave
    ([(40, 900), (200, 0)], 4, 2, 256, torch.float16),
    ([(150, 30), (40, 900)], 6, 2, 96, torch.bfloat16),          # zero-padded head
    (MANY, 3, 3, 64, torch.float16),
]


@pytest.mark.parametrize("reqs,hq,hkv,hd,dtype", BATCHES)
def test_batch_against_float64(reqs, hq, hkv, hd, dtype):
    print(f"case: prefill batch {len(reqs)} requests {hq}/{hkv}/{hd} {dtype}", flush=True)
    pd, g = padded_dim(hd), torch.Generator().manual_seed(len(reqs) + hd)
    nq, nk = sum(r[0] for r in reqs), sum(sum(r) for r in reqs)
    q = torch.randn((nq, hq, hd), generator=g).to(dtype)
    kv = [torch.randn((nk + 7, hkv, hd), generator=g).half() for _ in range(2)]
    kd, vd = (torch.nn.functional.pad(t, (0, pd - hd)).to(G.DEV) for t in kv)
    wide = torch.full((nq, hq + 1, hd), 7.0, dtype=dtype, device=G.DEV)
    out, qd, scale = wide[:, :hq], q.to(G.DEV), 1.0 / math.sqrt(hd)
    args, a, b = [], 0, 3
    for i, (new, ctx) in enumerate(reqs):
        args.append((a, new, b, new + ctx, i % 2))  # the sources take turns
        a, b = a + new, b + new + ctx
    run = lambda: ops.prefill_attention_batch(qd, out, args, hkv, hd, pd, scale, kd, vd, kd, vd)
    run()
    first = out.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, first)
    assert (wide[:, hq:] == 7.0).all()
    for new_start, new, k0, kn, _ in args:
        if new > 300:  # the first and last rows stand for the rest
            pick = torch.tensor([0, 1, 127, 128, new - 2, new - 1])
        else:
            pick = torch.arange(new)
        for sel in ([pick] if new <= 300 else [pick[i:i + 1] for i in range(len(pick))]):
            end = kn - new + int(sel[-1]) + 1
            want = _attention64(q[new_start + sel], kv[0][k0:k0 + end], kv[1][k0:k0 + end], scale)
            got = first[(new_start + sel).to(G.DEV)].double().cpu()
            # fp16 probabilities and output; a bf16 output rounds by up to 2^-8
            tol = 2e-3 + (1e-2 if dtype == torch.float16 else 1.4e-2) * want.abs()
            assert bool(((got - want).abs() <= tol).all()), (got - want).abs().max().item()


# more query blocks or shares than one launch's list of items holds: runs of
# whole blocks (both workgroup shapes), runs of shares, several requests in them
RUNS = [
    ([(41217, 0)], 8, 1, 128, torch.float16),
    ([(41000, 100)], 16, 2, 64, torch.float16),
    ([(21000, 0)], 2, 1, 128, torch.bfloat16),
    ([(20600, 1000)], 1, 1, 256, torch.float16),
    ([(20999, 0)], 2, 1, 64, torch.bfloat16),
    ([(9000, 0), (700, 5000), (12000, 300), (1, 50), (129, 0)], 1, 1, 128, torch.float16),
    ([(5000, 60000)], 1, 1, 96, torch.float16),
    ([(420, 2000)] * 63 + [(1500, 9)], 4, 1, 128, torch.bfloat16),
]


@pytest.mark.parametrize("reqs,hq,hkv,hd,dtype", RUNS)
def test_runs_against_float64(reqs, hq, hkv, hd, dtype):
    test_batch_against_float64(reqs, hq, hkv, hd, dtype)


@pytest.mark.parametrize("hq,hkv", [(1, 1), (7, 7), (8, 8), (9, 3), (16, 2), (24, 8), (40, 8)])
def test_head_orders(hq, hkv):
    """Every head is served once whatever the head count (multiples of 8 are
    dealt to the XCDs in runs), split keys and merges included."""
    test_batch_against_float64([(5, 2500), (130, 0)], hq, hkv, 128, torch.float16)
    test_batch_against_float64([(70, 20)], hq, hkv, 256, torch.bfloat16)


@pytest.mark.parametrize("hkv,hd,dtype,aligned", [
    (8, 128, torch.bfloat16, True), (8, 128, torch.float16, False), (3, 64, torch.float32, True),
    (2, 256, torch.bfloat16, False), (2, 96, torch.float16, True), (1, 80, torch.float32, False),
    (2, 100, torch.bfloat16, True)])
def test_gather_against_read_back_and_conversion(hkv, hd, dtype, aligned):
    print(f"case: prefill gather {hkv}/{hd} {dtype} aligned={aligned}", flush=True)
    pd, dev = padded_dim(hd), G.DEV
    ctxs, fresh = [0, 333, 1, 0, 64, 517], [5, 1, 0, 0, 130, 33]
    c = W.decode_case(11 + hd, len(ctxs), [max(1, x) for x in ctxs], hkv, hkv, hd)
    cache, _ = G.build_cache(c)
    signs = hadamard_signs(pd, dev)
    table = torch.from_numpy(c["block_table"]).to(dev)
    g = torch.Generator("cuda").manual_seed(hd)
    off = 0 if aligned else 1
    key, value = (torch.randn((sum(fresh) + 2, 2 * hkv * hd + 8), generator=g, device=dev).to(dtype)
                  [:, off:off + hkv * hd].view(-1, hkv, hd) for _ in range(2))
    reqs, rows = [], 2
    for i, (n, f) in enumerate(zip(ctxs, fresh)):
        reqs.append((i, n, 1 + sum(fresh[:i]), f, rows))
        rows += n + f
    ok = torch.full((rows + 3, hkv, pd), 7.0, dtype=torch.float16, device=dev)
    ov = torch.full_like(ok, 7.0)
    ops.prefill_gather(cache, table, key, value, reqs, hd, pd, signs, ok, ov)
    torch.cuda.synchronize()
    for i, n, f0, f, r0 in reqs:
        if n:
            a, b = (torch.empty((n, hkv, hd), dtype=torch.float16, device=dev) for _ in range(2))
            ops.dequant_paged(cache, table[i].contiguous(), n, hkv, hd, pd, signs, a, b)
            assert torch.equal(ok[r0:r0 + n, :, :hd], a) and torch.equal(ov[r0:r0 + n, :, :hd], b)
        assert torch.equal(ok[r0 + n:r0 + n + f, :, :hd], key[f0:f0 + f].half())
        assert torch.equal(ov[r0 + n:r0 + n + f, :, :hd], value[f0:f0 + f].half())
    assert (ok[2:rows, :, hd:] == 0).all() and (ov[2:rows, :, hd:] == 0).all()
    for t in (ok, ov):  # rows before and after untouched
        assert (t[:2] == 7.0).all() and (t[rows:] == 7.0).all()


def test_gather_of_more_requests_than_a_launch_takes():
    """130 requests in one call (64 a launch), against a call for each."""
    hkv, hd, dev = 2, 64, G.DEV
    ctxs, fresh = [(7 * i) % 50 for i in range(130)], [(5 * i) % 9 for i in range(130)]
    c = W.decode_case(5, len(ctxs), [max(1, x) for x in ctxs], hkv, hkv, hd)
    cache, pd = G.build_cache(c)
    table, signs = torch.from_numpy(c["block_table"]).to(dev), hadamard_signs(pd, dev)
    g = torch.Generator("cuda").manual_seed(3)
    key, value = (torch.randn((sum(fresh), hkv, hd), generator=g, device=dev).to(torch.bfloat16)
                  for _ in range(2))
    reqs = [(i, n, sum(fresh[:i]), f, sum(ctxs[:i]) + sum(fresh[:i]))
            for i, (n, f) in enumerate(zip(ctxs, fresh))]
    out = [torch.full((sum(ctxs) + sum(fresh), hkv, pd), 7.0, dtype=torch.float16, device=dev)
           for _ in range(4)]
    ops.prefill_gather(cache, table, key, value, reqs, hd, pd, signs, *out[:2])
    for r in reqs:
        ops.prefill_gather(cache, table, key, value, [r], hd, pd, signs, *out[2:])
    assert torch.equal(out[0], out[2]) and torch.equal(out[1], out[3])
    assert not (out[0] == 7.0).all(-1).any()


def test_forward_in_passes_of_bounded_rows(monkeypatch):
    """A step whose gathered rows exceed the bound goes in several passes: the
    same result.  (Few key tiles, so no block is split in either.)"""
    from types import SimpleNamespace

    from turboquant_amd import vllm_backend_fused as B
    hq, hkv, hd, dev = 4, 2, 128, G.DEV
    reqs = [(40, 100), (3, 300), (130, 0), (2, 17), (60, 250), (1, 90), (200, 30)]
    lens = [a + b for a, b in reqs]
    c = W.decode_case(9, len(reqs), lens, hq, hkv, hd)
    cache, pd = G.build_cache(c)
    n = sum(r[0] for r in reqs)
    starts = [sum(r[0] for r in reqs[:i]) for i in range(len(reqs) + 1)]
    i32 = lambda v, d: torch.tensor(v, dtype=torch.int32, device=d)
    meta = SimpleNamespace(
        max_query_len=200, num_actual_tokens=n,
        block_table=torch.from_numpy(c["block_table"]).to(dev), slot_mapping=None,
        seq_lens=i32(lens, dev), seq_lens_cpu=i32(lens, "cpu"),
        query_start_loc=i32(starts, dev), query_start_loc_cpu=i32(starts, "cpu"))
    g = torch.Generator("cuda").manual_seed(4)
    for dtype in (torch.float16, torch.bfloat16):
        q, k, v = (torch.randn((n, h * hd), generator=g, device=dev).to(dtype)
                   for h in (hq, hkv, hkv))
        impl = B.TurboQuantFusedImpl(hq, hd, 1.0 / math.sqrt(hd), hkv, None, None, "fp8")
        run = lambda: impl.forward(None, q, k, v, cache, meta, output=torch.empty_like(q)).clone()
        monkeypatch.undo()
        want = run()
        for rows in (1, 140, 500):  # a request a pass, then several
            monkeypatch.setattr(B, "GATHER_BYTES", rows * 4 * hkv * pd)
            assert torch.equal(run(), want), (dtype, rows)


def test_batch_refuses_what_it_cannot_read():
    q = torch.zeros((8, 4, 64), dtype=torch.float16, device=G.DEV)
    k = torch.zeros((8, 2, 64), dtype=torch.float16, device=G.DEV)
    call = lambda r, **kw: ops.prefill_attention_batch(q, q.clone(), r, 2, 64, 64, 1.0, k, k, **kw)
    for bad in ((0, 9, 0, 9, 0), (0, 4, 5, 4, 0), (0, 4, 0, 3, 0), (0, 4, 0, 4, 1), (-1, 2, 0, 2, 0)):
        with pytest.raises(RuntimeError):
            call([bad])
    assert call([]).shape == q.shape
