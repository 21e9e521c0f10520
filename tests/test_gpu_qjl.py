"""The QJL products of TurboQuantProd above padded size 128 (tq_qjl.hip) at
the edges of their tiles (128 vectors x 128 outputs, K steps of 32), odd row
lengths and the smallest calls, against 64-bit products of the same operands;
and the row kernels at row lengths off the float4 pieces."""
import pytest
import torch

from turboquant_amd import algorithm as A
from turboquant_amd import ops

pytestmark = pytest.mark.gpu

SHAPES = [(129, 1), (200, 127), (256, 128), (257, 129), (384, 300), (513, 3), (512, 256),
          (1000, 130), (1023, 129), (1024, 64)]


def _prod(dim, bits, n):
    q = A.TurboQuantProd(dim, bits, device="cuda:0", seed=5)
    x = torch.randn((n, dim), generator=torch.Generator("cuda").manual_seed(dim + n),
                    device="cuda") * 2.0
    return q, x, q.mse.rotation.padded_dim, q.mse._host_tables()


@pytest.mark.parametrize("dim,n", SHAPES)
def test_quantize_signs_against_64_bits(dim, n):
    bits = 2 + dim % 4
    print(f"case: qjl quantize dim={dim} n={n} bits={bits}", flush=True)
    q, x, pd, (bnd, cen) = _prod(dim, bits, n)
    args = (x, pd, bits - 1, q.mse.rotation.signs, bnd, cen)
    packed, norms, resid, rnorm = ops.prod_quantize(*args)
    sh, sl, _, _ = q.qjl.halves(pd)
    p2, n2, z, r2 = ops.prod_quantize_qjl_ws(*args, sh, sl)
    assert torch.equal(p2, packed) and torch.equal(n2, norms) and torch.equal(r2, rnorm)
    s64, r64 = q.qjl.S.double(), resid.double()
    proj = r64 @ s64.t()
    wrong = z != torch.where(proj >= 0, 1, -1)
    # hi + lo holds S to 2^-23 and r to 2^-23, the product drops lo lo (2^-22),
    # the sum of 3 K products rounds to 2^-24 each
    bound = (r64.abs() @ s64.abs().t()) * (2.0 ** -21 + 3 * dim * 2.0 ** -24)
    assert bool((proj.abs() <= bound)[wrong].all()), proj[wrong].abs().max().item()


@pytest.mark.parametrize("dim,n", [(50, 33), (64, 1), (97, 65), (128, 31), (128, 40003)])
def test_fused_signs_against_64_bits(dim, n):
    """Up to padded size 128, at row scales whose residual needs other powers of
    two (down to the clamped norm), with a zero and a NaN row."""
    bits = 2 + dim % 4
    print(f"case: fused qjl quantize dim={dim} n={n} bits={bits}", flush=True)
    q, x, pd, (bnd, cen) = _prod(dim, bits, n)
    x *= 10.0 ** torch.arange(-9, 16, 4, device="cuda").repeat(n // 7 + 1)[:n, None].float()
    if n > 2:
        x[1], x[2, 3] = 0.0, float("nan")
    args = (x, pd, bits - 1, q.mse.rotation.signs, bnd, cen)
    packed, norms, resid, rnorm = ops.prod_quantize(*args)
    sh, sl, _, _ = q.qjl.halves(pd)
    p2, n2, z, r2 = ops.prod_quantize_qjl(*args, sh, sl)
    assert torch.equal(p2, packed) and torch.equal(n2.view(torch.int32), norms.view(torch.int32))
    assert torch.equal(r2.view(torch.int32), rnorm.view(torch.int32))
    s64, r64 = q.qjl.S.double(), resid.double()
    proj = r64 @ s64.t()
    wrong = z != torch.where(proj >= 0, 1, -1)  # (a NaN row: all -1)
    # as above, and resid itself is rounded to 2^-24; below its norm's 2^-35 a
    # component is under the quantum of a subnormal lo (2^-24 of rows near 2^10)
    bound = ((r64.abs() @ s64.abs().t()) * (2.0 ** -20 + 3 * dim * 2.0 ** -24)
             + s64.abs().sum(1) * 2.0 ** -35)
    assert bool((proj.abs() <= bound)[wrong].all()), proj[wrong].abs().max().item()


@pytest.mark.parametrize("dim,n", [(33, 5), (50, 33), (64, 1), (66, 40), (97, 65), (100, 31),
                                   (128, 1), (128, 40003)])
@pytest.mark.parametrize("scale", [1.0, 1e-6, 1e4])
def test_matrix_and_its_halves_give_the_same_bits(dim, n, scale):
    """Up to padded size 128 the kernels split S as they load it: what the calls
    with halves made beforehand give, also where S is not aligned."""
    bits = 2 + dim % 4
    q, x, pd, (bnd, cen) = _prod(dim, bits, n)
    q.qjl.S *= scale
    sh, sl, th, tl = q.qjl.halves(pd)
    args = (x, pd, bits - 1, q.mse.rotation.signs, bnd, cen)
    want = ops.prod_quantize_qjl(*args, sh, sl)
    back = (dim, pd, bits - 1, q.mse.rotation.signs, cen)
    off = torch.empty(dim * dim + 1, device="cuda")[1:].view(dim, dim).copy_(q.qjl.S)
    for s in (q.qjl.S, off, q.qjl.S.t().contiguous().t()):
        for a, b in zip(ops.prod_quantize_qjl_matrix(*args, s), want):
            assert torch.equal(a, b)
        assert torch.equal(ops.prod_dequantize_qjl_matrix(*want, *back, s),
                           ops.prod_dequantize_qjl(*want, *back, th, tl))
    assert torch.equal(q.quantize(x)[2], want[2])
    with pytest.raises(RuntimeError):
        ops.prod_quantize_qjl_matrix(*args, q.qjl.S[:-1, :-1].contiguous())
    with pytest.raises(RuntimeError):
        ops.prod_dequantize_qjl_matrix(*want, *back, q.qjl.S.double())


@pytest.mark.parametrize("dim,n", SHAPES)
def test_dequantize_term_against_64_bits(dim, n):
    """z S alone: norms of zero and a weight of 1, with signs and with any
    other int8 values (the product is defined for them too)."""
    print(f"case: qjl dequantize dim={dim} n={n}", flush=True)
    q, x, pd, (bnd, cen) = _prod(dim, 4, n)
    packed, _, _, _ = ops.prod_quantize(x, pd, 3, q.mse.rotation.signs, bnd, cen)
    _, _, th, tl = q.qjl.halves(pd)
    s64 = q.qjl.S.double()
    zero = torch.zeros(n, device="cuda")
    gamma = torch.full((n,), 1.0 / q.qjl.dequant_scale, device="cuda")
    gen = torch.Generator("cuda").manual_seed(n)
    for z in (torch.randint(0, 2, (n, dim), generator=gen, device="cuda", dtype=torch.int8) * 2 - 1,
              torch.randint(-128, 128, (n, dim), generator=gen, device="cuda", dtype=torch.int8)):
        got = ops.prod_dequantize_qjl_ws(packed, zero, z, gamma, dim, pd, 3,
                                         q.mse.rotation.signs, cen, th, tl).double()
        want = z.double() @ s64
        bound = (z.double().abs() @ s64.abs()) * (2.0 ** -22 + (2 * dim + 4) * 2.0 ** -24)
        assert bool(((got - want).abs() <= bound).all()), (got - want).abs().max().item()


# either side of the lines between the kernel forms (tiles of 32, 64, 128),
# ragged in vectors, outputs and K
FORMS = [(1000, 256), (1000, 257), (1000, 2560), (1000, 2561), (1023, 2700), (1000, 5121),
         (257, 8193), (513, 3001), (130, 20011), (512, 5000), (1024, 10300)]


@pytest.mark.parametrize("dim,n", FORMS)
def test_every_form_against_64_bits(dim, n):
    test_quantize_signs_against_64_bits(dim, n)
    test_dequantize_term_against_64_bits(dim, n)


@pytest.mark.parametrize("dim", [200, 1000])
def test_a_vector_has_the_same_bits_in_any_batch(dim):
    """Alone, in batches that take 64 x 64 tiles and in one that takes 128 x 128
    tiles: the sum over K runs in the same order in all of them."""
    q, x, _, _ = _prod(dim, 4, 21001)
    out = q.quantize(x)
    whole = q.dequantize(*out)
    for a, b in ((0, 0), (0, 1), (63, 64), (21000, 21001), (7, 72), (100, 2147), (0, 2048)):
        assert torch.equal(q.dequantize(*[t[a:b].clone() for t in out]), whole[a:b]), (a, b)


@pytest.mark.parametrize("dim", [50, 98, 130, 258, 514, 1002, 1023])
def test_row_kernels_off_the_float4_pieces(dim):
    n = 67
    q, qc = (A.TurboQuantMSE(dim, 3, device=d, seed=2) for d in ("cuda:0", "cpu"))
    x = torch.randn((n, dim), generator=torch.Generator().manual_seed(dim))
    packed, norms = q.quantize(x.cuda())
    pc, nc = qc.quantize(x)
    same = (packed.cpu() == pc).all(-1)
    assert same.float().mean().item() >= 0.95
    assert torch.allclose(norms.cpu(), nc, rtol=1e-6)
    assert torch.equal(q.dequantize(packed, norms).cpu(), qc.dequantize(packed.cpu(), norms.cpu()))


def test_empty_batches_and_replaced_matrix():
    q, x, pd, _ = _prod(300, 4, 40)
    packed, norms, z, rnorm = q.quantize(x[:0])
    assert packed.shape == (0, 256) and z.shape == (0, 300) and rnorm.shape == (0,)
    before = q.quantize(x)[2]
    q.qjl.S.neg_()  # written in place: the operand halves are made again
    assert torch.equal(q.quantize(x)[2], -before)
    q.qjl.S = -q.qjl.S
    assert torch.equal(q.quantize(x)[2], before)


def test_first_call_inside_a_graph():
    """Operand halves made during a capture hold values only when the graph
    runs: they are not kept for eager calls, and replays are right."""
    q, x, _, _ = _prod(400, 3, 70)
    q.mse._host_tables()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        z = q.quantize(x)[2]
    eager = q.quantize(x)[2].clone()
    for _ in range(3):
        z.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, eager)


def test_what_the_product_with_s_refuses_is_refused():
    """Vectors of another length in the same padded size, and a matrix of
    another shape or type, as the torch product with S refuses them."""
    q, x, _, _ = _prod(400, 4, 2100)
    out = q.quantize(x)
    for other in (300, 399, 500):
        with pytest.raises(RuntimeError):
            q.quantize(torch.randn((4, other), device="cuda"))
    s = q.qjl.S
    for bad in (s.double(), s.half(), s[:300, :300], s[:, :300], s.cpu()):
        q.qjl.S = bad
        with pytest.raises(RuntimeError):
            q.quantize(x)
        with pytest.raises(RuntimeError):
            q.dequantize(*out)
    small = A.TurboQuantProd(100, 3, device="cuda:0")
    small.qjl.S = small.qjl.S[:90, :90].contiguous()
    with pytest.raises(RuntimeError):
        small.quantize(torch.randn((4, 100), device="cuda"))


@pytest.mark.parametrize("dim", [100, 400])
def test_matrix_written_between_calls_captures_and_replays(dim):
    """A write that torch does not count, a capture right after it, and a
    graph whose matrix changes before its replays: always today's S."""
    q, x, _, _ = _prod(dim, 4, 2100)
    first = [t.clone() for t in q.quantize(x)]
    xh = q.dequantize(*first)
    q.qjl.S.data.neg_()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        z = q.quantize(x)[2]
        back = q.dequantize(*first)
    want = -first[2]
    mse = q.mse.dequantize(first[0], first[1])
    for _ in range(4):
        z.zero_(), back.zero_()
        g.replay()
        assert torch.equal(q.quantize(x)[2], want)
        torch.cuda.synchronize()
        assert torch.equal(z, want)
        # x_mse -+ term, the term's magnitude within a rounding of each sum
        got = (back - mse) * (1 if torch.equal(want, first[2]) else -1)
        assert torch.allclose(got, xh - mse, rtol=1e-5, atol=2.0 ** -22 * xh.abs().max().item())
        q.qjl.S.data.neg_()
        want = -want


@pytest.mark.parametrize("dim", [129, 256, 300, 512, 1000, 1023, 1024])
@pytest.mark.parametrize("transposed", [False, True])
def test_scaled_operand(dim, transposed):
    """hi + lo over the row's power of two is S: to half an ulp of a 22-bit
    number, or, where lo is subnormal, half its quantum 2^-24 (rows reach 2^14
    at least).  Rows of any magnitude, an empty and an infinite one."""
    s = torch.randn((dim, dim), generator=torch.Generator("cuda").manual_seed(dim), device="cuda")
    s *= 10.0 ** torch.linspace(-33, 37, dim, device="cuda")[:, None]
    s[3] = 0.0
    s[5, 7] = float("inf")
    if transposed:
        s = s.t().contiguous()
    pd = A.next_power_of_2(dim)
    hi, lo, scale = ops.qjl_operand(s, pd, transposed)
    rows = s.double() if not transposed else s.double().t()
    got = (hi.double() + lo.double()) * scale.double()[:, None]
    assert (got[dim:] == 0).all() and (got[:, dim:] == 0).all() and (got[3] == 0).all()
    got, top = got[:dim, :dim], rows.abs().amax(1)
    fine = torch.isfinite(top)
    assert not fine[5] and got[5, 7] == float("inf") and torch.isfinite(got[5, :7]).all()
    bound = rows.abs() * 2.0 ** -22 + (top * 2.0 ** -38)[:, None]
    assert ((got - rows).abs() <= bound)[fine].all()
    keep = fine & (top > 0)
    big = hi[:dim].abs().amax(1).double()[keep]
    assert (big >= 2.0 ** 14).all() and (big <= 2.0 ** 15).all()


@pytest.mark.parametrize("k", [-100, -20, 20, 100])
def test_matrix_of_another_magnitude(k):
    """S over fp32's range: signs do not change with a power of two on S, the
    read-back term changes by it exactly."""
    q, x, pd, (_, cen) = _prod(700, 4, 2300)
    packed, norms, z, rn = q.quantize(x)
    zero, one = torch.zeros_like(norms), torch.ones_like(rn)
    term = q.dequantize(packed, zero, z, one)
    q.qjl.S *= 2.0 ** k
    assert torch.equal(q.quantize(x)[2], z)
    assert torch.equal(q.dequantize(packed, zero, z, one), term * 2.0 ** k)


@pytest.mark.parametrize("dim", [50, 64, 97, 128, 257, 1000])
def test_operand_halves(dim):
    q = A.QJL(dim, device="cuda:0", seed=3)
    pd = max(64, A.next_power_of_2(dim))
    cpu = A.QJL(dim, device="cpu", seed=3).halves(pd)
    for got, want in zip(q.halves(pd), cpu):
        assert got.is_contiguous() and torch.equal(got.cpu(), want)
