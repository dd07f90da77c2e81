"""f32 products on the bf16 matrix cores (f32x.hip): f32 precision over layouts,
ragged sides and K tails, with and without the epilogue's terms, and over the
exponents; values the split cannot represent (infinities, NaN, the largest
magnitudes); and the same bits from either tile, so from a batch and from its
elements alone."""
import pytest
import torch

import gemmkit_amd as gk

pytestmark = pytest.mark.gpu


def randn(n, seed, dev):
    return torch.randn(n, generator=torch.Generator().manual_seed(seed)).to(dev)


def strided(x, layout, pad, dev):
    """(flat tensor, rs, cs) holding x row- or column-major with padded rows."""
    rows, cols = x.shape
    if layout == "row":
        buf = torch.zeros(rows, cols + pad, device=dev)
        buf[:, :cols] = x
        return buf.reshape(-1), cols + pad, 1
    buf = torch.zeros(cols, rows + pad, device=dev)
    buf[:, :rows] = x.T
    return buf.reshape(-1), 1, rows + pad


# few roundings (the blocks of 600 x 700 and 700 x 650, two rounds of the CUs) and
# many, 64 x 64 and 128 x 128 tiles, sides around 64 and 128, K around the 32-k
# stages and their alternation between the two groups
@pytest.mark.parametrize("m,k,n", [(600, 128, 700), (700, 333, 650), (1030, 129, 1000),
                                   (1300, 131, 900), (1000, 191, 1025), (2049, 160, 2047),
                                   (1500, 255, 1601), (4100, 128, 1100)])
@pytest.mark.parametrize("la,lb,pad", [("row", "row", 0), ("row", "col", 3), ("col", "col", 1),
                                       ("col", "row", 5)])
def test_precision(dev, m, k, n, la, lb, pad):
    a, b = randn(m * k, 1, dev).view(m, k), randn(k * n, 2, dev).view(k, n)
    ab, rsa, csa = strided(a, la, pad, dev)
    bb, rsb, csb = strided(b, lb, pad, dev)
    c0, bias = randn(m * n, 3, dev), randn(n, 4, dev)
    c = c0.clone()
    gk.gemm_unchecked(m, k, n, 0.75, ab, rsa, csa, bb, rsb, csb, -1.25, c, n, 1)
    want = 0.75 * (a.double() @ b.double()) - 1.25 * c0.double().view(m, n)
    # |error| <= roundings * u * sum |terms|: one per product of parts, 8 per 32 k
    # in each of two groups' sums, which take every other 32 k; the product left out
    # (2^-34) and the four of the epilogue
    u = 2.0 ** -24
    terms = 0.75 * (a.abs().double() @ b.abs().double()) + 1.25 * c0.abs().double().view(m, n)
    roundings = 6 * ((k + 31) // 32) + 6
    err = (c.view(m, n).double() - want).abs()
    assert (err <= roundings * u * terms).all()
    assert err.norm() <= 1e-6 * want.norm()
    f = torch.zeros(m * n, device=dev)
    gk.gemm_fused_unchecked(m, k, n, 1.0, ab, rsa, csa, bb, rsb, csb, 0.0, f, n, 1, bias=bias,
                            bias_dim=gk.BIAS_PER_COL, act=gk.Activation.Relu)
    p = torch.zeros(m * n, device=dev)
    gk.gemm_unchecked(m, k, n, 1.0, ab, rsa, csa, bb, rsb, csb, 0.0, p, n, 1)
    assert torch.equal(f.view(m, n), torch.relu(p.view(m, n) + bias))


# rows of 64 x 64 and 128 x 128 tiles, with (600 x 700) and without accumulators of
# their own for the small products
@pytest.mark.parametrize("m,k,n", [(600, 128, 700), (1030, 129, 1000), (2049, 160, 2047)])
def test_sums_of_one_term_are_correctly_rounded(dev, m, k, n):
    """One nonzero per row of A: every output is one product, which the f32
    instructions round correctly.  Here the product of parts left out is below
    2^-34 of it, and the small ones' sum, 2^-7 of it, loses up to 2^-30 of it in each
    of its last two additions (its others are far smaller): with the last, rounded
    one half an ulp and 2^-6 ulp; 2^-5 allowed."""
    b = randn(k * n, 31, dev).view(k, n)
    v = randn(m, 32, dev)
    # the largest m and l against h, alike in sign: 1 + 2^-8 - 2^-17
    worst = torch.tensor(0x3F807FC0, dtype=torch.int32).view(torch.float32).item()
    b[:, ::7], v[::5] = worst, worst
    at = torch.arange(m, device=dev) * 37 % k
    a = torch.zeros(m, k, device=dev)
    a[torch.arange(m, device=dev), at] = v
    c = torch.zeros(m * n, device=dev)
    gk.gemm_unchecked(m, k, n, 1.0, a.view(-1), k, 1, b.reshape(-1), n, 1, 0.0, c, n, 1)
    want = v.double()[:, None] * b[at].double()
    ulp = 2.0 ** (torch.frexp(want).exponent.double() - 24)
    err = ((c.view(m, n).double() - want) / ulp).abs()
    assert err.max() <= 0.5 + 2.0 ** -5, err.max()


@pytest.mark.parametrize("m,k,n", [(600, 150, 700), (1300, 131, 900)])
@pytest.mark.parametrize("rs,ks,packed", [
    (1, 1500, False), (2, 3100, False), (3, 4600, True), (0, 1, False), (700, 1, False),
    (1500, 2, True), (700, -1, True), (-700, 1, False), (-1, 1500, True), (5, 7600, True),
    (3000, 4, True), (0, 3, False)])
def test_operand_strides(dev, m, k, n, rs, ks, packed):
    """Any strides of either operand: the bits of the call on row-major copies.  An
    operand without a short stride, which every tile would read a cache line per
    element, is packed into the workspace; others are read in place."""
    def operand(rows, seed):
        lo = min(0, rs * (rows - 1)) + min(0, ks * (k - 1))
        hi = max(0, rs * (rows - 1)) + max(0, ks * (k - 1))
        buf = randn(hi - lo + 1, seed, dev)
        at = torch.arange(rows, device=dev)[:, None] * rs + torch.arange(k, device=dev)[None] * ks
        return buf, -lo, buf[at - lo]

    a, a0, ac = operand(m, 61)
    b, b0, bc = operand(n, 62)  # B^T
    want, got = torch.zeros(m * n, device=dev), torch.zeros(m * n, device=dev)
    gk.gemm_unchecked(m, k, n, 1.0, ac.reshape(-1), k, 1, bc.reshape(-1), 1, k, 0.0, want, n, 1)
    ws = gk.Workspace()
    gk.gemm_unchecked(m, k, n, 1.0, a, rs, ks, b, ks, rs, 0.0, got, n, 1, ws=ws, a_off=a0, b_off=b0)
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))
    assert (ws.bytes() > 0) == packed


def test_strided_operand_under_capture(dev):
    """The pack is only for speed: with a workspace that capture cannot grow the
    operand is read in place, and the replays give the same bits."""
    m, k, n = 600, 150, 700
    a, b = randn(2 * m * k, 71, dev), randn(k * n, 72, dev)
    want, got = torch.zeros(m * n, device=dev), torch.zeros(m * n, device=dev)
    gk.gemm_unchecked(m, k, n, 1.0, a, 2 * k, 2, b, n, 1, 0.0, want, n, 1)
    ws = gk.Workspace()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    gk.set_synchronous(False)
    try:
        with torch.cuda.graph(graph):
            gk.gemm_unchecked(m, k, n, 1.0, a, 2 * k, 2, b, n, 1, 0.0, got, n, 1, ws=ws)
    finally:
        gk.set_synchronous(True)
    assert ws.bytes() == 0
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int32), want.view(torch.int32))


def special(m, k, n, seed, dev):
    """A and B with an infinity, a NaN, the largest f32, subnormals and rows of
    magnitudes whose unscaled parts would leave the bf16 range."""
    a, b = randn(m * k, seed, dev).view(m, k), randn(k * n, seed + 1, dev).view(k, n)
    a[3, 5] = float("inf")
    a[m // 2, 7] = float("nan")
    a[m - 1, k - 1] = 3.4028234e38  # rounds to an infinite bf16
    b[:, n - 1] *= 1e-25
    a[20] *= 1e-36                   # parts below the smallest normal bf16
    a[21] *= 1e-40                   # subnormal
    a[70, : k // 2] = 0.0
    b[9, 2] = float("-inf")
    return a, b


@pytest.mark.parametrize("m,k,n", [(600, 150, 500), (1400, 130, 1300)])
def test_values_outside_the_split(dev, m, k, n):
    a, b = special(m, k, n, 11, dev)
    c = torch.zeros(m * n, device=dev)
    gk.gemm_unchecked(m, k, n, 1.0, a.view(-1), k, 1, b.reshape(-1), n, 1, 0.0, c, n, 1)
    got, want = c.view(m, n).double(), a.double() @ b.double()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    big = want.abs() > 3.4028234e38  # infinite in f32
    assert torch.equal(torch.isinf(got), big & ~torch.isnan(want))
    ok = ~torch.isnan(want) & ~big
    terms = (a.nan_to_num(0, 0, 0).abs().double() @ b.nan_to_num(0, 0, 0).abs().double())
    # one rounding per k at most (the f32 instructions), and the subnormal grid
    bound = (k + 4) * (2.0 ** -24 * terms + 2.0 ** -149)
    assert ((got - want).abs()[ok] <= bound[ok]).all()


@pytest.mark.parametrize("m,k,n", [(600, 150, 500), (1400, 131, 1300)])
def test_precision_over_the_exponents(dev, m, k, n):
    """Rows of A and columns of B from the smallest subnormals to 2^100: parts and
    products of parts below the smallest normal numbers, results over all of f32."""
    ea = torch.arange(m, device=dev) * 53 % 251 - 150
    eb = torch.arange(n, device=dev) * 67 % 251 - 150
    a = (randn(m * k, 41, dev).view(m, k).double() * 2.0 ** ea.double()[:, None]).float()
    b = (randn(k * n, 42, dev).view(k, n).double() * 2.0 ** eb.double()[None, :]).float()
    c = torch.zeros(m * n, device=dev)
    gk.gemm_unchecked(m, k, n, 1.0, a.view(-1), k, 1, b.reshape(-1), n, 1, 0.0, c, n, 1)
    got, want = c.view(m, n).double(), a.double() @ b.double()
    terms = a.abs().double() @ b.abs().double()
    ok = terms < 2.0 ** 127  # no partial sum overflows
    # one rounding per k at most, and the subnormal grid
    bound = (k + 4) * (2.0 ** -24 * terms + 2.0 ** -149)
    assert ((got - want).abs()[ok] <= bound[ok]).all()
    assert (terms[ok] < 2.0 ** -126).any() and (terms[ok] > 2.0 ** 110).any()


@pytest.mark.parametrize("m,k,n", [(600, 150, 500), (1400, 131, 1300)])
def test_tiny_values_take_no_second_pass(dev, m, k, n):
    """Elements far below the others change no output, so none may come from the f32
    instructions, whose order of sums is another."""
    a, b = randn(m * k, 51, dev).view(m, k), randn(k * n, 52, dev).view(k, n)
    tiny = torch.tensor([1e-31, 1e-36, -1e-38, 1e-41, -1e-45], device=dev)
    out = []
    for scale in (0.0, 1.0):
        x, y = a.clone().view(-1), b.clone().view(-1)
        for t in (x, y):
            at = torch.arange(0, t.numel(), 997, device=dev)
            t[at] = scale * tiny[at % 5]
        c = torch.zeros(m * n, device=dev)
        gk.gemm_unchecked(m, k, n, 1.0, x, k, 1, y, n, 1, 0.0, c, n, 1)
        out.append(c)
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("specials", [False, True])
@pytest.mark.parametrize("batch,m,k,n", [(8, 1000, 128, 1000), (9, 600, 150, 500)])
def test_batch_equals_standalone(dev, batch, m, k, n, specials):
    """8 x (1000 x 128 x 1000) fills the CUs with 128 x 128 tiles, one of them
    takes 64 x 64 ones."""
    a, b = randn(batch * m * k, 5, dev).view(batch, m, k), randn(batch * k * n, 6, dev).view(batch, k, n)
    if specials:
        a[1], b[1] = special(m, k, n, 21, dev)
        a[batch - 1, 130] *= 1e-37
    c = torch.zeros(batch * m * n, device=dev)
    gk.gemm_batched_unchecked(batch, m, k, n, 1.0, a.reshape(-1), k, 1, m * k, b.reshape(-1), n, 1,
                              k * n, 0.0, c, n, 1, m * n)
    for z in range(batch):
        one = torch.zeros(m * n, device=dev)
        gk.gemm_unchecked(m, k, n, 1.0, a[z].reshape(-1), k, 1, b[z].reshape(-1), n, 1, 0.0, one, n, 1)
        assert torch.equal(c.view(batch, -1)[z].view(torch.int32), one.view(torch.int32)), z
