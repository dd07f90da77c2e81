"""Skinny products over a matrix of unit row stride (a few rows times W with W
row-major): equal bit for bit to the same call with W k-contiguous, so in the
same summing order, on ragged columns and K, unaligned rows, empty K ranges,
strided vectors, either side as the vectors, batches and every epilogue."""
import pytest
import torch

import gemmkit_amd as gk

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "bf16": torch.bfloat16, "i8": torch.int8}


def values(n, dt, seed, dev):
    g = torch.Generator().manual_seed(seed)
    if dt == torch.int8:
        return torch.randint(-128, 128, (n,), generator=g, dtype=dt).to(dev)
    return torch.randn(n, generator=g).to(dt).to(dev)


@pytest.mark.parametrize("dtype", ["f32", "bf16", "i8"])
# (vectors, k, n): fewer rows than a lane group, one and many groups, K below a
# step per range, ending inside a chunk, on a step, on a batch of loads, and
# (i8) long enough for 8 and 16 ranges
@pytest.mark.parametrize("shape", [(2, 1024, 17), (3, 1025, 33), (5, 1100, 64), (8, 2048, 1000),
                                   (9, 1536, 129), (16, 1984, 40), (4, 8200, 75), (2, 6144, 300),
                                   (15, 1601, 2050), (2, 16384, 65), (4, 4095, 257), (1, 8300, 70),
                                   # vectors beyond the LDS: one row group, 8-, 24- and
                                   # 32-row ones, K ending inside a step and a chunk,
                                   # more than eight vectors
                                   # i8: both sides of the widths it takes from the
                                   # GEMV (512, 1024, 4096 columns)
                                   (1, 2528, 512), (1, 2528, 513), (1, 2048, 1024),
                                   (1, 1627, 1025), (2, 2528, 4096), (2, 7552, 4097),
                                   (1, 1030, 8), (2, 2048, 9),
                                   (8, 16385, 40), (5, 14008, 2049), (8, 8190, 4100),
                                   (7, 9300, 8200), (16, 4104, 2048), (12, 5503, 2100),
                                   # 24- and 32-row groups in one round
                                   (12, 6100, 4500), (16, 8200, 4500), (9, 8190, 6200)],
                         ids=lambda s: "x".join(map(str, s)))
def test_unit_row_stride_equals_k_contiguous(dev, dtype, shape):
    m, k, n = shape
    dt = DT[dtype]
    pad = 16 // dt.itemsize
    kp = (k + pad - 1) // pad * pad
    a, w = values(m * k, dt, 1, dev), values(k * n, dt, 2, dev).view(k, n)
    a0 = torch.zeros(m, kp, dtype=dt, device=dev)
    a0[:, :k] = a.view(m, k)
    w0 = torch.zeros(n, kp, dtype=dt, device=dev)
    w0[:, :k] = w.T
    off = 1 + torch.zeros(1 + k * (n + 3), dtype=dt, device=dev)  # odd base, padded rows
    off[1:].view(k, n + 3)[:, :n] = w
    at = a.view(m, k).T.contiguous()  # vectors side by side
    cdt = torch.int32 if dt == torch.int8 else dt
    f = gk.gemm_i8_unchecked if dt == torch.int8 else gk.gemm_unchecked
    for alpha, beta in ((1, 0), (3, 2)):
        c0 = torch.arange(m * n, device=dev).remainder(7).to(cdt)
        outs = []
        for x, rsa, csa, b, rsb, csb, bo in ((a0, kp, 1, w0, 1, kp, 0), (a, k, 1, w, n, 1, 0),
                                             (a, k, 1, off, n + 3, 1, 1), (at, 1, m, w, n, 1, 0)):
            c = c0.clone()
            f(m, k, n, alpha, x, rsa, csa, b, rsb, csb, beta, c, n, 1, b_off=bo)
            outs.append(c)
        # the transposed product: W^T (n x k, column-major) times the vectors
        c = c0.view(m, n).T.clone(memory_format=torch.contiguous_format).reshape(-1)
        f(n, k, m, alpha, w, 1, n, a, 1, k, beta, c, m, 1)
        outs.append(c.view(n, m).T.contiguous().reshape(-1))
        for c in outs[1:]:
            assert torch.equal(c.view(torch.uint8), outs[0].view(torch.uint8))
    want = 3 * (a.view(m, k).double() @ w.double()).reshape(-1) + 2 * c0.double()
    if dt == torch.int8:
        assert torch.equal(outs[0].double(), want)
    else:
        # against 64 bits: one rounding per k at most of the sums, and the result's
        terms = 3 * (a.view(m, k).abs().double() @ w.abs().double()).reshape(-1) + 2 * c0.double()
        last = 2.0 ** (-24 if dt == torch.float32 else -8) * want.abs()
        assert ((outs[0].double() - want).abs() <= (k + 4) * 2.0 ** -24 * terms + last).all()
        # (sums of many parts: far below that)
        err = (outs[0].double() - want).norm() / want.norm()
        assert err <= (1e-6 if dt == torch.float32 else 4e-3), err


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_batch_and_packed_equal_standalone(dev, dtype):
    dt, batch, m, k, n = DT[dtype], 5, 6, 2052, 75
    a, b = values(batch * m * k, dt, 3, dev), values(batch * k * n, dt, 4, dev)
    c = torch.zeros(batch * m * n, dtype=dt, device=dev)
    gk.gemm_batched_unchecked(batch, m, k, n, 1.0, a, k, 1, m * k, b, n, 1, k * n, 0.0, c, n, 1,
                              m * n)
    for z in range(batch):
        one, pk = (torch.zeros(m * n, dtype=dt, device=dev) for _ in range(2))
        gk.gemm_unchecked(m, k, n, 1.0, a, k, 1, b, n, 1, 0.0, one, n, 1, a_off=z * m * k,
                          b_off=z * k * n)
        assert torch.equal(c[z * m * n:(z + 1) * m * n], one)
        w = gk.prepack_rhs(gk.MatRef.from_row_major(b[z * k * n:(z + 1) * k * n], k, n))
        gk.gemm_packed_b(1.0, gk.MatRef.from_row_major(a[z * m * k:(z + 1) * m * k], m, k), w, 0.0,
                         gk.MatMut.from_col_major(pk, m, n))
        assert torch.equal(pk.view(n, m).T.reshape(-1), one)


def shared_batch(dev, dtype, batch, m, k, n, ws, strided=False):
    """A batch on one row-major matrix (zero batch stride), strided in C (and A:
    vectors side by side)."""
    dt = DT[dtype]
    a, b = values(batch * m * k, dt, 7, dev), values(k * n, dt, 8, dev)
    rsa, csa = (1, m) if strided else (k, 1)
    cbs = m * n + 5
    c = torch.zeros(batch * cbs, dtype=dt, device=dev)

    def call(ws=ws):
        gk.gemm_batched_unchecked(batch, m, k, n, 1.0, a, rsa, csa, m * k, b, n, 1, 0, 0.0, c, n,
                                  1, cbs, ws=ws)

    def check():
        for z in (0, 1, batch // 2, batch - 2, batch - 1):
            one = torch.zeros(m * n, dtype=dt, device=dev)
            gk.gemm_unchecked(m, k, n, 1.0, a, rsa, csa, b, n, 1, 0.0, one, n, 1, a_off=z * m * k)
            assert torch.equal(c[z * cbs:z * cbs + m * n], one), z
        assert (c.view(batch, cbs)[:, m * n:] == 0).all()

    return call, check, c


@pytest.mark.parametrize("dtype,batch,m,k,n", [("bf16", 1500, 8, 1100, 600),
                                               ("f32", 1000, 16, 1000, 520),
                                               ("bf16", 400, 8, 8200, 1000)])
def test_shared_matrix_bounded_workspace(dev, dtype, batch, m, k, n):
    """Each element's partial sums (16 f32 slabs of its output beyond the LDS, 8
    below) would take 205 to 266 MB at once: at most 128 MiB are used at a time."""
    ws = gk.Workspace()
    call, check, _ = shared_batch(dev, dtype, batch, m, k, n, ws)
    call()
    assert (16 if k > 8192 else 8) * batch * m * n * 4 > 200e6
    assert ws.bytes() <= 130 << 20
    check()


@pytest.mark.parametrize("dtype,batch,m,k,n,strided", [
    ("f32", 300, 1, 256, 500, False), ("f32", 150, 3, 500, 333, False),
    ("f32", 40, 9, 300, 400, False), ("bf16", 300, 1, 700, 500, False),
    ("bf16", 600, 7, 600, 260, False), ("bf16", 100, 13, 800, 400, False),
    ("bf16", 300, 2, 1600, 24, True), ("f32", 300, 7, 900, 33, True), ("f32", 300, 16, 256, 16, True)])
def test_shared_matrix_of_short_rows_is_packed(dev, dtype, batch, m, k, n, strided):
    """One pack serves the batch; under capture, where the workspace cannot grow, one
    vector's matrix is read in place: the same bits every way."""
    ws = gk.Workspace()
    call, check, c = shared_batch(dev, dtype, batch, m, k, n, ws, strided)
    call()
    pad = 16 // DT[dtype].itemsize
    assert ws.bytes() >= n * (k + pad - 1) // pad * pad * DT[dtype].itemsize
    # (partial sums, or packed vectors, would take more)
    assert ws.bytes() < 8 * batch * m * n * 4 + strided * batch * m * k or m == 1
    check()
    # captured: with the arena of that call, and one vector with none
    for arena in (ws, gk.Workspace()):
        if arena is not ws and m > 1:  # (more vectors have partial sums in the workspace)
            continue
        held = arena.bytes()
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        gk.set_synchronous(False)
        try:
            with torch.cuda.graph(graph):
                call(arena)
        finally:
            gk.set_synchronous(True)
        assert arena.bytes() == held
        for _ in range(3):
            c.zero_()
            graph.replay()
            torch.cuda.synchronize()
            check()


@pytest.mark.parametrize("m,k,n,layout", [(16, 8208, 4500, "col"), (2, 2048, 300, "row")])
def test_i8_routes_without_workspace(dev, m, k, n, layout):
    """i8 takes the faster of two routes only while its partial sums have room: under
    capture with an empty arena that cannot grow, the one without any."""
    a, w = values(m * k, torch.int8, 9, dev), values(k * n, torch.int8, 10, dev)
    rsb, csb = (1, k) if layout == "col" else (n, 1)
    c = torch.zeros(m * n, dtype=torch.int32, device=dev)

    def call(ws):
        gk.gemm_i8_unchecked(m, k, n, 1, a, k, 1, w, rsb, csb, 0, c, n, 1, ws=ws)

    call(gk.Workspace())
    want = (a.view(m, k).double() @ torch.as_strided(w, (k, n), (rsb, csb)).double()).reshape(-1)
    assert torch.equal(c.double(), want)
    ws = gk.Workspace()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    gk.set_synchronous(False)
    try:
        with torch.cuda.graph(graph):
            call(ws)
    finally:
        gk.set_synchronous(True)
    assert ws.bytes() == 0
    for _ in range(3):
        c.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c.double(), want)


def test_nonfinite_columns_stay_apart(dev):
    """A row of infinities or NaN reaches its own outputs only, past K neither."""
    m, k, n = 3, 1030, 50
    a, w = values(m * k, torch.bfloat16, 5, dev), values(k * n, torch.bfloat16, 6, dev)
    w = torch.cat([w, torch.full((64 * n,), float("nan"), dtype=w.dtype, device=dev)])
    w.view(-1, n)[:k, 7] = float("inf")
    w.view(-1, n)[:k, 49] = float("nan")
    c = torch.zeros(m, n, dtype=torch.bfloat16, device=dev)
    gk.gemm_unchecked(m, k, n, 1.0, a, k, 1, w, n, 1, 0.0, c, n, 1)
    bad = ~torch.isfinite(c)
    assert bad[:, [7, 49]].all() and bad.sum() == 2 * m
