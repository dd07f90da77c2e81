"""The GEMV over a matrix of unit row stride (x * W with W row-major): equal bit
for bit to the same call with W k-contiguous, so in every summing order of the
row kernels (rows up to 8 KiB and beyond, one to four vectors), on ragged
columns and K, unaligned rows, both ways of splitting the work, batches,
alpha/beta and a strided vector."""
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


# by default most products of two to four vectors, and narrow i8 ones, take the
# skinny kernels: "0" keeps all on the GEMV
@pytest.mark.parametrize("skinny", ["1", "0"])
@pytest.mark.parametrize("dtype", ["f32", "bf16", "i8"])
# (vectors, k, n): one batch of chunks per slot and several, K ending inside a
# chunk, fewer columns than a lane's 16 bytes would leave whole, one group and
# enough groups to run whole, 256 lanes per row (K rows beyond 8 KiB)
@pytest.mark.parametrize("shape", [(1, 1024, 16), (1, 1025, 17), (1, 2048, 9000), (1, 4097, 65),
                                   (1, 9001, 33), (1, 16384, 129), (2, 2049, 40), (2, 8200, 100),
                                   (3, 1500, 130), (4, 2048, 2000), (4, 1031, 31),
                                   (1, 2064, 1100), (2, 2500, 4200)],
                         ids=lambda s: "x".join(map(str, s)))
def test_unit_row_stride_equals_k_contiguous(dev, monkeypatch, dtype, shape, skinny):
    monkeypatch.setenv("GEMMKIT_HIP_SKINNY", skinny)
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
    for alpha, beta in ((1, 0), (3, 2)):
        outs = []
        for x, rsa, csa, b, rsb, csb, bo in ((a0, kp, 1, w0, 1, kp, 0), (a, k, 1, w, n, 1, 0),
                                             (a, k, 1, off, n + 3, 1, 1), (at, 1, m, w, n, 1, 0)):
            c = torch.arange(m * n, device=dev).remainder(7).to(cdt)
            f = gk.gemm_i8_unchecked if dt == torch.int8 else gk.gemm_unchecked
            f(m, k, n, alpha, x, rsa, csa, b, rsb, csb, beta, c, n, 1, b_off=bo)
            outs.append(c)
        for c in outs[1:]:
            assert torch.equal(c.view(torch.uint8), outs[0].view(torch.uint8))
    if dt == torch.int8:
        want = a.view(m, k).double() @ w.double()
        assert torch.equal((outs[0] - 2 * torch.arange(m * n, device=dev).remainder(7)).double(),
                           3 * want.reshape(-1))


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_batch_of_column_matrices_equals_standalone(dev, dtype):
    dt, batch, m, k, n = DT[dtype], 5, 1, 4100, 75
    a, b = values(batch * m * k, dt, 3, dev), values(batch * k * n, dt, 4, dev)
    c = torch.zeros(batch * m * n, dtype=dt, device=dev)
    gk.gemm_batched_unchecked(batch, m, k, n, 1.0, a, k, 1, m * k, b, n, 1, k * n, 0.0, c, n, 1,
                              m * n)
    for z in range(batch):
        one = torch.zeros(m * n, dtype=dt, device=dev)
        gk.gemm_unchecked(m, k, n, 1.0, a, k, 1, b, n, 1, 0.0, one, n, 1, a_off=z * m * k,
                          b_off=z * k * n)
        assert torch.equal(c[z * m * n:(z + 1) * m * n], one)
