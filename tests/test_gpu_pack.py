"""The pack of operands the kernels cannot read in place: whatever the strides,
alignment and batch step of an operand, the product equals the same call on a
k-contiguous, aligned copy bit for bit (float) and the int64 product (i8)."""
import pytest
import torch

import gemmkit_amd as gk

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "bf16": torch.bfloat16, "i8": torch.int8}


def values(n, dtype, seed, dev):
    g = torch.Generator().manual_seed(seed)
    if dtype == torch.int8:
        return torch.randint(-128, 128, (n,), generator=g, dtype=torch.int8).to(dev)
    return torch.randn(n, generator=g).to(dtype).to(dev)


def run(batch, m, k, n, a, ra, b, rb, dtype, dev):
    """C of (tensor, offset, rs, cs, batch stride) operands, row-major C."""
    c = torch.zeros(batch * m * n, dtype=torch.int32 if dtype == torch.int8 else dtype, device=dev)
    if dtype == torch.int8:
        gk.gemm_i8_unchecked(m, k, n, 1, a, ra[1], ra[2], b, rb[1], rb[2], 0, c, n, 1,
                             a_off=ra[0], b_off=rb[0])
    else:
        gk.gemm_batched_unchecked(batch, m, k, n, 1.0, a, ra[1], ra[2], ra[3], b, rb[1], rb[2],
                                  rb[3], 0.0, c, n, 1, m * n, a_off=ra[0], b_off=rb[0])
    return c


# rows x K around the packs' blocks (4, 8 or 16 rows x k per lane, 64..256 per
# workgroup), row lengths and steps that miss every alignment, and the copy's
# workgroups: 64 chunks of a few rows (below, at and above one such), 256 of many
# rows, and many short rows
SHAPES = [(20, 17, 19), (33, 64, 65), (64, 129, 257), (130, 255, 128), (257, 300, 77),
          (40, 9001, 35), (300, 24, 1000), (18, 1025, 20), (5000, 4103, 17)]


@pytest.mark.parametrize("dtype", ["f32", "bf16", "i8"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("kind", ["tr", "tr+odd", "copy+odd", "gap", "neg"])
def test_strided_operands_equal_canonical(dev, dtype, shape, kind):
    m, k, n = shape
    dt = DT[dtype]
    batch = 1 if dtype == "i8" else 3
    pad = 16 // dt.itemsize
    kp = (k + pad - 1) // pad * pad
    av, bv = values(batch * m * k, dt, 1, dev), values(batch * n * k, dt, 2, dev)
    # canonical copies: k-contiguous rows at an aligned step
    a0 = torch.zeros(batch, m, kp, dtype=dt, device=dev)
    b0 = torch.zeros(batch, n, kp, dtype=dt, device=dev)
    a0[:, :, :k] = av.view(batch, m, k)
    b0[:, :, :k] = bv.view(batch, n, k)
    want = run(batch, m, k, n, a0, (0, kp, 1, m * kp), b0, (0, 1, kp, n * kp), dt, dev)
    if dtype == "i8":
        exact = a0[0, :, :k].double() @ b0[0, :, :k].double().T
        assert torch.equal(want.view(m, n).double(), exact)

    def strided(x, rows):
        """(tensor, (offset, row stride, k stride, batch stride)) of x [batch, rows, k]."""
        if kind in ("tr", "tr+odd"):  # unit row stride
            off, step = (0, rows) if kind == "tr" else (1, rows + 3)
            size, rs, ks, bs = k * step, 1, step, k * step + (kind == "tr+odd")
        elif kind == "copy+odd":  # k-contiguous, nothing aligned
            off, step = 1, k + 1 + k % 2
            size, rs, ks, bs = rows * step, step, 1, rows * step + 1
        elif kind == "gap":  # neither index contiguous
            off, step = 0, 2 * k + 1
            size, rs, ks, bs = rows * step, step, 2, rows * step
        else:  # k backwards
            off, step = k - 1, k
            size, rs, ks, bs = rows * step, step, -1, rows * step
        buf = torch.zeros(off + batch * bs + size, dtype=dt, device=dev)
        z = torch.arange(batch, device=dev)[:, None, None]
        r = torch.arange(rows, device=dev)[None, :, None]
        p = torch.arange(k, device=dev)[None, None, :]
        buf[(off + z * bs + r * rs + p * ks).reshape(-1)] = x.reshape(-1)
        return buf, (off, rs, ks, bs)

    ab, (ao, ars, aks, abs_) = strided(av, m)
    bb, (bo, brs, bks, bbs) = strided(bv, n)
    got = run(batch, m, k, n, ab, (ao, ars, aks, abs_), bb, (bo, bks, brs, bbs), dt, dev)
    assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
