"""The 128 x 256 tile on 16x16 matrix-core instructions: the same bits as the
256 x 256 tile (same instructions, same k order), for every output kind, on
ragged sides, K tails, padded and unaligned C, batches and fused epilogues."""
import pytest
import torch

import gemmkit_amd as gk

pytestmark = pytest.mark.gpu

TILES = ("256x256w8m16", "128x256w8m16")


def both(monkeypatch, call):
    out = []
    for t in TILES:
        monkeypatch.setenv("GEMMKIT_HIP_TILE", t)
        out.append(call())
    assert torch.equal(out[0].view(torch.uint8), out[1].view(torch.uint8))
    return out[0]


SHAPES = [(128, 192, 256, 0), (129, 136, 257, 3), (1, 640, 700, 0), (300, 1000, 512, 8),
          (511, 2048, 300, 1)]


@pytest.mark.parametrize("m,k,n,pad", SHAPES)
@pytest.mark.parametrize("batch", [1, 3])
def test_bf16(dev, monkeypatch, m, k, n, pad, batch):
    m = max(m, 20)  # (fewer rows take the vector route)
    g = torch.Generator().manual_seed(m + k)
    a = torch.randn(batch * m * k, generator=g).bfloat16().to(dev)
    b = torch.randn(batch * n * k, generator=g).bfloat16().to(dev)
    bias = torch.randn(n, generator=g).bfloat16().to(dev)
    ld = n + pad

    def f32out():
        c = torch.ones(batch * m * ld, device=dev)
        gk.gemm_batched_bf16_f32out(batch, 0.5, gk.MatRef(a, m, k, k, 1), m * k,
                                    gk.MatRef(b, k, n, 1, k), n * k, 2.0,
                                    gk.MatMut(c, m, n, ld, 1), m * ld)
        return c

    def fused():
        c = torch.ones(batch * m * ld, dtype=torch.bfloat16, device=dev)
        gk.gemm_batched_fused_unchecked(batch, m, k, n, 1.0, a, k, 1, m * k, b, 1, k, n * k, 0.0, c,
                                        ld, 1, m * ld, bias=bias, bias_dim=gk.BIAS_PER_COL,
                                        act=gk.Activation.Relu)
        return c
    got = both(monkeypatch, f32out).view(batch, m, ld)[:, :, :n].double()
    af, bf = a.double().view(batch, m, k), b.double().view(batch, n, k)
    want = 0.5 * (af @ bf.mT.contiguous()) + 2.0
    assert (got - want).norm() <= 1e-5 * want.norm()
    both(monkeypatch, fused)


@pytest.mark.parametrize("m,k,n,pad", SHAPES)
def test_i8(dev, monkeypatch, m, k, n, pad):
    m = max(m, 20)
    g = torch.Generator().manual_seed(m + k)
    a = torch.randint(-128, 128, (m * k,), generator=g, dtype=torch.int8).to(dev)
    b = torch.randint(-128, 128, (n * k,), generator=g, dtype=torch.int8).to(dev)
    ld = n + pad

    def i32():
        c = torch.ones(m * ld, dtype=torch.int32, device=dev)
        gk.gemm_i8_unchecked(m, k, n, 3, a, k, 1, b, 1, k, -2, c, ld, 1)
        return c
    got = both(monkeypatch, i32).view(m, ld)[:, :n].double()
    assert torch.equal(got, 3 * (a.double().view(m, k) @ b.double().view(n, k).T) - 2)
    for axis, count in ((0, m), (1, n)):
        scales = (torch.rand(count, generator=g) * 1e-3 + 1e-4).to(dev)
        bias = torch.randint(-65536, 65537, (count,), generator=g, dtype=torch.int32).to(dev)

        def q8():
            c = torch.zeros(m * ld, dtype=torch.int8, device=dev)
            gk.gemm_i8_requant_unchecked(m, k, n, a, k, 1, b, 1, k, 0.0, scales, 3, bias, c, ld, 1,
                                         axis=axis, relu=True)
            return c
        both(monkeypatch, q8)


def test_bf16_batch_equals_standalone(dev):
    """2048 x 256 x 2304 (144 half tiles) takes the half tile alone and the whole
    tile in a batch of three (one round instead of two)."""
    batch, m, k, n = 3, 2048, 256, 2304
    assert gk.debug_plan("bf16", "bf16", m, n, 2 * k)[0] == "128x256w8m16"
    g = torch.Generator().manual_seed(9)
    a = torch.randn(batch * m * k, generator=g).bfloat16().to(dev)
    b = torch.randn(batch * n * k, generator=g).bfloat16().to(dev)
    c = torch.zeros(batch * m * n, dtype=torch.bfloat16, device=dev)
    gk.gemm_batched_unchecked(batch, m, k, n, 1.0, a, k, 1, m * k, b, 1, k, n * k, 0.0, c, n, 1, m * n)
    for z in range(batch):
        one = torch.zeros(m * n, dtype=torch.bfloat16, device=dev)
        gk.gemm_unchecked(m, k, n, 1.0, a, k, 1, b, 1, k, 0.0, one, n, 1, a_off=z * m * k,
                          b_off=z * n * k)
        assert torch.equal(c[z * m * n:(z + 1) * m * n].view(torch.int16), one.view(torch.int16))
