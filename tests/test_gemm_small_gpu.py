"""The small-product kernel at the edges of its dispatch: each workgroup tile (16 x 16, 32 x 16,
32 x 32), each number of K-splitting waves, K at every kind of remainder of its steps and load
batches, in all four layouts, aligned or not. Operands are views into arrays filled with NaN, so a
value taken from outside them shows. Every element is held to |C - C64| <= (K + 2) 2^-24 sum |a||b|,
which bounds any order of K fp32 additions of products (exact for fp16 values, rounded once for
fp32)."""
import pytest

import gonngpu as G

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (17, 5, 15), (16, 16, 16), (33, 31, 17), (100, 130, 63), (256, 256, 33), (250, 250, 97),
          (256, 512, 48), (255, 511, 200), (200, 600, 100), (512, 512, 16), (511, 510, 32), (512, 512, 100),
          (500, 400, 257), (100, 132, 1000), (64, 64, 1519), (64, 64, 1536), (65, 70, 2047), (40, 24, 4097), (3, 2, 5001)]


def _view(rows, cols, pad, dtype, dev):
    import torch

    buf = torch.full((rows + 2, cols + pad), float("nan"), device=dev, dtype=dtype)
    v = buf[1 : 1 + rows, :cols]
    v.copy_(torch.randn((rows, cols), device=dev))
    return v


@pytest.mark.parametrize("pad", [0, 3, 8])
@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("shape", SHAPES)
def test_small_products(dev, shape, dtype, pad):
    import torch

    m, n, k = shape
    dt = torch.float16 if dtype == "f16" else torch.float32
    torch.manual_seed(m + 7 * n + 13 * k)
    for ta in (False, True):
        for tb in (False, True):
            a, b = _view(*((k, m) if ta else (m, k)), pad, dt, dev), _view(*((n, k) if tb else (k, n)), pad, dt, dev)
            c = torch.full((m, n), float("nan"), device=dev)
            print("small", shape, dtype, pad, ta, tb, flush=True)
            G.gemm(a, b, c, transA=ta, transB=tb)
            torch.cuda.synchronize()
            a64, b64 = (a.t() if ta else a).cpu().double(), (b.t() if tb else b).cpu().double()
            bound = (k + 2) * 2.0**-24 * (a64.abs() @ b64.abs())
            assert bool(((c.cpu().double() - a64 @ b64).abs() <= bound).all())


@pytest.mark.parametrize("m,n,k", [(512, 512, 512), (384, 500, 700), (100, 130, 1000), (1, 1000, 1000), (64, 128, 784),
                                   (255, 255, 2001), (256, 512, 784), (40, 1000, 600), (200, 24, 1250)])
def test_small_products_sum_k_in_short_chains(dev, m, n, k):
    """An fp32 MFMA rounds its sum once per product; a chain of c of them is off by about 2.5e-8
    sqrt(c / 2) of the result for normal operands (the rms of a rounding, times the growth of the
    partial sums). Chains of at most 64 products and the sum of the chains: 1.4e-7 to 1.6e-7; with
    K split over four waves of one chain each these products were 2.0e-7 to 2.9e-7 off."""
    import torch

    g = torch.Generator(device=dev).manual_seed(k)
    a, b = torch.randn((m, k), generator=g, device=dev), torch.randn((k, n), generator=g, device=dev)
    c = torch.empty((m, n), device=dev)
    G.gemm(a, b, c)
    ref = a.double() @ b.double()
    assert float((c.double() - ref).norm() / ref.norm()) <= 1.85e-7
