"""Products of at most 64 rows (csrc/gemm_rows.hip): NT and NN, fp32 and fp16, against float64 of the
stored operands. Rows at the edges of the 16-row blocks; columns at the edges of every tile width
(48 with N = 11008, 32 or 64 elsewhere, one column more than a tile); K shorter than one round of the
waves, with a remainder inside a step and inside a substep, and long enough to be cut into slices;
padded leading dimensions; X of any alignment; outputs with a pitch.

The bar is 1e-5 relative Frobenius, the library's for sums in fp32 of exact products (fp16) or of
products rounded once (fp32): K <= 11008 sums of random sign err by about 2^-24 sqrt(K) / 2 = 3e-6."""
import pytest

import gonngpu as G

pytestmark = pytest.mark.gpu


def _rel(c, ref):
    return float((c.double() - ref).norm() / ref.norm())


def _operand(torch, g, dev, rows, cols, pitch, dtype, std=1.0):
    wide = torch.full((rows, pitch), float("nan"), dtype=dtype, device=dev)
    wide[:, :cols] = (torch.randn((rows, cols), generator=g, device=dev) * std).to(dtype)
    return wide[:, :cols]


# (M, N, K)
SHAPES = [(1, 1024, 256), (2, 256, 1024), (3, 5000, 800), (16, 3000, 2000), (16, 11008, 520), (17, 1024, 4096),
          (32, 4096, 1032), (33, 2048, 8192), (48, 528, 8200), (49, 256, 4104), (64, 1040, 2056), (5, 4104, 264)]


@pytest.mark.parametrize("layout", ["nt", "nn"])
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_rows(dev, M, N, K, half, layout):
    import torch

    g = torch.Generator(device=dev).manual_seed(M + 3 * N + 5 * K)
    dt = torch.float16 if half else torch.float32
    for pad in (0, 8):
        x = _operand(torch, g, dev, M, K, K + pad, dt)
        w = _operand(torch, g, dev, *((N, K, K + pad) if layout == "nt" else (K, N, N + pad)), dt, 0.05)
        bias = torch.randn((N,), generator=g, device=dev)
        ref = x.double() @ (w.t() if layout == "nt" else w).double().contiguous()
        c = torch.full((M, N + 3), float("nan"), device=dev)[:, :N]
        print("rows", layout, M, N, K, half, pad, flush=True)
        G.gemm(x, w, c, transB=layout == "nt", bias=bias, act=G.ACT_RELU)
        assert _rel(c, (ref + bias.double()).clamp_min(0.0)) <= 1e-5
        again = torch.empty((M, N), device=dev)
        G.gemm(x, w, again, transB=layout == "nt", bias=bias, act=G.ACT_RELU)
        assert torch.equal(again, c)
        c0 = torch.randn((M, N), generator=g, device=dev)
        y = c0.clone()
        G.gemm(x, w, y, transB=layout == "nt", alpha=-0.5, beta=2.0)
        assert _rel(y, -0.5 * ref + 2.0 * c0.double()) <= 1e-5


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 4096, 777), (4, 1026, 3001), (16, 3002, 515), (9, 1001, 2050), (7, 1028, 1999)])
def test_rows_any_alignment(dev, M, N, K, half):
    """X with rows of odd length (element-wise loads) and W with rows of 16, 8, 4 or no multiple of
    bytes (narrower tiles, or the other kernels), both layouts."""
    import torch

    g = torch.Generator(device=dev).manual_seed(M + N + K)
    dt = torch.float16 if half else torch.float32
    x = torch.randn((M, K), generator=g, device=dev).to(dt)
    for layout in ("nt", "nn"):
        w = (torch.randn((N, K) if layout == "nt" else (K, N), generator=g, device=dev) * 0.05).to(dt)
        c = torch.full((M, N), float("nan"), device=dev)
        print("rows unaligned", layout, M, N, K, half, flush=True)
        G.gemm(x, w, c, transB=layout == "nt")
        assert _rel(c, x.double() @ (w.t() if layout == "nt" else w).double().contiguous()) <= 1e-5


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("layout", ["nt", "nn"])
def test_rows_captured_without_slices(dev, half, layout):
    """16 x 1024 x 4096 is cut into slices of K; under graph capture it runs in one launch."""
    import torch

    g = torch.Generator(device=dev).manual_seed(3)
    dt = torch.float16 if half else torch.float32
    x = torch.randn((16, 4096), generator=g, device=dev).to(dt)
    w = (torch.randn((1024, 4096) if layout == "nt" else (4096, 1024), generator=g, device=dev) * 0.05).to(dt)
    ref = x.double() @ (w.t() if layout == "nt" else w).double().contiguous()
    c = torch.empty((16, 1024), device=dev)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        G.gemm(x, w, c, transB=layout == "nt")
    for _ in range(3):
        c.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert _rel(c, ref) <= 1e-5
    eager = torch.empty_like(c)
    G.gemm(x, w, eager, transB=layout == "nt")
    assert _rel(eager, ref) <= 1e-5


@pytest.mark.parametrize("layout", ["nt", "nn"])
def test_rows_infinity_stays_in_its_row_and_column(dev, layout):
    """Rows past M and columns past N are read from the last ones and not stored; the remainder
    of K past its end is zero in both operands: infinities spread no further than IEEE sums do."""
    import torch

    g = torch.Generator(device=dev).manual_seed(4)
    M, N, K = 5, 1001, 1037
    x = torch.randn((M, K), generator=g, device=dev)
    w = torch.randn((K, N), generator=g, device=dev)
    x[4, K - 1] = float("inf")
    w[K - 1, N - 1] = float("-inf")
    w[3, 7] = float("nan")
    pitch = 1040
    ws = torch.full((N, pitch) if layout == "nt" else (K, pitch), float("nan"), device=dev)
    if layout == "nt":
        ws[:, :K] = w.t()
        wv = ws[:, :K]
    else:
        ws[:, :N] = w
        wv = ws[:, :N]
    xs = torch.full((M, pitch), float("nan"), device=dev)
    xs[:, :K] = x
    c = torch.empty((M, N), device=dev)
    G.gemm(xs[:, :K], wv, c, transB=layout == "nt")
    ref = x.double() @ w.double()
    assert torch.equal(torch.isnan(c), torch.isnan(ref)) and torch.equal(torch.isinf(c), torch.isinf(ref))
    fine = torch.isfinite(ref)
    assert _rel(c[fine], ref[fine]) <= 1e-5


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 8192, 1), (2, 8200, 15), (3, 8256, 16), (4, 11008, 31), (1, 16384, 130), (4, 8192, 200), (2, 32776, 255),
                                   (3, 10008, 256), (2, 32768, 401), (1, 65536, 1024)])
def test_rows_wide_with_little_k(dev, M, N, K, half):
    """X W of 1-4 rows and few k (gemv_nn_kernel): fewer k than waves, whole rounds of eight and a rest, columns past the
    last workgroup's, padded leading dimensions; an infinity stays in its row and column."""
    import torch

    g = torch.Generator(device=dev).manual_seed(M + 3 * N + 5 * K)
    dt = torch.float16 if half else torch.float32
    bias = torch.randn((N,), generator=g, device=dev)
    c0 = torch.randn((M, N), generator=g, device=dev)
    for pad in (0, 8):
        x = _operand(torch, g, dev, M, K, K + pad, dt)
        w = _operand(torch, g, dev, K, N, N + pad, dt, 0.05)
        ref = x.double() @ w.double().contiguous()
        c = torch.full((M, N + 3), float("nan"), device=dev)[:, :N]
        print("wide", M, N, K, half, pad, flush=True)
        G.gemm(x, w, c, bias=bias, act=G.ACT_RELU)
        assert _rel(c, (ref + bias.double()).clamp_min(0.0)) <= 3e-7  # K <= 1024: chains of 64 and a tree of 16, 1.5e-7
        y = c0.clone()
        G.gemm(x, w, y, alpha=-0.5, beta=2.0)
        assert _rel(y, -0.5 * ref + 2.0 * c0.double()) <= 3e-7
    x[M - 1, K - 1] = float("inf")
    w[K - 1, N - 1] = float("nan")
    G.gemm(x, w, c)
    ref = x.double() @ w.double().contiguous()
    assert torch.equal(torch.isnan(c), torch.isnan(ref)) and torch.equal(torch.isinf(c), torch.isinf(ref))


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 4096, 256), (2, 65536, 264), (8, 16400, 520), (12, 5001, 400), (16, 8192, 504), (4, 11008, 1016), (1, 8199, 1024),
                                   (2, 16384, 2048), (3, 9000, 328)])
def test_rows_four_waves(dev, M, N, K, half):
    """X W^T on tiles of 16 columns with 4 waves (plan_rows): waves with no whole step, one, and several
    with a rest; a ragged last tile; padded leading dimensions."""
    import torch

    g = torch.Generator(device=dev).manual_seed(M + 3 * N + 5 * K)
    dt = torch.float16 if half else torch.float32
    bias = torch.randn((N,), generator=g, device=dev)
    for pad in (0, 8):
        x = _operand(torch, g, dev, M, K, K + pad, dt)
        w = _operand(torch, g, dev, N, K, K + pad, dt, 0.05)
        ref = x.double() @ w.t().double().contiguous()
        c = torch.full((M, N + 3), float("nan"), device=dev)[:, :N]
        print("four waves", M, N, K, half, pad, flush=True)
        G.gemm(x, w, c, transB=True, bias=bias, act=G.ACT_RELU)
        assert _rel(c, (ref + bias.double()).clamp_min(0.0)) <= 1e-6
    x[M - 1, K - 1] = float("inf")
    w[N - 1, 0] = float("nan")
    G.gemm(x, w, c, transB=True)
    ref = x.double() @ w.t().double().contiguous()
    assert torch.equal(torch.isnan(c), torch.isnan(ref)) and torch.equal(torch.isinf(c), torch.isinf(ref))


@pytest.mark.parametrize("layout,M,N,K", [("nn", 4, 11008, 4096), ("nn", 1, 16384, 8192), ("nn", 32, 11008, 8192), ("nn", 16, 5000, 8192),
                                          ("nn", 2, 11008, 2400)])
def test_rows_sum_k_in_short_chains(dev, layout, M, N, K):
    """fp32: an MFMA rounds its sum once per product; chains of c products are off by about 2.5e-8 sqrt(c / 2) of
    the result (the rms of a rounding, times the growth of the sum). Chains of at most K / 16 products, and
    a sixth for adding them: 3.3e-7 at K = 4096, as the tiled kernels' (2.9e-7). One chain for each of 4
    waves was 5.7e-7 off there."""
    import torch

    g = torch.Generator(device=dev).manual_seed(K)
    x, w = torch.randn((M, K), generator=g, device=dev), torch.randn((K, N), generator=g, device=dev)
    c = torch.empty((M, N), device=dev)
    G.gemm(x, w.t().contiguous() if layout == "nt" else w, c, transB=layout == "nt")
    assert _rel(c, x.double() @ w.double()) <= 7.0 / 6.0 * 2.5e-8 * (K / 32) ** 0.5
