"""Large fp32 products on the bf16 matrix cores (csrc/gemm_split.hip): each value as three bf16
parts, six of the nine products of parts. Against float64 over tile edges, remainders, layouts,
strides and epilogues; against the fp32 matrix cores, which the same call takes under HIP graph
capture; and with values the parts do not hold (infinities, NaN, 2^36 and more), where the fp32
kernels that stand behind the call take over.

The bar: the sum of the dropped part products is at most 2^-23 of sum |a||b| per element and of
random sign (2^-27 rms), the fp32 sums add about 2^-24 per 32 k in a random walk: 4e-7 for normal
values at K = 4096, and 5e-7 is asserted (the fp32 matrix cores reach 1.2e-6 there)."""
import pytest

import gonngpu as G

pytestmark = pytest.mark.gpu
VARIANTS = [(False, False), (False, True), (True, False), (True, True)]


def _stored(t, trans):
    return t.transpose(-1, -2).contiguous() if trans else t.contiguous()


def _pitched(t, pad):
    """The same matrix with rows `pad` elements further apart."""
    import torch

    if not pad:
        return t
    wide = torch.full((t.shape[0], t.shape[1] + pad), float("nan"), device=t.device, dtype=t.dtype)
    wide[:, : t.shape[1]] = t
    return wide[:, : t.shape[1]]


def _rel(c, ref):
    return float((c.double() - ref).norm() / ref.norm())


def _captured(fn):
    import torch

    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        fn()
    g.replay()
    torch.cuda.synchronize()


# (M, N, K), both operands packed: one round of 128 x 128 tiles; ragged rows, columns and K, split over K; two rounds of
# 256 x 128 tiles; a K-tile count that its slices do not divide; K = 128 (four K-tiles).
SHAPES = [(2048, 2048, 1024), (777, 1234, 4099), (4096, 4096, 512), (1100, 1100, 4000), (8192, 8192, 128),
          (2561, 2500, 2030)]
# B split by the product kernel: 256-row and 128-row tiles, one launch and slices of K, ragged N, K of
# whole K-tiles, with a remainder of whole vectors (NT's loads) and an odd one (NN; NT packs it)
RAW_SHAPES = [(512, 11008, 1024), (512, 4096, 4096), (200, 1000, 2000), (160, 4100, 4132), (256, 5001, 2052),
              (500, 3000, 1533)]


@pytest.mark.parametrize("tA,tB", VARIANTS)
@pytest.mark.parametrize("M,N,K", SHAPES + RAW_SHAPES)
def test_split_against_f64_and_the_fp32_cores(dev, M, N, K, tA, tB):
    import torch

    g = torch.Generator(device=dev).manual_seed(M + 2 * N + 3 * K)
    A = torch.randn((M, K), generator=g, device=dev)
    B = torch.randn((K, N), generator=g, device=dev)
    a, b = _stored(A, tA), _stored(B, tB)
    c = torch.full((M, N), float("nan"), device=dev)
    print("split", M, N, K, tA, tB, flush=True)
    G.gemm(a, b, c, transA=tA, transB=tB)
    ref = A.double() @ B.double()
    assert _rel(c, ref) <= 5e-7
    again = torch.empty_like(c)
    G.gemm(a, b, again, transA=tA, transB=tB)
    assert torch.equal(c, again)
    c32 = torch.full((M, N), float("nan"), device=dev)
    _captured(lambda: G.gemm(a, b, c32, transA=tA, transB=tB))
    assert not torch.equal(c, c32), "the call took the fp32 matrix cores"
    assert _rel(c, ref) <= _rel(c32, ref)


@pytest.mark.parametrize("pads", [(0, 0, 0), (4, 8, 4), (1, 3, 5)])
@pytest.mark.parametrize("M,N,K", [(2048, 2048, 1024), (777, 1234, 4099), (512, 11008, 1024), (512, 4096, 4096)])
def test_split_epilogue_and_pitches(dev, M, N, K, pads):
    """alpha, beta over a prior C, bias and GELU, with leading dimensions wider than the rows
    (aligned to 16 bytes or not): C's padding stays, in one launch and over K slices."""
    import torch

    g = torch.Generator(device=dev).manual_seed(M + K)
    A = torch.randn((M, K), generator=g, device=dev)
    B = torch.randn((K, N), generator=g, device=dev) * 0.02
    C0 = torch.randn((M, N), generator=g, device=dev)
    bias = torch.randn((N,), generator=g, device=dev)
    a, b, c = _pitched(A, pads[0]), _pitched(B, pads[1]), _pitched(C0.clone(), pads[2])
    print("split epilogue", M, N, K, pads, flush=True)
    G.gemm(a, b, c, alpha=0.5, beta=-1.5, bias=bias, act=G.ACT_GELU)
    x = 0.5 * (A.double() @ B.double()) - 1.5 * C0.double() + bias.double()
    ref = 0.5 * x * (1.0 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x**3)))
    assert _rel(c, ref) <= 1e-6
    if pads[2]:
        assert torch.isnan(c.as_strided((M, pads[2]), (N + pads[2], 1), N)).all()


def test_split_batched(dev):
    import torch

    g = torch.Generator(device=dev).manual_seed(5)
    bs, M, N, K = 3, 1300, 1500, 1000
    A = torch.randn((bs, M, K), generator=g, device=dev)
    B = torch.randn((bs, N, K), generator=g, device=dev)
    c = torch.full((bs, M, N), float("nan"), device=dev)
    G.gemm(A, B, c, transB=True, batch=bs, strideA=M * K, strideB=N * K, strideC=M * N)
    for i in range(bs):
        assert _rel(c[i], A[i].double() @ B[i].double().t().contiguous()) <= 5e-7


# M, N, K, batch, layout, elements between the batches' B, form: parts of several batches or of a single one, or of
# K; "raw": B split by the product kernel (test_split_plan.py checks that each case is cut so)
CUTS = [(512, 1024, 4096, 48, "nn", 0, "batch-raw"), (400, 4096, 4096, 6, "nt", 1, "batch"),
        (512, 1000, 100000, 2, "nt", 0, "single-raw"), (512, 1000, 100000, 2, "nt", 4, "single-raw"),
        (512, 11008, 4096, 2, "nt", 1, "single"), (500, 1000, 200004, 1, "nt", 0, "k-raw"),
        (500, 1000, 200001, 1, "nn", 0, "k-raw")]


@pytest.mark.parametrize("M,N,K,batch,layout,gap,form", CUTS)
def test_split_cut_into_parts(dev, M, N, K, batch, layout, gap, form):
    """A batch cut into launches of several batches or of one, with batch strides that keep the rows
    of a K-contiguous B on 16 bytes or not, and K cut into parts with a raw B."""
    import torch

    g = torch.Generator(device=dev).manual_seed(M + N + gap)
    A = torch.randn((batch, M, K), generator=g, device=dev)
    stride = N * K + gap
    flat = torch.randn((batch * stride,), generator=g, device=dev) * 0.05
    shape = (N, K) if layout == "nt" else (K, N)
    B = flat.as_strided((batch, *shape), (stride, shape[1], 1))
    C0 = torch.randn((batch, M, N), generator=g, device=dev)
    bias = torch.randn((N,), generator=g, device=dev)
    c = C0.clone()
    print("split cut", M, N, K, batch, layout, gap, flush=True)
    G.gemm(A, B, c, transB=layout == "nt", batch=batch, strideA=M * K, strideB=stride, strideC=M * N, alpha=0.5,
           beta=0.5 if form.startswith("k") else 0.0, bias=bias, act=G.ACT_RELU)
    for i in range(batch):
        b = B[i].double().t().contiguous() if layout == "nt" else B[i].double()
        ref = 0.5 * (A[i].double() @ b) + bias.double()
        if form.startswith("k"):
            ref += 0.5 * C0[i].double()
        assert _rel(c[i], ref.clamp_min(0.0)) <= 1e-6  # 5e-7 of the product; the epilogue rounds twice more


def test_split_parts_of_k_beyond_the_kept_scratch(dev):
    """Operands whose packed form exceeds the scratch a stream keeps (512 MiB) run in parts of K,
    each adding to C: beta once, bias and activation once, at the end."""
    import torch

    g = torch.Generator(device=dev).manual_seed(6)
    M, N, K = 6200, 6100, 8000
    A = torch.randn((M, K), generator=g, device=dev)
    B = torch.randn((K, N), generator=g, device=dev) * 0.02
    C0 = torch.randn((M, N), generator=g, device=dev)
    bias = torch.randn((N,), generator=g, device=dev)
    c = C0.clone()
    before = G.memory_stats()[0]
    G.gemm(A, B, c, alpha=2.0, beta=0.5, bias=bias, act=G.ACT_RELU)
    torch.cuda.synchronize()
    assert G.memory_stats()[0] - before <= 512 << 20
    ref = (2.0 * (A.double() @ B.double()) + 0.5 * C0.double() + bias.double()).clamp_min(0.0)
    assert _rel(c, ref) <= 1e-6


@pytest.mark.parametrize("M,N,K", [(2048, 2048, 1024), (777, 1234, 4099), (2050, 2046, 1030), (512, 11008, 1024), (512, 4096, 4096)])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.4028234663852886e38, 2.0**36, -(2.0**40)])
@pytest.mark.parametrize("beta", [0.0, 0.5])
@pytest.mark.parametrize("side", ["a", "b"])
def test_split_values_it_does_not_hold(dev, M, N, K, value, side, beta):
    """One such value in either operand: the result is the fp32 matrix cores', with the
    infinities and NaN of the IEEE sums and nothing else touched."""
    import torch

    g = torch.Generator(device=dev).manual_seed(7)
    A = torch.randn((M, K), generator=g, device=dev)
    B = torch.randn((K, N), generator=g, device=dev)
    t = A if side == "a" else B
    t[t.shape[0] - 1, t.shape[1] - 1] = value
    if side == "a":
        B[K - 1, 5] = 0.0  # infinity times zero: NaN in that column only
    c = torch.full((M, N), 7.0, device=dev)
    G.gemm(A, B, c, beta=beta)
    c32 = torch.full((M, N), 7.0, device=dev)
    _captured(lambda: G.gemm(A, B, c32, beta=beta))
    ref = A.double() @ B.double() + 7.0 * beta
    fine = torch.isfinite(ref) & (ref.abs() < 3e38)
    rel = lambda x: float((x.double() - ref)[fine].norm() / ref[fine].norm())  # noqa: E731
    assert rel(c) <= max(1.5e-6, 1.5 * rel(c32))
    assert torch.equal(torch.isnan(c), torch.isnan(c32)) and torch.equal(torch.isinf(c), torch.isinf(c32))
    # the same operands without it, on the same scratch: the split again
    t[t.shape[0] - 1, t.shape[1] - 1] = 1.0
    G.gemm(A, B, c)
    assert _rel(c, A.double() @ B.double()) <= 5e-7


@pytest.mark.parametrize("tA,tB", VARIANTS)
@pytest.mark.parametrize("M,N,K", [(1100, 1100, 4000), (1100, 1100, 4004), (2048, 2048, 1044), (4100, 4100, 1024), (200, 1000, 2000),
                                   (1023, 1025, 4001), (3001, 2999, 517)])
def test_split_values_it_does_not_hold_on_every_fp32_form(dev, M, N, K, tA, tB):
    """The fp32 kernels behind a split product in its slices of K and in one launch, on both tiles,
    with a remainder of K % 32, aligned or not: alpha, beta, bias and activation once."""
    import torch

    g = torch.Generator(device=dev).manual_seed(M + K)
    A = torch.randn((M, K), generator=g, device=dev)
    B = torch.randn((K, N), generator=g, device=dev)
    A[3, K - 1] = float("inf")
    B[K - 1, 5] = float("nan")
    B[1, 7] = 2.0**37
    C0 = torch.randn((M, N), generator=g, device=dev)
    bias = torch.randn((N,), generator=g, device=dev)
    c = C0.clone()
    print("split fp32 form", M, N, K, tA, tB, flush=True)
    G.gemm(_stored(A, tA), _stored(B, tB), c, transA=tA, transB=tB, alpha=0.5, beta=2.0, bias=bias, act=G.ACT_RELU)
    ref = 0.5 * (A.double() @ B.double()) + 2.0 * C0.double() + bias.double()
    # the library's ReLU is fmaxf(x, 0): 0 for NaN
    ref = torch.where(torch.isnan(ref), torch.zeros_like(ref), ref.clamp_min(0.0))
    fine = torch.isfinite(ref)
    assert torch.equal(torch.isinf(c), torch.isinf(ref)) and not torch.isnan(c).any()
    col = torch.ones(N, dtype=torch.bool, device=dev)
    col[7] = False  # 2^37 times a normal value: its column apart
    for part in (fine & col, fine & ~col):
        assert _rel(c[part], ref[part]) <= 2e-6


@pytest.mark.parametrize("M,N,K", [(256, 4096, 4096), (200, 1000, 2000), (1100, 1100, 4000)])
def test_split_values_it_does_not_hold_cost_a_second_product_at_most(dev, M, N, K):
    """Few tiles and a long K: the fp32 kernels behind the split run in its slices of K, as the ordinary
    path would. (In one launch they took these calls from 42-128 us to 138-300, 3.6 to 4.9 times the same
    call with finite operands; now 1.1 to 2.3 times.)"""
    import torch

    g = torch.Generator(device=dev).manual_seed(M)
    A = torch.randn((M, K), generator=g, device=dev)
    B = torch.randn((K, N), generator=g, device=dev)
    c = torch.empty((M, N), device=dev)
    times = {}
    for kind in ("finite", "infinite"):
        if kind == "infinite":
            B[1, 1] = float("inf")
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        rounds = []
        for _ in range(5):
            torch.cuda._sleep(1000000)  # the calls queue up behind it
            start.record()
            for _ in range(10):
                G.gemm(A, B, c)
            end.record()
            torch.cuda.synchronize()
            rounds.append(start.elapsed_time(end))
        times[kind] = sorted(rounds)[2]
    assert times["infinite"] <= 3.0 * times["finite"], times


@pytest.mark.parametrize("scale", [2.0**-140, 2.0**-128, 2.0**-100, 2.0**-60, 2.0**35])
def test_split_range(dev, scale):
    """Rows of very small values (subnormal ones among them) and of the largest the split holds
    keep their relative precision: the parts hold every fp32 value below 2^36 exactly. A's rows
    alternate between that scale and 1; a subnormal has fewer bits, so its own rounding is in A
    before the product. B is of size 2^30 beside subnormals, so that no result is near fp32's own
    underflow and the middle and low parts of the subnormals count: without the middle ones a row
    at 2^-140 is 1.4e-3 off, without the low ones a row at 2^-128 2e-6."""
    import torch

    g = torch.Generator(device=dev).manual_seed(8)
    M, N, K = 2048, 2048, 1024
    A = torch.randn((M, K), generator=g, device=dev).clamp(-1.9, 1.9)
    A[::2] *= scale
    B = torch.randn((K, N), generator=g, device=dev)
    if scale < 2.0**-120:
        assert bool(((A != 0) & (A.abs() < 2.0**-126)).any())
        B *= 2.0**30
    c = torch.empty((M, N), device=dev)
    G.gemm(A, B, c)
    ref = A.double() @ B.double()
    err = (c.double() - ref).norm(dim=1)
    assert bool((err <= 5e-7 * ref.norm(dim=1)).all())


def test_split_integers_are_exact(dev):
    """Whole numbers whose products and sums fit 24 bits: every part product and sum is exact."""
    import torch

    g = torch.Generator(device=dev).manual_seed(9)
    A = torch.randint(-90, 91, (2048, 1024), generator=g, device=dev).float()
    B = torch.randint(-90, 91, (1024, 2048), generator=g, device=dev).float()
    c = torch.empty((2048, 2048), device=dev)
    G.gemm(A, B, c)
    assert torch.equal(c.double(), A.double() @ B.double())
