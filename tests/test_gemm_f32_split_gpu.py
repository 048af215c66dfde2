"""The f32 GEMM on the matrix cores (gemm_f32_split.h): three bf16 pieces per
value, six partial products, edges, persistent units, K splits and the f32
recomputation of what the pieces do not represent."""
import pytest

import nova_hip as nh

pytestmark = pytest.mark.gpu

LAYOUTS = ["NN", "NT", "TN", "TT"]


def _lay(t, kind):
    return t if kind == "N" else t.transpose(-1, -2).contiguous().transpose(-1, -2)


# (batch, M, N, K): one of each tile form, edges one off a tile, several
# units per workgroup, K below, at and past one step and ending in every
# remainder of a 16-byte chunk.
SHAPES = [(1, 64, 64, 32), (1, 63, 65, 33), (1, 1, 1, 1), (3, 65, 129, 31), (1, 130, 70, 66),
          (2, 257, 191, 35), (1, 72, 120, 0), (300, 97, 131, 71), (300, 97, 131, 127),  # 64 x 64, 2 x 3 x 300 units
          (1, 1500, 1700, 100), (1, 8192, 1538, 96), (1, 385, 9000, 130),
          (1, 2500, 4100, 61), (1, 4097, 510, 40)]


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_split_exact_on_integers(cuda, shape, layout):
    """Integers below 2^11 split into two pieces; products with small integers
    and their sums stay below 2^24, so every order gives the same sum."""
    import torch
    batch, M, N, K = shape
    g = torch.Generator().manual_seed(K)
    A = torch.randint(-1100, 1101, (batch, M, K), generator=g).float().to(cuda)
    B = torch.randint(-9, 10, (batch, K, N), generator=g).float().to(cuda)
    C = torch.full((batch, M, N), float("nan"), device=cuda)
    nh.gemm(_lay(A, layout[0]), _lay(B, layout[1]), C, f32_mfma=True)
    assert torch.equal(C.double(), torch.matmul(A.double(), B.double()))


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("flip", [False, True])
def test_split_represents_every_f32(cuda, layout, flip):
    """A times a permutation is A's columns, bit for bit: all 24 significand
    bits, from the smallest normal number to the largest, infinities and
    zeros of both signs; a NaN reaches its whole row and nothing else."""
    import torch
    g = torch.Generator().manual_seed(3)
    n = 200
    A = torch.randn(n, n, generator=g) * torch.exp2(torch.randint(-125, 126, (n, n), generator=g).float())
    A[0, :4] = torch.tensor([3.4028234663852886e38, -3.4e38, 1.1754943508222875e-38, 0.0])
    perm = torch.randperm(n, generator=g)
    P = torch.zeros(n, n)
    P[perm, torch.arange(n)] = 1.0
    a, b = (P.t().contiguous(), A.t().contiguous()) if flip else (A, P)
    C = nh.gemm(_lay(a.to(cuda), layout[0]), _lay(b.to(cuda), layout[1]), f32_mfma=True).cpu()
    assert torch.equal(C.t() if flip else C, A[:, perm])
    A[5, 7], A[9, 11] = float("inf"), float("nan")
    a, b = (P.t().contiguous(), A.t().contiguous()) if flip else (A, P)
    C = nh.gemm(_lay(a.to(cuda), layout[0]), _lay(b.to(cuda), layout[1]), f32_mfma=True).cpu()
    C = C.t() if flip else C
    ref = torch.matmul(A.double(), P.double()).float()  # inf * 0 is NaN across row 5 too
    assert torch.equal(torch.isnan(C), torch.isnan(ref))
    ok = ~torch.isnan(ref)
    assert torch.equal(C[ok], ref[ok])


@pytest.mark.parametrize("shape", [(300, 500, 384), (256, 1000, 5000), (200, 130, 50304),
                                   (9000, 16000, 6200), (190, 260, 1500), (700, 700, 2047)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("scale", [1e-25, 1.0, 1e12])
def test_split_error_bound(cuda, shape, scale):
    """Each output within (K / 2 + 8) 2^-24 of sum |a| |b|: the bound of an f32
    accumulation of pairs, whatever the magnitude of the operands."""
    import torch
    M, N, K = shape
    g = torch.Generator().manual_seed(M)
    A = (torch.randn(M, K, generator=g) * scale).to(cuda)
    B = (torch.randn(K, N, generator=g) * 1e-3).to(cuda)
    got = nh.gemm(A, B, f32_mfma=True).double()
    bound = (K / 2 + 8) * 2.0 ** -24 * torch.matmul(A.double().abs(), B.double().abs())
    assert bool(((got - torch.matmul(A.double(), B.double())).abs() <= bound).all())


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("flip", [False, True])
@pytest.mark.parametrize("K", [64, 1030])
def test_split_operands_of_any_magnitude(cuda, layout, flip, K):
    """Operands down to the smallest subnormal against ones that bring the
    products back (2^-118 to 2^-149 times 2^80 to 2^120, one magnitude per row),
    sums past what the split's own range holds (2^90), and products under the
    smallest subnormal.  Each output within the bound of an f32 accumulation of
    pairs, plus half the smallest subnormal for each product and each sum."""
    import torch
    g = torch.Generator().manual_seed(5)
    M, N = 150, 70
    rows = torch.tensor([-118, -122, -125, -126, -130, -140, -148, -20, 30, 0.0])
    A = torch.randn(M, K, generator=g).double() * torch.exp2(rows.double())[torch.arange(M) % 10, None]
    A[17], A[140] = 0.0, -0.0
    cols = torch.tensor([120, 100, 80, 60, -30, -129, 0.0])
    B = torch.randn(K, N, generator=g).double() * torch.exp2(cols.double())[None, torch.arange(N) % 7]
    A, B = A.float(), B.float()
    a, b = (B.t().contiguous(), A.t().contiguous()) if flip else (A, B)
    C = nh.gemm(_lay(a.to(cuda), layout[0]), _lay(b.to(cuda), layout[1]), f32_mfma=True).cpu()
    C = (C.t() if flip else C).double()
    ref, scale = A.double() @ B.double(), A.double().abs() @ B.double().abs()
    finite = scale < 3.4e38  # no sum of some of the products overflows
    bound = (K / 2 + 8) * 2.0 ** -24 * scale + K * 2.0 ** -149
    assert bool(((C - ref).abs() <= bound)[finite].all())
    assert not bool(torch.isfinite(C[ref.abs() > 3.5e38]).any())


@pytest.mark.parametrize("shape", [(300, 260, 40), (300, 260, 0), (2100, 1900, 64), (130, 140, 2100)],
                         ids=lambda s: "x".join(map(str, s)))
def test_split_zero_sums_are_positive(cuda, shape):
    """Sums of zeros of either sign and sums that cancel are +0 in every tile."""
    import torch
    M, N, K = shape
    A = torch.zeros(M, K, device=cuda)
    B = torch.ones(K, N, device=cuda)
    A[::3] = -0.0
    A[1::3, ::2], A[1::3, 1::2] = 1.5, -1.5
    A[1::3, K // 2 * 2:] = 0.0
    C = nh.gemm(A, B, f32_mfma=True)
    assert bool((C == 0).all()) and not bool(torch.signbit(C).any())


@pytest.mark.parametrize("K", [100, 4100])
def test_split_operands_inside_larger_tensors(cuda, K):
    """Rows with odd strides at odd offsets, infinities all around: nothing
    outside [M, K] and [K, N] reaches a result, and the padding of C stays."""
    import torch
    M, N = 131, 203
    g = torch.Generator().manual_seed(K)
    A = torch.randint(-50, 51, (M, K), generator=g).float()
    B = torch.randint(-9, 10, (K, N), generator=g).float()
    ref = (A.double() @ B.double()).float()
    for layout in LAYOUTS:

        def embed(t, kind):
            c = t if kind == "N" else t.t()
            big = torch.full((c.shape[0] + 3, c.shape[1] + 5), float("inf"), device=cuda)
            big[1:1 + c.shape[0], 3:3 + c.shape[1]] = c.to(cuda)
            v = big[1:1 + c.shape[0], 3:3 + c.shape[1]]
            return v if kind == "N" else v.t()

        big = torch.full((M, N + 3), 5.0, device=cuda)
        nh.gemm(embed(A, layout[0]), embed(B, layout[1]), big[:, 1:1 + N], f32_mfma=True)
        assert torch.equal(big[:, 1:1 + N].cpu(), ref), layout
        assert bool((big[:, 0] == 5.0).all()) and bool((big[:, 1 + N:] == 5.0).all())


def test_split_sums_of_one_large_and_many_small_terms(cuda):
    """Gradients of a 50304-class loss with respect to the head's input, rows
    of nearly equal small terms and one large one at a random place: the sum
    over rows is within twice what 8 sums of f32 fused multiply-adds in pairs
    give (1.5e-6); sums of 6288 terms on this kernel are at 3.7e-6."""
    import torch
    N, V, D = 4096, 50304, 128
    g = torch.Generator(device=cuda).manual_seed(0)
    flat = torch.randn(N, D, device=cuda, generator=g)
    w = torch.randn(D, V, device=cuda, generator=g) * 0.02
    p = torch.softmax(flat @ w, 1)
    p[torch.arange(N, device=cuda), torch.randint(0, V, (N,), device=cuda, generator=g)] -= 1.0
    dl = p / N
    got = nh.gemm(dl, w.t(), f32_mfma=True).double().sum(0)
    ref = torch.cat([dl[i:i + 1024].double() @ w.t().double() for i in range(0, N, 1024)]).sum(0)
    assert float((got - ref).norm() / ref.norm()) < 3e-6


@pytest.mark.parametrize("epi", [nh.EPI_BIAS, nh.EPI_BIAS_GELU, nh.EPI_GELU])
@pytest.mark.parametrize("shape", [(65, 67, 40), (300, 1001, 512), (8192, 384, 64), (100, 130, 4096)],
                         ids=lambda s: "x".join(map(str, s)))
def test_split_epilogues(cuda, shape, epi):
    """Bias and GELU on exact sums: within 2e-6 of the value's scale, the error
    of tanhf and a handful of f32 operations."""
    import torch
    M, N, K = shape
    g = torch.Generator().manual_seed(N)
    A = torch.randint(-8, 9, (M, K), generator=g).float().to(cuda) / 64
    B = torch.randint(-8, 9, (K, N), generator=g).float().to(cuda) / 16
    bias = torch.randn(N, generator=g).to(cuda)
    got = nh.gemm(A, B, bias=bias if epi != nh.EPI_GELU else None, epilogue=epi, f32_mfma=True).double()
    ref = A.double() @ B.double()
    if epi != nh.EPI_GELU:
        ref = ref + bias.double()
    if epi != nh.EPI_BIAS:
        ref = torch.nn.functional.gelu(ref, approximate="tanh")
    assert bool(((got - ref).abs() <= 2e-6 * (1 + ref.abs())).all())
