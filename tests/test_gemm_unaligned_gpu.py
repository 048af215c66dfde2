"""The 16-bit GEMM of rows at any 2-byte alignment (gemm_mfma.hip) with K past
what the small-K kernel takes.  Integer-valued operands: every sum is exact,
whatever its order, so f32 outputs are the 64-bit product bit for bit and
16-bit outputs its rounding."""
import pytest

import nova_hip as nh

pytestmark = pytest.mark.gpu

LAYOUTS = ["NN", "NT", "TN", "TT"]


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("shape", [(1, 65, 67, 577), (2, 63, 129, 641), (1, 1, 1, 1025), (1, 300, 201, 1001),
                                   (3, 1500, 1701, 515), (1, 2100, 2051, 1026), (1, 130, 70, 4099)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("offset", [(0, 0), (1, 3), (5, 2)])
def test_unaligned_exact(cuda, shape, layout, offset):
    """Odd sizes, odd row strides, slices starting at any element of a tensor
    filled with infinities around them, in both operand types."""
    import torch
    batch, M, N, K = shape
    g = torch.Generator().manual_seed(K)
    A = torch.randint(-4, 5, (batch, M, K), generator=g).to(cuda)
    B = torch.randint(-4, 5, (batch, K, N), generator=g).to(cuda)
    ref = torch.matmul(A.double(), B.double())
    for dt, out in ((torch.bfloat16, torch.float32), (torch.float16, torch.bfloat16)):

        def embed(t, kind, o):
            c = (t if kind == "N" else t.transpose(1, 2)).to(dt)
            big = torch.full((batch, c.shape[1] + 1, c.shape[2] + 7), float("inf"), device=cuda, dtype=dt)
            big[:, :c.shape[1], o:o + c.shape[2]] = c
            v = big[:, :c.shape[1], o:o + c.shape[2]]
            return v if kind == "N" else v.transpose(1, 2)

        big = torch.full((batch, M, N + 3), 5.0, device=cuda, dtype=out)
        nh.gemm(embed(A, layout[0], offset[0]), embed(B, layout[1], offset[1]), big[:, :, 1:1 + N])
        assert torch.equal(big[:, :, 1:1 + N], ref.float().to(out)), dt
        assert bool((big[:, :, 0] == 5.0).all()) and bool((big[:, :, 1 + N:] == 5.0).all())


@pytest.mark.parametrize("epi", [nh.EPI_BIAS, nh.EPI_BIAS_GELU, nh.EPI_GELU])
@pytest.mark.parametrize("out", ["f32", "bf16"])
def test_unaligned_epilogues(cuda, epi, out):
    """Bias and GELU on exact sums: the rounding of bf16, or in f32 2e-6 of the
    value's scale (tanhf and a handful of f32 operations)."""
    import torch
    M, N, K = 70, 131, 1001
    g = torch.Generator().manual_seed(2)
    A = torch.randint(-4, 5, (M, K), generator=g).to(cuda)
    B = torch.randint(-4, 5, (K, N), generator=g).to(cuda)
    bias = torch.randn(N, generator=g).to(cuda).to(torch.bfloat16)
    ref = (A.double() @ B.double()) / 64
    od = torch.float32 if out == "f32" else torch.bfloat16
    got = nh.gemm((A / 64).to(torch.bfloat16), B.to(torch.bfloat16),
                  bias=bias if epi != nh.EPI_GELU else None, epilogue=epi, out_dtype=od).double()
    if epi != nh.EPI_GELU:
        ref = ref + bias.double()
    if epi != nh.EPI_BIAS:
        ref = torch.nn.functional.gelu(ref, approximate="tanh")
    tol = 2e-6 * (1 + ref.abs()) if out == "f32" else 2.0 ** -8 * ref.abs() + 1e-6
    assert bool(((got - ref).abs() <= tol).all())


@pytest.mark.parametrize("M,N", [(3, 65), (130, 5), (1, 2)])
def test_unaligned_operand_slices_shorter_than_a_chunk(cuda, M, N):
    """Operands whose K stride is zero: the whole slice is one line of M (or N)
    elements, down to two bytes."""
    import torch
    K = 577
    g = torch.Generator().manual_seed(M)
    for dt in (torch.bfloat16, torch.float16):
        a = torch.randint(-4, 5, (M,), generator=g).to(cuda).to(dt)
        b = torch.randint(-4, 5, (N,), generator=g).to(cuda).to(dt)
        C = nh.gemm(a.as_strided((1, M, K), (0, 1, 0)), b.as_strided((1, K, N), (0, 0, 1)))
        assert torch.equal(C[0].double(), K * torch.outer(a.double(), b.double())), dt
