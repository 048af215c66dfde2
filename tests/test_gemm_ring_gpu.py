"""The ring GEMM (gemm_ring.h): 16-byte aligned operand rows, any M, N, K.

Integer-valued operands make every product and partial sum exact in f32, so
the result is one value whatever the order of the sums: f32 outputs equal the
64-bit product bit for bit and 16-bit outputs its rounding.  The shapes sit
at the edges of each tile form and of the K steps and K groups: one short of,
at and one past a tile where the alignment allows, K below, at and past one
step, an odd number of steps for two groups, and fewer steps than groups."""
import pytest

import nova_hip as nh

pytestmark = pytest.mark.gpu

# (batch, M, N, K, out): the tile whose edges each is sized for.  (Which form runs
# it is the estimate's choice; FORMS below reaches them all.)
SHAPES = [
    (1, 1000, 3800, 136, "bf16"),    # 256 x 192, ragged last row and column
    (1, 1032, 11008, 328, "f32"),    # 256 x 192, one row group past a tile
    (3, 1536, 2200, 128, "bf16"),    # 256 x 128
    (1, 2048, 2056, 456, "f16"),     # 128 x 128 in two K groups, one chunk past N
    (2, 1000, 1112, 320, "f32"),     # 128 x 128, an odd number of K steps
    (1, 6000, 384, 200, "f32"),      # 64 x 128
    (7, 200, 264, 72, "bf16"),       # 64 x 64
    (1, 440, 4672, 72, "f32"),       # 64 x 64, K one chunk past a step
    (1, 16, 1000, 1544, "bf16"),     # 64 x 64 in two K groups, 25 steps
    (1, 8, 8, 8, "f32"),             # one tile, one chunk of K: the second group has none
    (1, 64, 64, 64, "f16"),
    (1, 72, 120, 0, "f32"),          # no K: zeros (A's rows 1 apart: the unaligned kernel's)
]

# One shape per form, by the smallest estimate: ragged in M, N and K.
FORMS = [
    (3, 200, 11008, 136, "bf16"),    # 256 x 192
    (7, 2048, 264, 136, "f32"),      # 256 x 128
    (1, 1500, 2056, 200, "f16"),     # 128 x 128 in two K groups
    (2, 200, 2056, 136, "f32"),      # 64 x 128, three stages
    (1, 200, 264, 136, "bf16"),      # 64 x 64, three stages
    (1, 200, 264, 200, "f32"),       # 64 x 64 in two K groups
    (20, 200, 264, 72, "f16"),       # 64 x 64, two stages
    (2, 200, 8200, 72, "bf16"),      # 64 x 128, two stages
    (2, 200, 8200, 128, "f32"),
    (2, 256, 8200, 8, "f32"),
]


def _case(cuda, shape, layout, dt, seed):
    import torch
    batch, M, N, K, out = shape
    g = torch.Generator().manual_seed(seed)
    td = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
    A = torch.randint(-4, 5, (batch, M, K), generator=g).to(cuda)
    B = torch.randint(-4, 5, (batch, K, N), generator=g).to(cuda)
    ref = torch.matmul(A.double(), B.double())
    A, B = A.to(td[dt]), B.to(td[dt])
    if layout[0] == "T":
        A = A.transpose(1, 2).contiguous().transpose(1, 2)
    if layout[1] == "T":
        B = B.transpose(1, 2).contiguous().transpose(1, 2)
    return A, B, ref, td[out]


@pytest.mark.parametrize("layout", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("shape", SHAPES + FORMS, ids=lambda s: "x".join(map(str, s)))
def test_ring_exact(cuda, shape, layout):
    import torch
    for dt in ("bf16", "f16"):
        A, B, ref, out = _case(cuda, shape, layout, dt, 7)
        C = torch.full(ref.shape, float("nan"), device=cuda, dtype=out)
        nh.gemm(A, B, C)
        assert torch.equal(C, ref.to(torch.float32).to(out)), dt


@pytest.mark.parametrize("pad", [1, 8])
@pytest.mark.parametrize("shape", [(1, 300, 400, 136, "f32"), (2, 1000, 1112, 320, "bf16")],
                         ids=lambda s: "x".join(map(str, s)))
def test_ring_output_rows_unaligned_or_padded(cuda, shape, pad):
    """Output rows that 16-byte stores cannot address (pad 1), or with room
    between them (pad 8): the outputs are exact and the room is untouched."""
    import torch
    A, B, ref, out = _case(cuda, shape, "NT", "bf16", 3)
    batch, M, N, _, _ = shape
    big = torch.full((batch, M, N + pad), 77.0, device=cuda, dtype=out)
    nh.gemm(A, B, big[:, :, :N])
    assert torch.equal(big[:, :, :N], ref.to(torch.float32).to(out))
    assert bool((big[:, :, N:] == 77.0).all())


@pytest.mark.parametrize("shape", [(1, 200, 264, 72), (1, 16, 1000, 1544), (1, 2048, 2056, 128),
                                   (1, 1000, 3800, 136)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("out", ["f32", "bf16"])
@pytest.mark.parametrize("epi", [nh.EPI_BIAS, nh.EPI_BIAS_GELU, nh.EPI_GELU])
def test_ring_epilogues(cuda, shape, out, epi):
    """Bias and GELU on exact sums: within the rounding of the output type
    (2^-8 of the value for bf16) or, in f32, within 2e-6 of the value's scale,
    the error of tanhf and a handful of f32 operations."""
    import torch
    A, B, ref, od = _case(cuda, shape + (out,), "NT", "bf16", 5)
    A, ref = A / 64, ref / 64  # exact: a power of two
    bias = torch.randn(shape[2], generator=torch.Generator().manual_seed(1)).to(cuda).to(torch.bfloat16)
    got = nh.gemm(A, B, bias=bias if epi != nh.EPI_GELU else None, epilogue=epi, out_dtype=od).double()
    if epi != nh.EPI_GELU:
        ref = ref + bias.double()
    if epi != nh.EPI_BIAS:
        ref = torch.nn.functional.gelu(ref, approximate="tanh")
    tol = 2e-6 * (1 + ref.abs()) if out == "f32" else 2.0 ** -8 * ref.abs() + 1e-6
    assert bool(((got - ref).abs() <= tol).all()), float(((got - ref).abs() - tol).max())


def test_ring_values_beyond_k_do_not_leak(cuda):
    """Operands that are slices of larger tensors holding infinities: nothing
    outside [M, K] and [K, N] reaches a result."""
    import torch
    M, N, K = 72, 136, 72
    for layout in ("NN", "NT", "TN", "TT"):
        A, B, ref, out = _case(cuda, (1, M, N, K, "f32"), layout, "bf16", 9)

        def embed(t):
            cont = t if t.stride(2) == 1 else t.transpose(1, 2)
            big = torch.full((1, cont.shape[1] + 8, cont.shape[2] + 8), float("inf"), device=cuda,
                             dtype=t.dtype)
            big[:, :cont.shape[1], :cont.shape[2]] = cont
            v = big[:, :cont.shape[1], :cont.shape[2]]
            return v if t.stride(2) == 1 else v.transpose(1, 2)

        C = nh.gemm(embed(A), embed(B))
        assert torch.equal(C, ref.to(torch.float32)), layout


def test_ring_without_k(cuda):
    """K = 0 with rows that are 16-byte aligned: the epilogue of zeros."""
    import torch
    buf = torch.full((72 * 8,), float("nan"), device=cuda, dtype=torch.bfloat16)
    bias = torch.randn(120, generator=torch.Generator().manual_seed(1)).to(cuda).to(torch.bfloat16)
    A = buf.as_strided((1, 72, 0), (576, 8, 1))
    B = torch.empty(1, 0, 120, device=cuda, dtype=torch.bfloat16)
    C = nh.gemm(A, B, bias=bias, epilogue=nh.EPI_BIAS)
    assert torch.equal(C[0], bias.float().expand(72, 120))
