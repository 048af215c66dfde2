"""The exact f32 GEMM's 16x16-tile form on both sides of two tiles per CU (one
output per thread up to there, two from there on): every output equals the
k-ascending sum of separately rounded products bit for bit, at whole and
partial tiles and at K below, at and past a stage of 128.
"""
import numpy as np
import pytest

import nova_hip as nh

pytestmark = pytest.mark.gpu


def _sequential(a, b):
    acc = np.zeros(a.shape[:-1] + b.shape[-1:], np.float32)
    for k in range(a.shape[-1]):
        acc = acc + a[..., k, None] * b[..., k, None, :]
    return acc


@pytest.mark.parametrize("layout", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("shape", [
    (1, 500, 256, 128),   # 512 tiles: one output per thread on 256 CUs
    (1, 500, 260, 128),   # 544: two
    (1, 496, 284, 4), (1, 508, 300, 124), (1, 512, 272, 132), (1, 480, 288, 260),
    (3, 236, 188, 388),   # three batches of 180 tiles
], ids=str)
def test_exact_tiny_form_is_sequential(cuda, shape, layout):
    import torch
    batch, M, N, K = shape
    g = np.random.default_rng(M * 7 + K)
    a = g.uniform(-1, 1, (batch, M, K)).astype(np.float32)
    b = g.uniform(-1, 1, (batch, K, N)).astype(np.float32)
    A, B = torch.from_numpy(a).to(cuda), torch.from_numpy(b).to(cuda)
    if layout[0] == "T":
        A = A.transpose(1, 2).contiguous().transpose(1, 2)
    if layout[1] == "T":
        B = B.transpose(1, 2).contiguous().transpose(1, 2)
    got = nh.gemm(A, B).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), _sequential(a, b).view(np.uint32))
