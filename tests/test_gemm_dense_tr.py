"""The dense GEMM with transposing LDS reads at its edges: rows that do not fill a 64- or 128-row
tile, fewer k-tiles than pipeline stages and every remainder of them, split-K slices, strided A
and B, each output dtype; and the shapes it leaves to the other kernels."""

from __future__ import annotations

import pytest
import torch

import _pk

pytestmark = pytest.mark.gpu


def _rel(y, ref):
    return ((y.double() - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N,split", [
    (64, 32, 256, 1), (65, 64, 256, 1), (128, 96, 512, 1), (200, 160, 256, 1), (256, 192, 256, 1),
    (300, 224, 768, 1), (2049, 352, 4096, 1), (130, 256, 512, 4), (257, 512, 256, 2),
    (256, 320, 264, 1), (48, 128, 256, 1)])
def test_against_fp64(cuda, dtype, M, K, N, split):
    g = torch.Generator(device=cuda).manual_seed(M + K + N)
    a = torch.randn(M, K + 8, generator=g, device=cuda).to(dtype)[:, :K]
    b = torch.randn(K, N + 16, generator=g, device=cuda).to(dtype)[:, 8:N + 8]
    ref = a.double() @ b.double()
    y = _pk.gemm_dense(a, b, torch.float32, split)
    # exact products, fp32 sums of at most 512 of them: K roundings of 2^-24 at the very most
    assert _rel(y, ref) <= K * 2.0 ** -24
    assert torch.equal(y, _pk.gemm_dense(a, b, torch.float32, split))
    for dt in (torch.float16, torch.bfloat16):
        assert torch.equal(_pk.gemm_dense(a, b, dt, split), y.to(dt))
