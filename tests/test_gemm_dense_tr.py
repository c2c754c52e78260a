"""The dense GEMM with transposing LDS reads at its edges: rows that do not fill a 64- or 128-row
tile, fewer k-tiles than pipeline stages and every remainder of them, split-K slices, strided A
and B, each output dtype; and the shapes it leaves to the other kernels."""

from __future__ import annotations

import pytest
import torch

import _pk

def _rel(y, ref):
    return ((y.double() - ref).norm() / ref.norm()).item()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N,split", [
    (64, 32, 256, 1), (65, 64, 256, 1), (128, 96, 512, 1), (200, 160, 256, 1), (256, 192, 256, 1),
    (300, 224, 768, 1), (2049, 352, 4096, 1), (130, 256, 512, 4), (257, 512, 256, 2),
    (256, 320, 264, 1), (48, 128, 256, 1), (2100, 64, 4096, 1), (1000, 512, 1024, 8)])
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


@pytest.mark.parametrize("M,N,K,split,rows", [
    (1024, 4096, 4096, 1, 64), (2048, 2048, 512, 1, 64), (2048, 4096, 4096, 1, 128),  # 256, 256 and 512 of 64
    (3072, 4096, 2048, 1, 128), (3072, 3072, 1088, 1, 128), (4096, 3072, 4096, 1, 128),  # three rounds for two
    (4096, 4096, 4096, 1, 128), (512, 512, 8192, 4, 64), (1024, 1024, 16384, 8, 128), (64, 65536 + 256, 32, 1, 64),
    (2048, 4096, 1024, 1, 0), (2048, 4096, 1088, 1, 128), (2048, 4096, 288, 1, 128), (2048, 3840, 512, 1, 128),
    (1024, 1024, 4096, 8, 0), (1024, 768, 4096, 8, 128), (3072, 3584, 256, 1, 0),  # short slices, whole rounds
    (48, 256, 64, 1, 0), (256, 264, 64, 1, 0)])
def test_tile_rows(M, N, K, split, rows):
    """64-row tiles only where they need no round more than 128-row ones (three rounds of them for
    two took 1.06 to 1.2 times as long), and another kernel for short slices of K on a chip full
    of tiles (up to 1.3 times as long)."""
    assert _pk.lib().pk_gemm_f16_tile_rows(M, N, K, split) == rows
    assert _pk.lib().pk_gemm_f16_tile_rows(M, N, K + 1, split) < 0
