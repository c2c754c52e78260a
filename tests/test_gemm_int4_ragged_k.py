"""int4_gemm where K is not a multiple of 64 or 128: the large-tile kernel's K tail (32 rows of its
last k-tile) and its use below 64 rows, on widths of whole words only, against the fp64 product."""

from __future__ import annotations

import pytest
import torch

import _pk
import gemm_int4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [32, 96, 160, 1056, 4160, 4128])
@pytest.mark.parametrize("M,N", [(5, 64), (16, 1032), (63, 520), (64, 264), (200, 4104), (300, 512)])
def test_against_fp64(cuda, M, K, N):
    g = torch.Generator(device=cuda).manual_seed(M + K + N)
    # rows continue past K with NaN, which must not be read into the sums
    wide = torch.full((M, K + 64), float("nan"), device=cuda, dtype=torch.float16)
    wide[:, :K] = torch.randn(M, K, generator=g, device=cuda).half()
    a = wide[:, :K]
    codes = torch.randint(-8, 8, (K, N), generator=g, device=cuda, dtype=torch.int8)
    wp = gemm_int4.pack_int4_n(codes)
    ref = 0.03 * (a.double() @ codes.double())
    y = gemm_int4.int4_gemm(a, wp, 0.03)
    # exact products of the codes, fp32 sums of K of them (1.4e-5 is seen)
    assert torch.isfinite(y).all() and (y - ref).norm() <= 6e-5 * ref.norm()
    assert torch.equal(y, gemm_int4.int4_gemm(a, wp, 0.03))
