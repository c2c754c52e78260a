"""The pipelined fp8 GEMM where M, K or N do not fill its tiles: fewer than 256 rows, k-tiles of 64
and pairs of them that K ends within (K % 16 == 0), single k-tiles, narrow N, both B layouts,
operands whose rows continue past K with NaN bytes, against the fp64 product."""

from __future__ import annotations

import pytest
import torch

import _pk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N", [
    (1, 16, 16), (16, 64, 32), (17, 80, 48), (255, 128, 128), (256, 144, 272), (257, 192, 256),
    (300, 208, 144), (64, 1040, 512), (511, 2000, 1008), (2050, 1104, 4112)])
@pytest.mark.parametrize("layout", [0, 1])
def test_against_fp64(cuda, M, K, N, layout):
    g = torch.Generator(device=cuda).manual_seed(M * 7 + K + N)

    def rows(r, c, pad):  # r x c e4m3 values in rows of c + pad bytes, NaN (0x7f) past c
        buf = torch.full((r, c + pad), 0x7F, dtype=torch.uint8, device=cuda)
        buf[:, :c] = torch.randn(r, c, generator=g, device=cuda).to(torch.float8_e4m3fn).view(torch.uint8)
        return buf.view(torch.float8_e4m3fn)[:, :c]

    a = rows(M, K, 64)
    b = rows(K, N, 16) if layout == 0 else rows(N, K, 48).t()
    ref = 0.5 * (a.double() @ b.double())
    # the fp8 MFMA's adder keeps about 2^-15 of the largest sum it adds; 1e-4 as the other
    # fp8 tests hold it to
    y = _pk.fp8_gemm(a, b, 0.5, torch.float32)
    assert torch.isfinite(y).all() and (y - ref).norm() <= 1e-4 * ref.norm()
    for dt in (torch.float16, torch.bfloat16):
        assert torch.equal(_pk.fp8_gemm(a, b, 0.5, dt), y.to(dt))
