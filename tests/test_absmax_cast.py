"""The fp8 quantization's absmax (one launch, answered through a mailbox) and its cast by a
maximum in device memory, at the edges of their 16-byte chunks and workgroups: the CPU oracle's
bytes and scale, on offset views, with NaN and infinities, and zero refused as before."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

import _pk
import gemm_fp8
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,off", [(1, 0), (7, 1), (16, 0), (4096, 0), (4097, 3), (65551, 8), (3000001, 0)])
def test_bytes_and_scale(cuda, dtype, n, off):
    g = torch.Generator().manual_seed(n)
    x = (torch.randn(n + off, generator=g) * 3).to(dtype)[off:]
    x[n // 2] = -11.0 if n < 10 else 77.0
    for at in {0, n // 3, n - 1}:  # the maximum in the first, a middle and the last element
        y = x.clone()
        y[at] = -200.0
        yg = torch.empty(n + off, dtype=dtype, device=cuda)[off:]
        yg.copy_(y)
        y8, scale = gemm_fp8.quantize(yg)
        assert scale == 448.0 / 200.0
        want = oracle.e4m3_from_f32((y.float() * np.float32(scale)).to(dtype).float().numpy())
        assert np.array_equal(y8.view(torch.uint8).cpu().numpy(), want)
        assert _pk.absmax(yg).item() == 200.0


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_non_finite_and_zero(cuda, dtype):
    x = torch.linspace(-4, 4, 1000).to(dtype).to(cuda)
    x[123] = float("inf")
    x8, scale = gemm_fp8.quantize(x)
    got = x8.float().cpu()
    assert scale == 0.0 and math.isnan(got[123]) and got.nan_to_num().abs().max() == 0
    x[700] = float("nan")
    x8, scale = gemm_fp8.quantize(x)
    assert math.isnan(scale) and bool(x8.float().isnan().all())
    assert math.isnan(_pk.absmax(x).item())
    with pytest.raises(ZeroDivisionError):
        gemm_fp8.quantize(torch.zeros_like(x))
    assert gemm_fp8.quantize(torch.ones_like(x))[1] == 448.0  # counters are clean again


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_every_16_bit_value(cuda, dtype):
    bits = torch.arange(65536, dtype=torch.int32).to(torch.int16)
    x = bits.view(dtype)
    for scale in (1.0, 0.37, 2.0 ** -9):
        out = _pk.cast_e4m3(x.to(cuda), scale).view(torch.uint8).cpu().numpy()
        with np.errstate(invalid="ignore", over="ignore"):
            want = oracle.e4m3_from_f32((x.float() * np.float32(scale)).to(dtype).float().numpy())
        nan = x.isnan().numpy()  # torch drops a NaN's sign where it rounds to bf16
        assert np.array_equal(out[~nan], want[~nan]) and (out[nan] & 0x7f == 0x7f).all()


def test_refused_under_capture(cuda):
    """The scale goes to the host, so a capture cannot hold the call; the capture goes on."""
    x = torch.full((64,), 3.0, device=cuda)
    gemm_fp8.quantize(x)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        with pytest.raises(RuntimeError, match="captured"):
            gemm_fp8.quantize(x)
        y = _pk.cast_e4m3(x, 2.0)
    for v in (1.0, 5.0):
        x.fill_(v)
        graph.replay()
        torch.cuda.synchronize()
        assert bool((y.float() == 2 * v).all())
