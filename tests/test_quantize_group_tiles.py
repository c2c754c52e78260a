"""pk_quantize_group at the edges of its tiles (256 or 64 columns, row sets of 8 or 128, groups
held in registers up to 128 rows), on rows it loads in whole chunks and element by element, and
at quotients on and beside a rounding tie: bit for bit the CPU oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import _pk
import oracle

pytestmark = pytest.mark.gpu


def _weights(K: int, N: int, dtype: torch.dtype, seed: int) -> torch.Tensor:
    """Normal weights; some rows a whole number and a half of the group's scale, exactly or one
    step of the dtype beside it."""
    g = torch.Generator().manual_seed(seed)
    w = (torch.randn(K, N, generator=g) * 0.02).to(dtype).float()
    n = min(N, 8)
    w[0, :n] = 0.07 * (1 + torch.arange(n))
    s = w[:, :n].abs().amax(0) / 7
    for i, k in enumerate(range(1, min(K, 9))):
        w[k, :n] = s * (i - 3.5)
    w = w.to(dtype)
    if K > 10:
        w[9, :n] = torch.nextafter(w[1, :n], torch.zeros((), dtype=dtype))
    return w


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("K,N,group,pad", [
    (128, 256, 128, 0), (1, 8, 128, 0), (130, 264, 128, 0), (96, 520, 32, 8), (129, 72, 0, 0),
    (700, 64, 0, 0), (1030, 136, 513, 0), (300, 264, 100, 5), (260, 40, 0, 3)])
def test_codes_scales_and_values(cuda, dtype, K, N, group, pad):
    w = _weights(K, N, dtype, K + N)
    wide = torch.zeros(K, N + pad, dtype=dtype, device=cuda)
    wide[:, pad:] = w.to(cuda)  # pad elements of offset and row stride
    qw, sc, fake = _pk.quantize_group(wide[:, pad:], 4, group, half_math=False, want_qweight=True,
                                      want_scales=True, want_fake=True, scale_dtype=torch.float32)
    codes, s32, _ = oracle.rtn_group_codes(w.float().numpy(), 4, group or K)
    assert np.array_equal(qw.cpu().numpy().view(np.uint8), oracle.pack_int4_n(codes))
    assert np.array_equal(sc.cpu().numpy().view(np.uint32), s32.view(np.uint32))
    want = torch.from_numpy(oracle.rtn_layer(w.float().numpy(), 4, group or None)).to(dtype)
    assert torch.equal(fake.cpu().view(torch.uint8), want.view(torch.uint8))


@pytest.mark.parametrize("N", [1, 7, 65])
@pytest.mark.parametrize("bits", [2, 8, 15])
def test_odd_widths_and_bits(cuda, N, bits):
    w = torch.randn(333, N, generator=torch.Generator().manual_seed(N))
    for group in (50, None):
        _, _, fake = _pk.quantize_group(w.to(cuda), bits, group, half_math=False, want_qweight=False,
                                        want_scales=False, want_fake=True)
        want = oracle.rtn_layer(w.numpy(), bits, group)
        assert np.array_equal(fake.cpu().numpy().view(np.uint32), want.view(np.uint32))


def test_extremes(cuda):
    """Zeros, values below the 1e-12 floor, the largest fp32 numbers, infinities and NaN, in
    columns of their own beside an ordinary one."""
    w = torch.randn(200, 8, generator=torch.Generator().manual_seed(3))
    w[:, 1] = 0.0
    w[:, 2] *= 1e-14
    w[:, 3] *= 1e-42
    w[:, 4] *= 3e37
    w[5, 5] = float("inf")
    w[6, 6] = float("nan")
    for group in (128, None):
        qw, _, fake = _pk.quantize_group(w.to(cuda), 4, group, half_math=False, want_qweight=True,
                                         want_scales=False, want_fake=True)
        with np.errstate(invalid="ignore"):
            want = oracle.rtn_layer(w.numpy(), 4, group)
        assert np.array_equal(fake.cpu().numpy(), want, equal_nan=True)
        g = group or 200
        for j in (5, 6):  # a NaN quotient is code 0
            bad = qw.cpu().numpy().view(np.uint32)[:, 0] >> (4 * j) & 15
            r0 = (5 if j == 5 else 6) // g * g
            assert bad[5 if j == 5 else 6] == 0 and (bad[r0:r0 + g] == 0).all()


@pytest.mark.parametrize("group", [64, None])
def test_expanded_and_overlapping_weights(cuda, group):
    """Weights whose rows share memory give the bits of their contiguous copy."""
    g = torch.Generator().manual_seed(4)
    row, col = torch.randn(72, generator=g).to(cuda), torch.randn(192, 1, generator=g).to(cuda)
    for w in (row.expand(192, 72), col.expand(192, 72), row[:1].expand(192, 72),
              torch.randn(4096, generator=g).to(cuda).as_strided((192, 72), (8, 1))):
        outs = [_pk.quantize_group(x, 4, group, half_math=False, want_qweight=True, want_scales=True,
                                   want_fake=True) for x in (w, w.contiguous())]
        assert all(torch.equal(a, b) for a, b in zip(*outs))
    codes = (row * 3).round().clamp(-8, 7).to(torch.int8).expand(192, 72)
    assert torch.equal(_pk.pack_int4(codes), _pk.pack_int4(codes.contiguous()))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("K,N,group,half_math", [(130, 264, 128, 0), (700, 72, 0, 0), (1030, 40, 513, 0),
                                                 (96, 13, 32, 0), (333, 8, 0, 1)])
def test_in_place(cuda, dtype, K, N, group, half_math):
    """Values written over the weights: those of a separate buffer, also in the rows on and beside a
    rounding tie, which are read a second time."""
    w = _weights(K, N, dtype, K + N).to(cuda)
    if half_math and dtype == torch.float32:
        half_math = 0
    want = _pk.quantize_group(w, 4, group, half_math=bool(half_math), want_qweight=False,
                              want_scales=False, want_fake=True)[2]
    dt = _pk.pk_dtype(dtype)
    rc = _pk.lib().pk_quantize_group(w.data_ptr(), dt, K, N, N, 4, group, half_math, None, None, dt,
                                     w.data_ptr(), dt, _pk.stream_of(w))
    assert rc == _pk.PK_OK and torch.equal(w, want)
