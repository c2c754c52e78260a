"""The strip layout's batch kernel (pk_w4a16_gemm_strips_rows): every number of strips per workgroup
(with a last workgroup that has fewer), 128-row blocks that do not divide among the waves, 16-row
activation blocks with a remainder, every kind of group, bias and output dtype, strided
activations; and QuantLinear's rule for it."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import _pk
import gemm_int4
import oracle
import quant_linear

SHAPES = [(128, 16), (384, 48), (1152, 4096 + 16), (1024, 8192 + 48), (2176, 16400)]


def _layer(K, N, group, seed):
    g = torch.Generator().manual_seed(seed)
    w = (torch.randn(K, N, generator=g) * 0.02).half()
    codes, _, s16 = oracle.rtn_group_codes(w.numpy(), 4, group or K)
    return codes, s16 if group else None


def _want(a, codes, s16, group, scale, bias):
    """fp64 product of the same codes and scales."""
    w = torch.from_numpy(codes).double()
    if s16 is not None:
        w = w * torch.from_numpy(s16.astype(np.float64)).repeat_interleave(group, 0)
    y = scale * (a.double() @ w.to(a.device))
    return y if bias is None else y + bias.double()


@pytest.mark.gpu
@pytest.mark.parametrize("K,N", SHAPES)
@pytest.mark.parametrize("group", [128, 64, 32, 0, -1])
def test_against_fp64(cuda, K, N, group):
    group = K if group < 0 else group  # -1: one group over all of K
    codes, s16 = _layer(K, N, group, K + N)
    qw = torch.from_numpy(oracle.pack_int4_n(codes)).to(cuda).view(torch.int32)
    qs = _pk.strip_weights(qw)
    ss = None if s16 is None else _pk.strip_scales(torch.from_numpy(s16).to(cuda))
    g = torch.Generator(device=cuda).manual_seed(N)
    bias = torch.randn(N, generator=g, device=cuda)
    for M in (5, 16, 17, 32, 33, 64):
        a = torch.randn(M, K + 8, generator=g, device=cuda).half()[:, :K]
        want = _want(a, codes, s16, group, 0.5, bias)
        y = _pk.w4a16_gemm_strips(a, qs, ss, group, 0.5, torch.float32, bias=bias, rows=True)
        # exact products, fp32 sums of K of them in blocks of 128: K / 128 + 128 roundings of
        # 2^-24 on sums of the size of the result bound the 2-norm error far below 2e-5
        assert (y - want).norm() <= 2e-5 * want.norm(), (M, group)
        assert torch.equal(y, _pk.w4a16_gemm_strips(a, qs, ss, group, 0.5, torch.float32, bias=bias, rows=True))
        for dt in (torch.float16, torch.bfloat16):  # one rounding of the same fp32 sums
            z = _pk.w4a16_gemm_strips(a, qs, ss, group, 0.5, dt, bias=bias, rows=True)
            assert torch.equal(z, y.to(dt))


@pytest.mark.gpu
def test_prepared_call_and_limits(cuda):
    codes, s16 = _layer(512, 4352, 128, 1)
    qw = torch.from_numpy(oracle.pack_int4_n(codes)).to(cuda).view(torch.int32)
    qs, ss = _pk.strip_weights(qw), _pk.strip_scales(torch.from_numpy(s16).to(cuda))
    call = _pk.PreparedStrips(qs, ss, 128, 1.0, torch.float16)
    assert call.rows_from == _pk.strip_rows_from(512, 4352, 128)
    for M in (6, 9, 64):
        a = torch.randn(M, 512, device=cuda).half()
        assert torch.equal(call(a), _pk.w4a16_gemm_strips(a, qs, ss, 128, 1.0, torch.float16, rows=True))
    for M in (0, 65):
        with pytest.raises(_pk.PicoKernelsError):
            call(torch.zeros(M, 512, device=cuda, dtype=torch.float16))
    with pytest.raises(_pk.PicoKernelsError):
        _pk.w4a16_gemm_strips(torch.zeros(4, 512, device=cuda, dtype=torch.float16), qs, ss, 128, 1.0,
                              torch.float16, rows=True)


@pytest.mark.gpu
@pytest.mark.parametrize("scheme", ["group", "per_input"])
@pytest.mark.parametrize("out_f", [1024, 4112])
def test_quant_linear_batches(cuda, scheme, out_f):
    """QuantLinear agrees with itself without the strip copy at every row count around the rule's
    ends, for fp16 and bf16 inputs and a 3-D input."""
    lin = torch.nn.Linear(1280, out_f, device=cuda, dtype=torch.float16)
    q = quant_linear.QuantLinear.from_linear(lin, 128, None if scheme == "group" else "rtn")
    assert q.decode and q._on_strips(9) and q._on_strips(33) and not q._on_strips(65)
    for M in (1, 4, 5, 8, 9, 16, 33, 64, 65):
        for dt in (torch.float16, torch.bfloat16):
            x = torch.randn(M, 1280, device=cuda).to(dt)
            y = q(x)
            ref = x.double() @ q.dequantized_weight().double().t() + q.bias.double()
            assert (y.double() - ref).norm() <= (1e-3 if dt == torch.float16 else 6e-3) * ref.norm()
            if M == 16:
                assert torch.equal(q(x.view(2, 8, -1)).view(M, -1), y)


@pytest.mark.gpu
@pytest.mark.parametrize("out_f", [1024, 17424])
def test_quant_linear_batch_forms(cuda, out_f):
    """Decode rows and batches in forms other than contiguous, aligned rows: a misaligned base, a
    row pitch that is a multiple of 16 bytes or not, the second half of wider rows, transposed
    and expanded rows; each gives the contiguous copy's bits."""
    lin = torch.nn.Linear(256, out_f, device=cuda, dtype=torch.float16)
    q = quant_linear.QuantLinear.from_linear(lin, 128)
    rows = [M for M in (5, 9, 16, 32) if M > q.decode_rows and q._on_strips(M)]
    assert len(rows) >= 2
    for M in [1, 2, q.decode_rows] + rows:
        flat = torch.randn(M * 272 + 1, device=cuda).half()
        forms = (flat[1:M * 256 + 1].view(M, 256), flat[:M * 264].view(M, 264)[:, :256],
                 flat[:M * 264].view(M, 264)[:, 1:257], flat[:M * 257].view(M, 257)[:, :256],
                 flat[:M * 256].view(256, M).t(), flat[:256].expand(M, 256),
                 torch.randn(M, 512, device=cuda).half()[:, 256:])
        for x in forms:
            assert torch.equal(q(x), q(x.clone(memory_format=torch.contiguous_format)))
            xb = x.bfloat16() if x.stride(0) else x[:1].bfloat16().expand(M, 256)
            assert torch.equal(q(xb), q(xb.clone(memory_format=torch.contiguous_format)))
        x = forms[0].view(1, M, 256)
        assert torch.equal(q(x)[0], q(forms[0].clone()))


# (K, N, group (0: one scale per input), rows, whether the strip copy serves them), on both sides of
# the rule's lines; the calls kept off the strip copy took up to 2.1 times as long on it.
RULE = [
    (8064, 9216, 128, 64, False), (8064, 9216, 128, 28, True),      # packed-B GEMM in 7 slices
    (7040, 5120, 0, 35, False), (7040, 5120, 0, 32, True),
    (13952, 6144, 128, 33, True), (9856, 12032, 128, 64, True),     # one slice
    (3712, 11520, 0, 54, False), (3712, 11520, 128, 54, True),
    (4096, 14352, 0, 48, False), (4096, 14352, 128, 48, True),      # register-dequant kernel
    (13824, 8208, 0, 33, False), (6144, 8208, 0, 33, False), (2048, 12928, 128, 33, False),
    (3072, 8864, 128, 41, False), (14336, 3408, 0, 47, False), (10240, 3984, 0, 34, False),
    (8192, 3696, 128, 38, False), (9216, 3248, 128, 33, True),
    (13312, 1920, 128, 31, False), (8192, 1536, 128, 11, False),    # few strips of a long K
    (8192, 1536, 128, 24, False), (4096, 1536, 128, 24, True), (4096, 512, 0, 40, False),
    (6144, 8960, 128, 26, False), (6144, 8960, 128, 10, True),      # 140 workgroups
    (7168, 17408, 128, 9, False), (7168, 17408, 128, 32, False),    # 272 workgroups
    (5120, 28672, 128, 16, True), (5120, 28672, 128, 17, False), (5120, 28672, 128, 8, False),
    (768, 27136, 0, 9, False), (10368, 19200, 0, 6, False), (10368, 19200, 0, 32, False),
    (4096, 14336, 128, 32, True), (4096, 14336, 128, 33, False), (4096, 4096, 128, 64, True),
    (4096, 4096, 128, 65, False), (14336, 4096, 128, 16, True), (14336, 4096, 128, 17, False),
]


@pytest.mark.parametrize("K,N,group,rows,strips", RULE)
def test_rule(K, N, group, rows, strips):
    layer = quant_linear.QuantLinear(K, N, bias=False, group_size=group or 128, device="meta",
                                     scheme="group" if group else "per_input")
    assert layer.decode and layer._on_strips(rows) is strips


@pytest.mark.parametrize("K,N,group,rows", [(4096, 4096, 128, 9), (4096, 4112, 128, 5), (2048, 4112, 128, 6),
                                            (4096, 16384, 128, 5), (4096, 16400, 128, 9),
                                            (10496, 6144, 32, 9), (11264, 10752, 64, 9),
                                            (11264, 10752, 256, 5), (11264, 10752, 0, 5)])
def test_rows_from(K, N, group, rows):
    """Where the decode kernel hands over to the batch kernel: at 5..8 rows the latter takes up to
    1.34 times as long with groups shorter than a block."""
    assert _pk.strip_rows_from(K, N, group) == rows
