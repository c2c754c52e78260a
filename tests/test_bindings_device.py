"""Every binding that hands tensor addresses to a kernel refuses tensors that are not on the
GPU (a host address given to a kernel would fault the device instead of failing the call).
Checked without a GPU: the refusal comes before any library call."""

from __future__ import annotations

import pytest
import torch

import _pk

f16, i32, u8 = torch.float16, torch.int32, torch.uint8


def _z(*shape, dtype=torch.float32):
    return torch.zeros(*shape, dtype=dtype)


CASES = [
    ("w4a16_gemm", lambda: _pk.w4a16_gemm(_z(1, 256, dtype=f16), _z(256, 32, dtype=i32), None, 0,
                                          1.0, f16)),
    ("w4a16_gemm_strips", lambda: _pk.w4a16_gemm_strips(_z(1, 256, dtype=f16), _z(256, 32, dtype=i32),
                                                        None, 0, 1.0, f16)),
    ("w4a16_gemm_partials", lambda: _pk.w4a16_gemm_partials(_z(1, 256, dtype=f16),
                                                            _z(256, 32, dtype=i32), None, 0, 2)),
    ("w4a16_prep_activations", lambda: _pk.w4a16_prep_activations(_z(1, 256), None, 1.0)),
    ("splitk_reduce", lambda: _pk.splitk_reduce(_z(2, 1, 8), 1.0, _z(1, 8))),
    ("fp8_gemm", lambda: _pk.fp8_gemm(_z(16, 16, dtype=u8), _z(16, 16, dtype=u8), 1.0, torch.float32)),
    ("gemm_dense", lambda: _pk.gemm_dense(_z(16, 16, dtype=f16), _z(16, 16, dtype=f16),
                                          torch.float32, 1)),
    ("absmax", lambda: _pk.absmax(_z(8))),
    ("cast_e4m3", lambda: _pk.cast_e4m3(_z(8), 1.0)),
    ("quantize_int4", lambda: _pk.quantize_int4(_z(8), 1.0)),
    ("pack_int4", lambda: _pk.pack_int4(_z(2, 8, dtype=torch.int8))),
    ("unpack_int4", lambda: _pk.unpack_int4(_z(2, 4, dtype=u8))),
    ("quantize_group", lambda: _pk.quantize_group(_z(128, 8), 4, 128, half_math=False,
                                                  want_qweight=True, want_scales=True,
                                                  want_fake=False)),
    ("gptq_block", lambda: _pk.gptq_block(_z(8, 8), _z(8, 8), _z(8, 8), 0, 8, 4, 0)),
    ("flash_decode", lambda: _pk.flash_decode(_z(1, 1, 64, dtype=f16), _z(1, 1, 256, 64, dtype=f16),
                                              _z(1, 1, 256, 64, dtype=f16), 128, 0.125)),
]


@pytest.mark.parametrize("name,call", CASES, ids=[c[0] for c in CASES])
def test_host_tensors_are_refused(name, call):
    with pytest.raises(ValueError, match=f"{name}: every tensor must be on one GPU"):
        call()


ROW_FORMS = {
    "second half of one row": lambda: _z(1, 512)[:, 256:], "odd pitch, one row": lambda: _z(1, 257)[:, :256],
    "misaligned": lambda: _z(513)[1:].view(2, 256), "misaligned, one row": lambda: _z(257)[1:].view(1, 256),
    "expanded": lambda: _z(256).expand(3, 256), "columns": lambda: _z(256, 3).t(),
    "overlapping": lambda: _z(600).as_strided((3, 256), (4, 1)), "no rows": lambda: _z(0, 256),
}


@pytest.mark.parametrize("form", ROW_FORMS)
def test_rows_for_the_kernels(form):
    """Whatever form activations come in, the rows handed to a kernel have unit inner stride,
    16-byte alignment and a pitch of at least their length -- also where torch calls the tensor
    contiguous as it is (any base; one row of any pitch)."""
    base = ROW_FORMS[form]()
    x = torch.arange(base.numel(), dtype=torch.float32).view(base.shape)
    if base.stride(0) >= base.shape[1] or base.shape[0] == 1:
        base.copy_(x)
    rows = _pk._rows_ok(base)
    assert rows.stride(1) == 1 and rows.stride(0) >= 256 and rows.stride(0) % 4 == 0
    assert rows.data_ptr() % 16 == 0 and torch.equal(rows, base)


@pytest.mark.parametrize("q,v", [((1, 4, 1, 64), (2, 4, 256, 64)), ((2, 3, 1, 64), (2, 4, 256, 64)),
                                 ((2, 8, 1, 64), (2, 4, 256, 64)), ((2, 4, 1, 32), (2, 4, 256, 64)),
                                 ((2, 4, 1, 64), (2, 4, 128, 64)), ((2, 4, 1, 64), (1, 4, 256, 64)),
                                 ((2, 4, 1, 64), (2, 4, 256, 32)), ((2, 4, 0, 64), (2, 4, 256, 64)),
                                 ((2, 4, 32), (2, 4, 256, 64)), ((2, 4, 1, 1, 64), (2, 4, 256, 64)),
                                 ((2, 4), (2, 4, 256, 64)), ((2, 4, 1, 64), (4, 256, 64))])
def test_decode_shapes_are_checked(monkeypatch, q, v):
    """q and v that do not fit k's (B, H, N, D) are refused before any library call: the kernel
    would read past their ends, or answer for other heads than q's."""
    monkeypatch.setattr(_pk, "_gpu_args", lambda *a: None)
    monkeypatch.setattr(_pk, "stream_of", lambda t: pytest.fail("past the checks"))
    with pytest.raises(ValueError, match="flash_decode: q"):
        _pk.flash_decode(_z(*q, dtype=f16), _z(2, 4, 256, 64, dtype=f16), _z(*v, dtype=f16), 128, 0.125)


PITCHES = {  # (rows, columns, strides) and whether the kernel can read it in place
    "expanded row": (5, 16, (0, 1), False), "expanded column": (5, 16, (1, 0), False),
    "overlapping rows": (5, 16, (8, 1), False), "columns": (5, 16, (1, 5), False),
    "contiguous": (5, 16, (16, 1), True), "wider rows": (5, 16, (24, 1), True),
    "one row": (1, 16, (3, 1), True), "one expanded row": (1, 16, (0, 1), True),
    "one column": (5, 1, (3, 7), True), "one expanded column": (5, 1, (0, 1), False),
}


@pytest.mark.parametrize("call,form", [("quantize_group", f) for f in PITCHES]
                         + [("pack_int4", f) for f in PITCHES if PITCHES[f][1] % 2 == 0])
def test_pitch_handed_to_the_kernel(monkeypatch, call, form):
    """The row pitch a kernel is told is the tensor's own, or the tensor is copied: a pitch
    below the row length rounded up to it would send the reads past the end."""
    rows, cols, strides, in_place = PITCHES[form]
    dt = torch.int8 if call == "pack_int4" else torch.float32
    t = torch.zeros(200, dtype=dt).as_strided((rows, cols), strides)
    seen = []

    class Lib:
        def pk_quantize_group(self, w, dtype, K, N, ld, *rest):
            seen.append((w, K, N, ld))
            return 0

        def pk_pack_int4(self, q, K, N, ld, *rest):
            seen.append((q, K, N, ld))
            return 0

    monkeypatch.setattr(_pk, "lib", Lib)
    monkeypatch.setattr(_pk, "_gpu_args", lambda *a: None)
    monkeypatch.setattr(_pk, "stream_of", lambda t: 0)
    if call == "pack_int4":
        _pk.pack_int4(t)
    else:
        _pk.quantize_group(t, 4, None, half_math=False, want_qweight=False, want_scales=False, want_fake=True)
    (address, K, N, ld), = seen
    assert (K, N) == (rows, cols) and (address == t.data_ptr()) == in_place
    assert ld == (t.stride(0) if in_place and rows > 1 else cols)


@pytest.mark.parametrize("rows", [1, 9, 64])
def test_rows_far_apart(monkeypatch, rows):
    """Rows that span 2 GiB or more, as the kernels on the row layout take them, are packed for the
    strip kernels, whose offsets have 32 bits."""
    seen = []

    class Calls:
        def pk_w4a16_gemm_strips_rows(self, a, lda, *rest):
            seen.append(lda)
            return 0

        pk_w4a16_gemm_strips = pk_w4a16_gemm_strips_rows

    monkeypatch.setattr(_pk, "_calls", Calls())
    monkeypatch.setattr(_pk, "_gpu_args", lambda *a: None)
    monkeypatch.setattr(_pk, "stream_of", lambda t: 0)
    weights = torch.empty(256, 32, dtype=i32, device="meta")
    for pitch in ((1 << 30) // rows // 8 * 8 - 8, (1 << 30) // rows // 8 * 8 + 8):
        a = torch.empty(rows * pitch, dtype=f16, device="meta").view(rows, pitch)[:, :256]
        _pk.w4a16_gemm_strips(a, weights, None, 0, 1.0, f16, rows=rows > 8)
        assert rows * seen[-1] < 1 << 30 and seen[-1] == (pitch if rows * pitch < 1 << 30 else 256)
