"""The activation cast that posts its range check's answer to the host (pk_w4a16_prep_checked):
the same fp16 values as the plain pass and the right answer at its unit edges (2048 k of a row),
with more units than workgroups, on rows it cannot load in 16-byte chunks, for the one element
that overflows wherever it stands, and from several threads and streams at once."""

from __future__ import annotations

import threading

import pytest
import torch

import _pk

pytestmark = pytest.mark.gpu


def _run(x, s=None, mul=1.0):
    with _pk.checked_activations(x, s, mul, "t") as y:
        pass
    return y


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,K,pad", [(1, 8, 0), (3, 2048, 0), (2, 2056, 3), (700, 4104, 8), (2100, 128, 0)])
def test_values_and_answer(cuda, dtype, M, K, pad):
    g = torch.Generator(device="cuda").manual_seed(M + K)
    wide = torch.randn(M, K + pad, generator=g, device=cuda).to(dtype)
    x = wide[:, pad:]
    s = torch.rand(K, generator=g, device=cuda) + 0.5
    for scale, mul in ((None, 1.0), (s, 0.25)):
        assert torch.equal(_run(x, scale, mul), _pk.w4a16_prep_activations(x, scale, mul))
    x[0, 0], x[-1, -1] = float("inf"), float("nan")  # not finite before the cast: no overflow
    _run(x)
    for m, k in ((0, K - 1), (M - 1, 0), (M // 2, K // 2)):
        keep = x[m, k].clone()
        x[m, k] = -7e4
        with pytest.raises(ValueError, match="exceed fp16's range"):
            _run(x)
        with pytest.raises(ValueError):
            _run(x, s, 2.0)
        _run(x, s, 0.25)  # in range after the scales
        x[m, k] = keep
    _run(x)


def test_threads_and_streams(cuda):
    good = torch.ones(64, 4096, device=cuda, dtype=torch.bfloat16)
    bad = good.clone()
    bad[63, 4095] = 1e5
    torch.cuda.synchronize()
    wrong = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for n in range(50):
                over = (n + i) % 3 == 0
                try:
                    _run(bad if over else good)
                    raised = False
                except ValueError:
                    raised = True
                if raised != over:
                    wrong.append((i, n))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not wrong and not any(t.is_alive() for t in threads)


@pytest.mark.parametrize("ahead", [0, 1, 8])
def test_waits_for_its_own_pass_only(cuda, ahead):
    """Whatever is queued before the pass (8192^3 products of about a millisecond each), the answer
    comes when the pass is done, with what was launched behind it still under way."""
    a = torch.ones(8192, 8192, device=cuda, dtype=torch.float16)
    out = torch.empty_like(a)
    x = torch.ones(8, 4096, device=cuda, dtype=torch.bfloat16)
    torch.mm(a, a, out=out)
    _run(x)
    for value in (1.0, 1e5):
        x[7, 4095] = value
        torch.cuda.synchronize()
        for _ in range(ahead):
            torch.mm(a, a, out=out)
        try:
            with _pk.checked_activations(x, None, 1.0, "t") as y:
                for _ in range(60):
                    torch.mm(a, a, out=out)
            raised = False
        except ValueError:
            raised = True  # (the message's maximum synchronises)
        else:
            assert not torch.cuda.current_stream().query()
        torch.cuda.synchronize()
        assert raised == (value > 65504) and torch.equal(y, x.half())


def test_capture_runs_the_plain_pass(cuda):
    x = torch.full((4, 256), 1e5, device=cuda, dtype=torch.bfloat16)
    _run(torch.ones_like(x))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = _run(x)
    for v, want in ((2.0, 2.0), (1e5, float("inf"))):
        x.fill_(v)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, torch.full_like(y, want))
