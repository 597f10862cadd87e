"""The K = 16384 down projection on its E3M2 form (calls of thousands of rows): the quantizer's
codes against the INT4 quantizer's, the GEMM against the INT4 kernel's, and which calls take it."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import w4a4_oracle as orc
from tests import w4a4_inputs as inp

pytestmark = pytest.mark.gpu
K = 16384


@pytest.fixture(scope="module")
def ext(cuda):
    from pi05_fast.w4a4 import extension

    extension.preload()
    return extension


def _same(a: torch.Tensor, b: torch.Tensor) -> bool:
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


def _weight(ext, gen, n, cuda):
    """An MFMA-layout weight and its E3M2 form."""
    packed = inp.random_packed(gen, n, K).to(cuda)
    return ext.repack_weight(packed, k=K, tiled=False), ext.repack_weight_e3m2(packed, k=K)


@pytest.mark.parametrize("m", [1, 17, 129, 300])
def test_quantizer_equals_int4(ext, cuda, m):
    from pi05_fast.w4a4.pack import codes_from_e3m2_fragments, codes_from_fragment_major

    x = inp.geglu_activations(inp.generator(8100 + m), m, K)
    x[m // 2] = 0
    k16 = min(16, m)  # exact half-integer quotients: x = FWHT(y) / K is exact in fp16
    rng = np.random.default_rng(m)
    y = np.zeros((k16, K), np.float64)
    for r in range(k16):
        y[r, 0] = 7.0
        y[r, rng.choice(np.arange(1, K), size=48, replace=False)] = rng.choice(np.arange(-6.5, 7.0, 1.0), size=48)
    x[:k16] = torch.from_numpy((orc.fwht_unnormalized((y / 16).astype(np.float32)).astype(np.float64) / K).astype(np.float16))
    x = x.to(cuda)
    q, sa = ext.quantize(x)
    q6 = torch.empty(ext._q6_bytes(m, K), dtype=torch.uint8, device=cuda)
    s6 = torch.empty(m, dtype=torch.float32, device=cuda)
    ext._check(ext.load_int4_gemm().pi05w4a4_quantize_e3m2_k16384(x.data_ptr(), m, q6.data_ptr(), s6.data_ptr(),
                                                                  ext._stream(x.device)), "quantize")
    torch.cuda.synchronize()
    c4 = orc.unpack_nibbles(inp.to_np(codes_from_fragment_major(q.cpu(), m, K)), K)
    assert np.array_equal(inp.to_np(codes_from_e3m2_fragments(q6.cpu(), m, K)).astype(np.int32), c4.astype(np.int32))
    assert torch.equal(sa.view(torch.int32), s6.view(torch.int32))


@pytest.mark.parametrize("residual", [False, True])
@pytest.mark.parametrize("m,n", [(1, 2048), (113, 32), (200, 2080), (1000, 288)])
def test_gemm_edges(ext, cuda, m, n, residual):
    """Tile heights, ragged rows and columns (called directly: below the row count of the rule)."""
    gen = inp.generator(8200 + m + n)
    w4, w6 = _weight(ext, gen, n, cuda)
    x = inp.geglu_activations(gen, m, K).to(cuda)
    r = torch.randn(m, n, generator=gen).half().to(cuda) if residual else None
    want = ext.int4_gemm_residual(x, w4, r) if residual else ext.int4_gemm(x, w4)
    assert _same(ext._run_e3m2_rows(x, w6, K, m, r)[0], want)


def test_rule(ext, cuda, monkeypatch):
    """Rows on both sides of the rule, views, and the calls that stay on the INT4 weight."""
    monkeypatch.setattr(ext, "E3M2_MIN_ROWS_K16384", 256)
    gen = inp.generator(8300)
    w4, w6 = _weight(ext, gen, 64, cuda)
    big = torch.zeros(3 * 100 * K + 8, dtype=torch.float16, device=cuda)
    big[1 : 1 + 3 * 100 * K] = inp.geglu_activations(gen, 300, K).to(cuda).view(-1)
    odd = big[1 : 1 + 3 * 100 * K].view(3, 100, K)  # 2-byte aligned
    x = odd.clone()
    r = torch.randn(3, 64, 100, generator=gen).half().to(cuda).transpose(1, 2)  # not contiguous
    want, want_r, want_255 = ext.int4_gemm(x, w4), ext.int4_gemm_residual(x, w4, r), ext.int4_gemm(x.view(300, K)[:255], w4)

    calls = []
    real = ext._run_e3m2_rows
    monkeypatch.setattr(ext, "_run_e3m2_rows", lambda *a: calls.append(a[3]) or real(*a))
    ext.register_e3m2_form(w4, w6, K)
    assert _same(ext.int4_gemm(x, w4), want) and _same(ext.int4_gemm(odd, w4), want)
    assert _same(ext.int4_gemm(x.transpose(0, 1), w4), want.transpose(0, 1).contiguous())
    assert _same(ext.int4_gemm_residual(x, w4, r), want_r)
    assert calls == [300] * 4
    assert _same(ext.int4_gemm(x.view(300, K)[:255], w4), want_255) and calls == [300] * 4
    with pytest.raises(RuntimeError):
        ext.int4_gemm_residual(x, w4, r[:, :, :32])
    # infinities and NaN give what they give on the INT4 weight
    bad = x.clone()
    bad[0, 3, 7], bad[1, 5, 11], bad[2, 9, 13] = float("inf"), float("nan"), -float("inf")
    got = ext.int4_gemm(bad, w4)
    ext.clear_weight_caches()
    assert torch.allclose(got, ext.int4_gemm(bad, w4), rtol=0, atol=0, equal_nan=True) and len(calls) == 5
    # a weight written in place leaves its form
    ext.register_e3m2_form(w4, w6, K)
    w4.zero_()
    assert not ext.int4_gemm(x, w4).any() and len(calls) == 5


@pytest.mark.parametrize("m", [256, 768, 1000])
def test_warming(ext, cuda, monkeypatch, m):
    """Buffers to warm change nothing in the outputs, the weight in them stands for the form that
    the call reads, and what the quantizer refuses stays refused."""
    monkeypatch.setattr(ext, "E3M2_MIN_ROWS_K16384", 256)
    gen = inp.generator(8500 + m)
    w4, w6 = _weight(ext, gen, 64, cuda)
    x, r = inp.geglu_activations(gen, m, K).to(cuda), torch.randn(m, 64, generator=gen).half().to(cuda)
    want = ext.int4_gemm_residual(x, w4, r)
    ext.register_e3m2_form(w4, w6, K)
    big = torch.ones(1 << 20, dtype=torch.uint8, device=cuda)
    seen = []
    real = ext._warm_args
    monkeypatch.setattr(ext, "_warm_args", lambda warm, who: seen.append(list(warm)) or real(warm, who))
    assert _same(ext.int4_gemm_residual(x, w4, r, warm=[w4, big]), want)
    assert len(seen) == 1 and seen[0][0] is w6 and seen[0][1].data_ptr() == big.data_ptr()
    for bad in ([big.cpu()], [big[::2]], [big] * 5):
        with pytest.raises(RuntimeError):
            ext.int4_gemm_residual(x, w4, r, warm=bad)


def test_weight_loaded_under_inference_mode(ext, cuda, monkeypatch):
    """No E3M2 form is kept for it, and its calls run on the INT4 weight."""
    from pi05_fast.w4a4.apply import load_time_weight

    monkeypatch.setattr(ext, "E3M2_MIN_ROWS_K16384", 256)
    gen = inp.generator(8400)
    packed = inp.random_packed(gen, 64, K)
    x = inp.geglu_activations(gen, 300, K).to(cuda)
    want = ext.int4_gemm(x, packed.to(cuda))
    with torch.inference_mode():
        w, shuffled = load_time_weight(packed, "layers.0.mlp.down_proj", K, 64, torch.device(cuda))
        assert not shuffled and ext.e3m2_form(w, K) is None
        assert _same(ext.int4_gemm(x, w), want)


def test_entry_refusals(ext, cuda):
    lib = ext.load_int4_gemm()
    b = torch.zeros(1 << 20, dtype=torch.uint8, device=cuda).data_ptr()
    st = ext._stream(torch.device(cuda))
    assert lib.pi05w4a4_quantize_e3m2_k16384(None, 4, b, b, st) != 0
    assert lib.pi05w4a4_quantize_e3m2_k16384(b + 2, 4, b, b, st) != 0
    assert lib.pi05w4a4_quantize_e3m2_k16384(b, -1, b, b, st) != 0
    assert lib.pi05w4a4_quantize_e3m2_k16384(None, 0, None, None, st) == 0
    assert lib.pi05w4a4_gemm_e3m2_rows(b, b, 4, K, b, 40, None, b, st) != 0
    assert lib.pi05w4a4_gemm_e3m2_rows(b, b, 4, 100, b, 32, None, b, st) != 0
    assert lib.pi05w4a4_gemm_e3m2_rows(b, b, 4, K, b, 32, b + 2, b, st) != 0
    assert lib.pi05w4a4_gemm_e3m2_rows(b, b, 4, K, None, 32, None, b, st) != 0
    assert lib.pi05w4a4_gemm_e3m2_rows(b, b, 112 * 65536, K, b, 32, None, b, st) != 0
