"""The K = 16384 quantizer at the edges of its two forms (whole rows up to four per CU, half
rows beyond) and every rotated quantizer at the edges of its order of the rows (128-row runs
dealt to the XCDs by 16-row blocks, the rest in order), against the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import w4a4_oracle as orc
from tests import w4a4_inputs as inp

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext(cuda):
    from pi05_fast.w4a4 import extension

    extension.preload()
    return extension


def _edge_rows(gen, m: int, k: int) -> torch.Tensor:
    """Activations with rows of zeros, fp16 subnormals, the largest values and one nonzero."""
    x = inp.activations(gen, m, k)
    x[0::7] = 0
    x[1::7] = (torch.randint(-1023, 1024, (x[1::7].shape), generator=gen).float() * 2.0**-24).half()
    x[2::7] = torch.where(x[2::7] < 0, -65504.0, 65504.0).half()
    x[3::7] = 0
    x[3::7, k - 3] = -1.5
    return x


def _check(ext, x: torch.Tensor, cuda, m: int, k: int) -> None:
    from pi05_fast.w4a4.pack import codes_from_fragment_major

    q, sa = ext.quantize(x.to(cuda))
    torch.cuda.synchronize()
    q_ref, s_ref = orc.quant_activation(x.numpy())
    got = orc.unpack_nibbles(inp.to_np(codes_from_fragment_major(q.cpu(), m, k)), k)
    assert np.array_equal(got.astype(np.int32), q_ref.astype(np.int32))
    assert np.array_equal(inp.to_np(sa).view(np.int32), s_ref.view(np.int32))


@pytest.mark.parametrize("m", [16, 127, 128, 129, 145, 256])
@pytest.mark.parametrize("k", [2048, 16384])
def test_row_order_edges(ext, cuda, m, k):
    _check(ext, _edge_rows(inp.generator(7000 + m + k), m, k), cuda, m, k)


@pytest.mark.parametrize("over", [0, 1, 115])
def test_half_row_form_edges(ext, cuda, over):
    m = 4 * torch.cuda.get_device_properties(cuda).multi_processor_count + over
    _check(ext, _edge_rows(inp.generator(7500 + over), m, 16384), cuda, m, 16384)


def test_half_row_form_ties(ext, cuda):
    """Exact half-integer quotients in the half-row form (x = FWHT(y) / K is exact in fp16)."""
    k, m = 16384, 4 * torch.cuda.get_device_properties(cuda).multi_processor_count + 16
    rng = np.random.default_rng(75)
    y = np.zeros((16, k), np.float64)
    for r in range(16):
        y[r, 0] = 7.0 if r % 2 == 0 else -7.0
        y[r, rng.choice(np.arange(1, k), size=48, replace=False)] = rng.choice(np.arange(-6.5, 7.0, 1.0), size=48)
    x16 = (orc.fwht_unnormalized((y / 16).astype(np.float32)).astype(np.float64) / k).astype(np.float16)
    x = inp.activations(inp.generator(7600), m, k)
    x[m - 16 :] = torch.from_numpy(x16)
    _check(ext, x, cuda, m, k)


@pytest.mark.parametrize("m", [1, 3, 127, 129, 511, 512, 513])
@pytest.mark.parametrize("k", [64, 960, 1088, 4096, 4160, 8192, 8256])
def test_unrotated_rows_match_oracle(ext, cuda, m, k):
    """The unrotated quantizer at the edges of its wave-per-row forms (K = 1024, 2048, 4096,
    8192; 512 rows; runs of 128 rows), with rows whose codes are exact ties:
    the codes and row sums of every form are the oracle's."""
    from pi05_fast.w4a4.pack import codes_from_fragment_major, qcorr_from_fragment_major

    gen = inp.generator(31 * k + m)
    x = _edge_rows(gen, m, k)
    ties = (torch.randint(-7, 7, x[4::7].shape, generator=gen).float() + 0.5).half()
    ties[:, 5] = 7.0  # the row's scale is 1: every other value lies between two codes
    x[4::7] = ties
    _check(ext, x, cuda, m, k)
    q, _ = ext.quantize(x.to(cuda))
    codes = orc.unpack_nibbles(inp.to_np(codes_from_fragment_major(q.cpu(), m, k)), k)
    want = -128 * codes[:, 1::2].astype(np.int64).sum(axis=1)
    assert np.array_equal(inp.to_np(qcorr_from_fragment_major(q.cpu(), m, k)), want)


@pytest.mark.parametrize("k", [2112, 4096, 8192])
def test_unrotated_infinities_and_nan(ext, cuda, k):
    """Rows with infinities and NaN: a wave per row (600 rows) gives the codes, scales and row sums
    of a workgroup per row (the first 500 of them alone)."""
    from pi05_fast.w4a4.pack import codes_from_fragment_major, qcorr_from_fragment_major

    x = _edge_rows(inp.generator(7700 + k), 600, k)
    x[5, 9], x[12, 100], x[19, k - 1] = float("inf"), float("nan"), -float("inf")
    x[26], x[33, ::2], x[40, ::3] = float("nan"), float("inf"), float("nan")
    out = []
    for m in (600, 500):
        q, sa = ext.quantize(x[:m].to(cuda))
        codes = inp.to_np(codes_from_fragment_major(q.cpu(), m, k))[:500]
        out.append((codes, inp.to_np(sa).view(np.int32)[:500], inp.to_np(qcorr_from_fragment_major(q.cpu(), m, k))[:500]))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
