"""The prefix attention with 128 query rows per workgroup (from three rounds of 32-row
workgroups on): ragged rows and keys, masks that hide whole steps and whole rows, head
groupings, and the calls that stay on the 32-row kernel, against that kernel on the same
sequences and against fp32."""

from __future__ import annotations

import pytest
import torch

from tests.test_gpu_attention import D, _inputs, _reference, _rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext(cuda):
    from pi05_fast.w4a4 import extension

    extension.preload()
    return extension


def _batch(cuda, s, n_rep, kvh):
    """The smallest batch with more than two rounds of 32-row workgroups."""
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    return 2 * cus // (-(-s * n_rep // 32) * kvh) + 1


def _mask(kind, b, s, cuda):
    if kind is None:
        return None
    neg = torch.finfo(torch.float16).min
    m = torch.zeros(b, 1, s, s, dtype=torch.float16, device=cuda)
    i = torch.arange(s, device=cuda)
    if kind == "causal":
        m.masked_fill_(i[None, :] > i[:, None], neg)
    elif kind == "padding":  # other lengths per sequence
        for x in range(b):
            m[x, 0, :, max(1, s - 7 * x % s) :] = neg
    elif kind == "front":  # the first keys hidden by -inf: whole steps before any visible key
        m[:, :, :, : s - 1 - s // 4] = float("-inf")
    elif kind == "lowest":  # rows that see no key: the scores collapse onto the type's lowest value
        m[:, :, ::3, :] = neg
    elif kind == "bias":  # the row's largest score arrives late, far above the earlier ones
        m += (i[None, :] // 16).half() * 3.0
    return m


# s * n_rep around multiples of 32 and 128, s around multiples of 32 and 64; kvh > 1
CASES = [(1, 8, 1, None), (8, 8, 1, "causal"), (31, 8, 1, "front"), (33, 8, 1, "lowest"), (64, 8, 1, "bias"),
         (97, 8, 1, "padding"), (389, 8, 1, "front"), (776, 8, 1, "lowest"), (1024, 8, 1, "causal"),
         (1023, 8, 1, "bias"), (65, 2, 2, "padding"), (130, 1, 3, "causal"), (43, 3, 1, "bias")]


@pytest.mark.parametrize("s,n_rep,kvh,kind", CASES)
def test_wide_attention_matches_one_sequence_at_a_time(ext, cuda, s, n_rep, kvh, kind):
    h, b = n_rep * kvh, _batch(cuda, s, n_rep, kvh)
    q, k, v, cos, sin = _inputs(b, s, h, kvh, cuda, seed=s + n_rep)
    mask = _mask(kind, b, s, cuda)
    with torch.no_grad():
        got, keys = ext.prefix_attention(q, k, v, cos, sin, mask, D**-0.5, h, kvh)
        one = [ext.prefix_attention(q[i : i + 1], k[i : i + 1], v[i : i + 1], cos[i : i + 1], sin[i : i + 1],
                                    None if mask is None else mask[i : i + 1], D**-0.5, h, kvh) for i in range(min(b, 24))]
    torch.cuda.synchronize()
    n = len(one)
    want = torch.cat([o for o, _ in one])
    assert torch.equal(keys[:n], torch.cat([x for _, x in one]))
    assert torch.isfinite(got).all()
    # Same scores; the probabilities are rounded to fp16 before (here) or after (there) their
    # division by the row sum, and the outputs once each: three roundings of 2^-12 (root mean
    # square of a half ulp over its binade: 2^-11 / sqrt(3) at most), independent.
    assert _rel_l2(got[:n], want) <= 3 * 2.0**-11
    # fp32 reference (fp16 rounding of the scores): the attention tests' bar; rows that see no
    # key have other scores there, and the late maximum's scores of ~190 round to 1/8
    if kind not in ("lowest", "bias"):
        ref = torch.cat([_reference(q[i : i + 1], k[i : i + 1], v[i : i + 1], cos[i : i + 1], sin[i : i + 1],
                                    None if mask is None else mask[i : i + 1], D**-0.5, h, kvh) for i in range(b - 2, b)])
        assert _rel_l2(got[b - 2 :], ref) <= 2e-3


def test_wide_attention_rows_of_infinities(ext, cuda):
    """Rows hidden by -inf alone and rows with a +inf score are NaN, and only they."""
    s, h = 100, 8
    b = _batch(cuda, s, h, 1)
    q, k, v, cos, sin = _inputs(b, s, h, 1, cuda, seed=9)
    mask = torch.zeros(b, 1, s, s, dtype=torch.float16, device=cuda)
    mask[:, :, 5] = float("-inf")
    mask[:, :, 70, 40] = float("inf")
    with torch.no_grad():
        got, _ = ext.prefix_attention(q, k, v, cos, sin, mask, D**-0.5, h, 1)
        one, _ = ext.prefix_attention(q[:1], k[:1], v[:1], cos[:1], sin[:1], mask[:1], D**-0.5, h, 1)
    nan = torch.zeros(b, s, dtype=torch.bool, device=cuda)
    nan[:, [5, 70]] = True
    assert torch.equal(got.isnan().all(-1), nan) and torch.equal(got.isnan().any(-1), nan)
    assert torch.equal(one.isnan().any(-1), nan[:1])


def test_wide_attention_strided_inputs(ext, cuda):
    """Queries and values as views of one QKV buffer, a broadcast mask with padded rows."""
    s, h = 75, 8
    b = _batch(cuda, s, h, 1)
    q, k, v, cos, sin = _inputs(b, s, h, 1, cuda, seed=11)
    qkv = torch.cat([q, k, v], dim=-1)
    buf = torch.full((1, 1, s, 88), float("nan"), dtype=torch.float16, device=cuda)
    mask = buf[..., :s]
    mask.copy_(_mask("causal", 1, s, cuda))
    with torch.no_grad():
        want, _ = ext.prefix_attention(q, k, v, cos, sin, mask.expand(b, 1, s, s).contiguous(), D**-0.5, h, 1)
        got, _ = ext.prefix_attention(*qkv.split([h * D, D, D], dim=-1), cos, sin, mask, D**-0.5, h, 1)
    assert torch.equal(got, want)


def test_scaling_that_is_no_fp16_number_keeps_its_products(ext, cuda):
    """Scores scaled by an fp32 factor stay on the 32-row kernel: the same bits in a batch."""
    s, h = 64, 8
    b = _batch(cuda, s, h, 1)
    q, k, v, cos, sin = _inputs(b, s, h, 1, cuda, seed=12)
    with torch.no_grad():
        got, _ = ext.prefix_attention(q, k, v, cos, sin, None, 0.0623, h, 1)
        one, _ = ext.prefix_attention(q[3:4], k[3:4], v[3:4], cos[3:4], sin[3:4], None, 0.0623, h, 1)
    assert torch.equal(got[3:4], one)
