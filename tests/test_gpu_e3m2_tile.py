"""The E3M2 GEMM's main tile at its edges: every tile height (plain, paired and with a
residual), ragged rows and columns, the shortest k ranges (one to five 128-deep blocks, odd
counts among them) and grids in which a workgroup walks several tiles, against exact integer
arithmetic on the same codes."""

from __future__ import annotations

import ctypes

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


def _q6(codes: torch.Tensor) -> torch.Tensor:
    """E3M2 fragments (int32 words) of codes [M, K] in [-7, 7]: per 16 rows x 128 k the
    dwords 0-3 of 64 lanes, then their dwords 4-5; lane L holds codes 32 (L / 16) .. of row L % 16."""
    m, k = codes.shape
    pad = torch.zeros((-m) % 16, k, dtype=codes.dtype, device=codes.device)
    c = torch.cat([codes, pad]).to(torch.int64).view(-1, 16, k // 128, 4, 32).permute(0, 2, 3, 1, 4).reshape(-1, 64, 32)
    mag = torch.tensor([0, 0x0C, 0x10, 0x12, 0x14, 0x15, 0x16, 0x17], device=codes.device)
    v = mag[c.abs()] | ((c < 0).to(torch.int64) << 5)
    d = torch.zeros(c.size(0), 64, 6, dtype=torch.int64, device=codes.device)
    for j in range(32):
        w, s = divmod(6 * j, 32)
        d[..., w] |= (v[..., j] << s) & 0xFFFFFFFF
        if s > 26:
            d[..., w + 1] |= v[..., j] >> (32 - s)
    d = torch.where(d >= 2**31, d - 2**32, d).to(torch.int32)
    return torch.cat([d[..., :4].reshape(-1, 256), d[..., 4:].reshape(-1, 128)], dim=1).reshape(-1).contiguous()


def _gemm(ext, q6, sa, m, k, ws, ns, outs, gelu):
    lib = ext.load_int4_gemm()
    g = len(ws)
    ext._check(lib.pi05w4a4_gemm_e3m2(
        q6.data_ptr(), sa.data_ptr(), m, k, g, (ctypes.c_void_p * g)(*[w.data_ptr() for w in ws]),
        (ctypes.c_int32 * g)(*ns), (ctypes.c_void_p * g)(*[o.data_ptr() for o in outs]), int(gelu),
        ext._stream(sa.device)), "pi05w4a4_gemm_e3m2")


# (rows, k, columns): tile heights 64-112 rows, one tile and several per workgroup
SHAPES = [(1, 128, 64), (65, 256, 96), (112, 384, 32), (113, 512, 1056), (176, 640, 160), (330, 2048, 288),
          (700, 512, 16384), (1000, 256, 16384), (784, 1024, 8224)]


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_gelu_pairs(ext, cuda, m, k, n):
    gen = inp.generator(9000 + m + k)
    codes = torch.randint(-7, 8, (m, k), generator=gen, dtype=torch.int32).to(cuda)
    sa = (torch.rand(m, generator=gen) * 0.02 + 0.001).to(cuda)
    packed = [inp.random_packed(gen, n, k).to(cuda) for _ in range(2)]
    w6 = [ext.repack_weight_e3m2(w, k=k) for w in packed]
    y = torch.full((m, n), float("nan"), dtype=torch.float16, device=cuda)
    _gemm(ext, _q6(codes), sa, m, k, w6, [n, n], [y, y], True)
    want = []
    for w in packed:
        b = torch.from_numpy(orc.unpack_nibbles(inp.to_np(w[:, : k // 8]), k).astype(np.float32)).to(cuda)
        acc = codes.float() @ b.t()  # integers below 2^24: exact
        want.append(((acc * sa[:, None]) * w[:, k // 8].view(torch.float32)[None]).half())
    assert torch.equal(y.view(torch.int16), ext.gelu_tanh_mul(*want).view(torch.int16))


# tile heights 64, 80, 80, 96, 96, 64, 112, 112, 112, 112 rows
@pytest.mark.parametrize("m,k,n", [(64, 512, 90144), (225, 256, 24608), (240, 2048, 24608), (241, 384, 24608),
                                   (288, 512, 24608), (128, 128, 40960), (300, 384, 24608), (784, 512, 16384),
                                   (2240, 2048, 4096), (336, 256, 24608)])
def test_plain_groups(ext, cuda, m, k, n):
    """Two weights of different widths whose 112-row tiles fill the device (the main tile)."""
    gen = inp.generator(9500 + m + k)
    codes = torch.randint(-7, 8, (m, k), generator=gen, dtype=torch.int32).to(cuda)
    sa = (torch.rand(m, generator=gen) * 0.02 + 0.001).to(cuda)
    ns = [n, 8192 + 32]
    packed = [inp.random_packed(gen, nn, k).to(cuda) for nn in ns]
    w6 = [ext.repack_weight_e3m2(w, k=k) for w in packed]
    outs = [torch.full((m, nn), float("nan"), dtype=torch.float16, device=cuda) for nn in ns]
    _gemm(ext, _q6(codes), sa, m, k, w6, ns, outs, False)
    for w, y in zip(packed, outs):
        b = torch.from_numpy(orc.unpack_nibbles(inp.to_np(w[:, : k // 8]), k).astype(np.float32)).to(cuda)
        want = (((codes.float() @ b.t()) * sa[:, None]) * w[:, k // 8].view(torch.float32)[None]).half()
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))


# tile heights 64, 80, 96 and 112 rows on odd and even counts of k blocks; then (the last two) more
# tiles than two per CU, so that a workgroup goes on to a second tile past its epilogue
@pytest.mark.parametrize("m,k,n", [(64, 256, 288), (70, 384, 2080), (96, 2048, 288), (200, 640, 96), (1000, 512, 16416),
                                   (1500, 1024, 16384)])
def test_rows_with_residual(ext, cuda, m, k, n):
    gen = inp.generator(9800 + m + k)
    codes = torch.randint(-7, 8, (m, k), generator=gen, dtype=torch.int32).to(cuda)
    sa = (torch.rand(m, generator=gen) * 0.02 + 0.001).to(cuda)
    packed = inp.random_packed(gen, n, k).to(cuda)
    w6 = ext.repack_weight_e3m2(packed, k=k)
    res = torch.randn(m, n, generator=gen).half().to(cuda)
    q6 = _q6(codes)
    b = torch.from_numpy(orc.unpack_nibbles(inp.to_np(packed[:, : k // 8]), k).astype(np.float32)).to(cuda)
    want = (((codes.float() @ b.t()) * sa[:, None]) * packed[:, k // 8].view(torch.float32)[None]).half()
    for r, ref in ((None, want), (res, want + res)):
        y = torch.full((m, n), float("nan"), dtype=torch.float16, device=cuda)
        ext._check(ext.load_int4_gemm().pi05w4a4_gemm_e3m2_rows(
            q6.data_ptr(), sa.data_ptr(), m, k, w6.data_ptr(), n, ext._ptr(r), y.data_ptr(), ext._stream(sa.device)),
            "pi05w4a4_gemm_e3m2_rows")
        assert torch.equal(y.view(torch.int16), ref.view(torch.int16))
