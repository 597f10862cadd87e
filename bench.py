#!/usr/bin/env python3
"""Benchmark: W4A4 PaliGemma-2B-shaped prefix LM on one MI355X.

    python bench.py [--steps K] [--warmup W] [--tokens 776] [--batch 1] [--layers 18]

Workload (`value`): one forward of the 18-layer Gemma-2B-shaped prefix LM (hidden 2048,
8x256 heads, 1 KV head, intermediate 16384) over a 776-token prefix, batch 1, every
q/k/v/o/gate/up/down projection running the W4A4 path (FWHT + INT4 quant, int8-MFMA
GEMM), RoPE + attention as the two prefix-attention kernels and each RMSNorm as one kernel.  Weights are synthetic packed INT4 (random codes with the
statistics of a packed N(0, 0.02) weight), inputs synthetic N(0, 1/sqrt(2048)) prefix
embeddings, all resident in HBM.  Timed region: K replays of the whole forward captured
in one HIP graph, bracketed by device synchronisation; `value` = ms per forward.

Per-kernel figures (`gemms`, `roofline`): each W4A4 kernel of the forward is launched
through the C ABI with preallocated buffers at the forward's shapes.  After a warm-up of
about 0.3 s of back-to-back launches (clocks settle), `--kernel-iters` launches are
captured in one HIP graph; HIP events recorded on the launching stream (torch's current
stream, which the library uses) bracket each of 5 replays, and the median per-launch
time gives the kernel duration, int8 TOPS and the fraction of the MI355X dense int8 MFMA
peak (GEMMs) or of HBM bandwidth (quantizers).  The graph removes host launch gaps
between the back-to-back kernels.  The non-W4A4 kernels of the forward (prefix attention,
its K/V prep, RMSNorm) are timed the same way under `other_kernels`.
The dominant kernel of the forward (the gate/up GEMM with its fused GELU-tanh*up
epilogue, ~29% of the forward) is the `roofline` object; its `traffic` (HBM bytes per
launch) comes from the rocprofv3 FETCH_SIZE/WRITE_SIZE summary committed under profiles/.

`in_forward` times the same kernels inside the real graph-replayed forward from their own
begin/end timestamps (torch.profiler over 10 replays, the timestamps rocprofv3's kernel
trace reads), scaled by one factor so that the forward's kernels sum to the unprofiled
replay time (the profiler slows every kernel by a few %).  `roofline.in_forward` is the
dominant kernel's figure from it.  `in_forward.event_pairs` keeps a second estimate: HIP
events around each library call of the eager forward, with a bounded spin kernel queued
ahead so that the host has enqueued the whole forward before the GPU runs it, each class
corrected by the event-pair cost that the same kernel shows alone (`pair_offset_us`:
graph-timed launch against event pairs around eager launches).

`cpu_baseline` times the reference's W4A4 semantics in PyTorch on the host CPU (the
oracle's torch restatement of pack.py:113-145, both integer matmul forms) on one decoder
layer's projection calls at the same M and scales it to the full depth.

Prints one JSON line.
"""

from __future__ import annotations

import argparse
import ctypes
import itertools
import json
import os
import re
import statistics
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
for _p in (ROOT / "pi05-pytorch-fast_amd", ROOT):
    if str(_p) not in sys.path:
        sys.path.insert(0, str(_p))

METRIC = "W4A4 prefix-LM ms @776 tok; int8 TOPS & % MFMA peak per GEMM (1 MI355X)"
INT8_PEAK_TOPS = 5000.0   # MI355X dense int8 MFMA, published
FP16_PEAK_TFLOPS = 2500.0  # MI355X dense fp16 MFMA, published
FP6_PEAK_TOPS = 10100.0    # MI355X dense fp6 / fp4 MFMA, published
HBM_PEAK_GBS = 8000.0     # MI355X HBM3E, published
# HBM-side traffic per launch of the W4A4 kernels (rocprofv3 FETCH_SIZE / WRITE_SIZE summary).
TRAFFIC_FILE = ROOT / "profiles" / "w4a4_kernels_776tok_traffic.md"
# The forward's gate/up weights take the E3M2 operand form at load unless PI05_W4A4_E3M2=0.
E3M2_GATE_UP = os.environ.get("PI05_W4A4_E3M2", "1") != "0"


def parse_args():
    ap = argparse.ArgumentParser(description=__doc__.splitlines()[0])
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--tokens", type=int, default=776)
    ap.add_argument("--batch", type=int, default=1)
    ap.add_argument("--layers", type=int, default=18)
    ap.add_argument("--kernel-iters", type=int, default=100, help="launches per timed graph replay")
    ap.add_argument("--kernel-warmup-s", type=float, default=0.3, help="eager warm-up per kernel (s)")
    ap.add_argument("--no-graph", action="store_true", help="time eager forwards instead of graph replays")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--cpu-seconds", type=float, default=15.0, help="budget of the CPU baseline")
    ap.add_argument("--unfused-gelu", action="store_true",
                    help="gate/up as two fp16 outputs + eager gelu*up instead of the fused epilogue")
    ap.add_argument("--only-kernel", default="",
                    help="skip the forward; launch only this kernel class (for rocprofv3 --pmc runs)")
    ap.add_argument("--no-extra-points", action="store_true",
                    help="skip the 640/768-token, batch-8 and eager-attention forward points")
    ap.add_argument("--forward-only", action="store_true",
                    help="time the graph-replayed forward only (no per-kernel table, no CPU baseline): "
                         "for a kernel trace of the real forward")
    return ap.parse_args()


# ----------------------------------------------------------------------------- kernels
class KernelBench:
    """Back-to-back launches of one W4A4 kernel through the C ABI, timed with HIP events
    recorded on the launching stream."""

    def __init__(self, torch, ext, dev, iters, warm_s=0.3, reps=5):
        self.torch, self.ext, self.dev, self.iters = torch, ext, dev, iters
        self.warm_s, self.reps = warm_s, reps
        self.lib = ext.load_int4_gemm()

    def _stream(self):
        return ctypes.c_void_p(self.torch.cuda.current_stream(self.dev).cuda_stream)

    def _time(self, fn, iters: int | None = None) -> float:
        """Median microseconds per launch of `fn` over `reps` replays of a graph holding
        `iters` launches (default: the bench's), after an eager warm-up of about `warm_s`
        seconds."""
        torch = self.torch
        iters = iters or self.iters
        fn()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        while time.perf_counter() - t0 < self.warm_s:
            for _ in range(20):
                fn()
            torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(iters):
                fn()
        graph.replay()
        torch.cuda.synchronize()
        per_launch = []
        for _ in range(self.reps):
            e0 = torch.cuda.Event(enable_timing=True)
            e1 = torch.cuda.Event(enable_timing=True)
            e0.record()
            graph.replay()
            e1.record()
            torch.cuda.synchronize()
            per_launch.append(e0.elapsed_time(e1) * 1e3 / iters)
        del graph
        us = statistics.median(per_launch)
        self.last_pair_us = self._pair_us(fn)
        self.last_pair_offset_us = round(self.last_pair_us - us, 3)
        return us

    def _pair_us(self, fn, reps: int = 40) -> float:
        """Median interval of an event pair recorded around one eager launch of `fn`, with
        the queue primed by a bounded spin kernel (the way in_forward_times times each call
        of the real forward): the launch's time plus what the two markers add to it.  Its
        difference to the graph-timed launch is the event-pair cost of this kernel, taken off
        the in-forward times of its class."""
        torch = self.torch
        fn()
        torch.cuda.synchronize()
        torch.cuda._sleep(50_000_000)  # ~25 ms at ~2 GHz: longer than enqueuing the pairs
        pairs = []
        for _ in range(reps):
            e0 = torch.cuda.Event(enable_timing=True)
            e1 = torch.cuda.Event(enable_timing=True)
            e0.record()
            fn()
            e1.record()
            pairs.append((e0, e1))
        torch.cuda.synchronize()
        return statistics.median(a.elapsed_time(b) * 1e3 for a, b in pairs)

    def _check(self, rc):
        if rc != 0:
            raise RuntimeError(self.lib.pi05w4a4_last_error().decode())

    def _packed(self, n, k, gen):
        torch = self.torch
        w = torch.randint(-(2**31), 2**31 - 1, (n, k // 8 + 1), dtype=torch.int32, device=self.dev,
                          generator=gen)
        w[:, -1] = (torch.rand(n, device=self.dev, generator=gen) * 0.05 + 0.01).view(torch.int32)
        return self.ext.repack_weight(w, k=k)

    def quant(self, m, k):
        torch, lib, P = self.torch, self.lib, self.ext._ptr
        x = torch.randn(m, k, device=self.dev, dtype=torch.float16)
        q = torch.empty(int(lib.pi05w4a4_q_words(m, k)), dtype=torch.int32, device=self.dev)
        sa = torch.empty(m, dtype=torch.float32, device=self.dev)
        us = self._time(lambda: self._check(lib.pi05w4a4_quantize(P(x), m, k, P(q), P(sa), self._stream())))
        nbytes = 2.0 * m * k + m * k / 2 + 4 * m
        gbs = nbytes / (us * 1e-6) / 1e9
        return {"m": m, "k": k, "avg_us": round(us, 3), "bytes": nbytes, "gbs": round(gbs, 1),
                "frac_hbm": round(gbs / HBM_PEAK_GBS, 4), "pair_offset_us": self.last_pair_offset_us}

    def rmsnorm_quant(self, m, k=2048, e3m2=False):
        """The RMSNorm + K = 2048 activation quant kernel; `e3m2`: its E3M2-fragment form
        (the gate/up input)."""
        torch, lib, P = self.torch, self.lib, self.ext._ptr
        x = torch.randn(m, k, device=self.dev, dtype=torch.float16)
        w = torch.randn(k, device=self.dev, dtype=torch.float16) * 0.1
        if e3m2:
            q = torch.empty(int(lib.pi05w4a4_q_e3m2_bytes(m, k)), dtype=torch.uint8, device=self.dev)
        else:
            q = torch.empty(int(lib.pi05w4a4_q_words(m, k)), dtype=torch.int32, device=self.dev)
        sa = torch.empty(m, dtype=torch.float32, device=self.dev)
        fn = lib.pi05w4a4_rmsnorm_quantize_e3m2 if e3m2 else lib.pi05w4a4_rmsnorm_quantize
        us = self._time(lambda: self._check(fn(P(x), P(w), 1e-6, 1, m, k, P(q), P(sa), self._stream())))
        nbytes = 2.0 * m * k + 2 * k + m * k * (0.75 if e3m2 else 0.5) + 4 * m
        gbs = nbytes / (us * 1e-6) / 1e9
        return {"m": m, "k": k, "avg_us": round(us, 3), "bytes": nbytes, "gbs": round(gbs, 1),
                "frac_hbm": round(gbs / HBM_PEAK_GBS, 4), "pair_offset_us": self.last_pair_offset_us}

    def gemm(self, m, k, ns, gelu=False, residual=False, copies=1, e3m2=False):
        """One W4A4 GEMM launch shape.  With `copies` > 1 (plain grouped GEMM only), that
        many weight sets are packed and the timed graph cycles through them, one set per
        launch, so that weights come from HBM rather than from the L2 / Infinity Cache.
        `e3m2`: the same codes in the E3M2 operand form (pi05w4a4_gemm_e3m2, FP6 MFMA)."""
        torch, lib, P = self.torch, self.lib, self.ext._ptr
        gen = torch.Generator(device=self.dev).manual_seed(20260923 + k + sum(ns))
        x = torch.randn(m, k, device=self.dev, dtype=torch.float16, generator=gen)
        if e3m2:
            q = torch.empty(int(lib.pi05w4a4_q_e3m2_bytes(m, k)), dtype=torch.uint8, device=self.dev)
        else:
            q = torch.empty(int(lib.pi05w4a4_q_words(m, k)), dtype=torch.int32, device=self.dev)
        sa = torch.empty(m, dtype=torch.float32, device=self.dev)
        quant = lib.pi05w4a4_quantize_e3m2 if e3m2 else lib.pi05w4a4_quantize
        self._check(quant(P(x), m, k, P(q), P(sa), self._stream()))
        if copies > 1 and (gelu or residual or e3m2):
            raise ValueError("weight copies are for the plain grouped INT4 GEMM")
        ws = [self._packed(n, k, gen) for n in ns]
        if e3m2:
            ws = [self.ext.repack_weight_e3m2(w, k=k) for w in ws]
        g = len(ns)
        n_arr = (ctypes.c_int32 * g)(*ns)
        wsb = 0 if e3m2 else int(lib.pi05w4a4_gemm_workspace_bytes(m, k, g, n_arr, 1 if gelu else 0))
        work = torch.empty(max(wsb, 16), dtype=torch.uint8, device=self.dev)
        if e3m2:
            w_arr = (ctypes.c_void_p * g)(*[w.data_ptr() for w in ws])
            outs = [torch.empty(m, n, dtype=torch.float16, device=self.dev) for n in (ns[:1] if gelu else ns)]
            y_arr = (ctypes.c_void_p * g)(*([outs[0].data_ptr(), None] if gelu else [o.data_ptr() for o in outs]))
            fn = lambda: self._check(lib.pi05w4a4_gemm_e3m2(  # noqa: E731
                P(q), P(sa), m, k, g, w_arr, n_arr, y_arr, 1 if gelu else 0, self._stream()))
            out_bytes = 2.0 * m * sum(o.size(1) for o in outs)
        elif gelu:
            out = torch.empty(m, ns[0], dtype=torch.float16, device=self.dev)
            fn = lambda: self._check(lib.pi05w4a4_gemm_gelu_up(  # noqa: E731
                P(q), P(sa), m, k, P(ws[0]), P(ws[1]), ns[0], P(out), P(work), wsb, self._stream()))
            out_bytes = 2.0 * m * ns[0]
        elif residual:
            res = torch.randn(m, ns[0], device=self.dev, dtype=torch.float16)
            out = torch.empty(m, ns[0], dtype=torch.float16, device=self.dev)
            fn = lambda: self._check(lib.pi05w4a4_gemm_residual(  # noqa: E731
                P(q), P(sa), m, k, P(ws[0]), ns[0], P(res), P(out), P(work), wsb, self._stream()))
            out_bytes = 4.0 * m * ns[0]
        else:
            outs = [torch.empty(m, n, dtype=torch.float16, device=self.dev) for n in ns]
            y_arr = (ctypes.c_void_p * g)(*[o.data_ptr() for o in outs])
            sets = [ws] + [[self._packed(n, k, gen) for n in ns] for _ in range(copies - 1)]
            w_arrs = [(ctypes.c_void_p * g)(*[w.data_ptr() for w in s]) for s in sets]
            turn = itertools.cycle(w_arrs)
            fn = lambda: self._check(lib.pi05w4a4_gemm_multi(  # noqa: E731
                P(q), P(sa), m, k, g, next(turn), n_arr, y_arr, P(work), wsb, self._stream()))
            out_bytes = 2.0 * m * sum(ns)
        us = self._time(fn, iters=copies if copies > 1 else None)
        n = sum(ns)
        ops = 2.0 * m * n * k
        nbytes = m * k / 2 + 4 * m + n * k / 2 + 4 * n + out_bytes
        tops = ops / (us * 1e-6) / 1e12
        rec = {"m": m, "k": k, "n": n, "avg_us": round(us, 3), "ops": ops, "tops": round(tops, 1),
               "frac_int8_peak": round(tops / INT8_PEAK_TOPS, 4), "bytes": nbytes,
               "gbs": round(nbytes / (us * 1e-6) / 1e9, 1), "workspace_bytes": wsb,
               "pair_offset_us": self.last_pair_offset_us}
        if e3m2:
            # The same int products on the FP6 MFMA, whose dense peak is twice the int8 one;
            # its operands take 1.5x the INT4 bytes.
            rec.update({"operands": "e3m2 (v_mfma_f32_16x16x128_f8f6f4)",
                        "frac_fp6_peak": round(tops / FP6_PEAK_TOPS, 4),
                        "operand_bytes": m * k * 0.75 + 4 * m + n * k * 0.75 + 4 * n + out_bytes})
        return rec


    def qkv_block(self, m, warm, copies=200, ns=(2048, 256, 256), k=2048, fused=False):
        """The QKV block of a decoder layer as launched: RMSNorm + quant, then the QKV GEMM,
        the timed graph cycling `copies` weight sets (from HBM, as in `gemm(copies=...)`).
        `warm`: the norm + quant launch reads the set its GEMM is about to use into the
        Infinity Cache (pi05w4a4_rmsnorm_quantize_warm).  `fused` (M <= 4): the one launch of
        pi05w4a4_quant_gemm_small instead, which quantizes inside the GEMM launch."""
        torch, lib, P = self.torch, self.lib, self.ext._ptr
        gen = torch.Generator(device=self.dev).manual_seed(20261202 + m)
        x = torch.randn(m, k, device=self.dev, dtype=torch.float16, generator=gen)
        nw = torch.randn(k, device=self.dev, dtype=torch.float16, generator=gen) * 0.1
        q = torch.empty(int(lib.pi05w4a4_q_words(m, k)), dtype=torch.int32, device=self.dev)
        sa = torch.empty(m, dtype=torch.float32, device=self.dev)
        g = len(ns)
        n_arr = (ctypes.c_int32 * g)(*ns)
        wsb = int(lib.pi05w4a4_gemm_workspace_bytes(m, k, g, n_arr, 0))
        work = torch.empty(max(wsb, 16), dtype=torch.uint8, device=self.dev)
        outs = [torch.empty(m, n, dtype=torch.float16, device=self.dev) for n in ns]
        y_arr = (ctypes.c_void_p * g)(*[o.data_ptr() for o in outs])
        sets = [[self._packed(n, k, gen) for n in ns] for _ in range(copies)]
        w_arrs = [(ctypes.c_void_p * g)(*[w.data_ptr() for w in s]) for s in sets]
        warm_bytes = (ctypes.c_size_t * g)(*[w.numel() * w.element_size() for w in sets[0]])
        turn = itertools.cycle(range(copies))

        def fn():
            i = next(turn)
            if fused:
                self._check(lib.pi05w4a4_quant_gemm_small(P(x), P(nw), 1e-6, 1, m, k, g, w_arrs[i], n_arr, y_arr,
                                                          None, self._stream()))
                return
            if warm:
                self._check(lib.pi05w4a4_rmsnorm_quantize_warm(P(x), P(nw), 1e-6, 1, m, k, P(q), P(sa), w_arrs[i],
                                                               warm_bytes, g, self._stream()))
            else:
                self._check(lib.pi05w4a4_rmsnorm_quantize(P(x), P(nw), 1e-6, 1, m, k, P(q), P(sa), self._stream()))
            self._check(lib.pi05w4a4_gemm_multi(P(q), P(sa), m, k, g, w_arrs[i], n_arr, y_arr, P(work), wsb,
                                                self._stream()))

        return round(self._time(fn, iters=copies), 3)

    def gelu_quant(self, m, k=2048, n=16384, fused=True):
        """Gate/up with the GELU-tanh*up epilogue and the down projection's activation quant
        of its output: one launch (pi05w4a4_gemm_gelu_up_quant) or, with fused=False, the
        GEMM then pi05w4a4_quantize (two launches)."""
        torch, lib, P = self.torch, self.lib, self.ext._ptr
        gen = torch.Generator(device=self.dev).manual_seed(20261203 + m)
        x = torch.randn(m, k, device=self.dev, dtype=torch.float16, generator=gen)
        q = torch.empty(int(lib.pi05w4a4_q_words(m, k)), dtype=torch.int32, device=self.dev)
        sa = torch.empty(m, dtype=torch.float32, device=self.dev)
        self._check(lib.pi05w4a4_quantize(P(x), m, k, P(q), P(sa), self._stream()))
        wg, wu = self._packed(n, k, gen), self._packed(n, k, gen)
        h = torch.empty(m, n, dtype=torch.float16, device=self.dev)
        dq = torch.empty(int(lib.pi05w4a4_q_words(m, n)), dtype=torch.int32, device=self.dev)
        dsa = torch.empty(m, dtype=torch.float32, device=self.dev)
        ctl = torch.zeros(int(lib.pi05w4a4_mlp_ctl_words(m)), dtype=torch.int32, device=self.dev)
        if fused:
            fn = lambda: self._check(lib.pi05w4a4_gemm_gelu_up_quant(  # noqa: E731
                P(q), P(sa), m, k, P(wg), P(wu), n, P(h), P(dq), P(dsa), P(ctl), None, None, 0, 0, 0,
                self._stream()))
        else:
            def fn():
                self._check(lib.pi05w4a4_gemm_gelu_up(P(q), P(sa), m, k, P(wg), P(wu), n, P(h), None, 0,
                                                      self._stream()))
                self._check(lib.pi05w4a4_quantize(P(h), m, n, P(dq), P(dsa), self._stream()))
        us = self._time(fn)
        if lib.pi05w4a4_mlp_status(0) != 0:
            raise RuntimeError("a bounded wait of the fused gate/up + down quant ran out")
        ops = 2.0 * m * 2 * n * k
        return {"m": m, "k": k, "n": 2 * n, "avg_us": round(us, 3), "ops": ops, "launches": 1 if fused else 2,
                "tops": round(ops / (us * 1e-6) / 1e12, 1), "pair_offset_us": self.last_pair_offset_us}

    def qkv_rope(self, b, s, h=2048):
        """The QKV GEMMs with RoPE and the attention's K/V layout in the epilogue
        (pi05w4a4_gemm_qkv_rope, one KV head of 256) at B x S tokens."""
        torch, lib, P = self.torch, self.lib, self.ext._ptr
        m = b * s
        gen = torch.Generator(device=self.dev).manual_seed(20261202 + m)
        x = torch.randn(m, h, device=self.dev, dtype=torch.float16, generator=gen)
        q = torch.empty(int(lib.pi05w4a4_q_words(m, h)), dtype=torch.int32, device=self.dev)
        sa = torch.empty(m, dtype=torch.float32, device=self.dev)
        self._check(lib.pi05w4a4_quantize(P(x), m, h, P(q), P(sa), self._stream()))
        wq, wk, wv = (self._packed(n, h, gen) for n in (2048, 256, 256))
        wk = self.ext.rope_pair_weight(wk)
        cos = torch.rand(m, 256, device=self.dev, generator=gen).half()
        sin = torch.rand(m, 256, device=self.dev, generator=gen).half()
        yq = torch.empty(m, 2048, dtype=torch.float16, device=self.dev)
        kr = torch.empty(m, 256, dtype=torch.float16, device=self.dev)
        yv = torch.empty(m, 256, dtype=torch.float16, device=self.dev)
        kv = torch.empty(int(lib.pi05w4a4_attn_kv_mfma_elems(b, s, 1, 256)), dtype=torch.float16, device=self.dev)
        us = self._time(lambda: self._check(lib.pi05w4a4_gemm_qkv_rope(
            P(q), P(sa), m, h, P(wq), 2048, P(wk), P(wv), P(cos), P(sin), b, s, P(yq), P(kr), P(yv), P(kv),
            self._stream())))
        ops = 2.0 * m * 2560 * h
        return {"m": m, "k": h, "n": 2560, "avg_us": round(us, 3), "ops": ops,
                "tops": round(ops / (us * 1e-6) / 1e12, 1), "pair_offset_us": self.last_pair_offset_us}

    def attention(self, b, s, h=8, kvh=1):
        """The two prefix-attention kernels (K RoPE + V transpose, then attention) at one
        decoder layer's shapes, zero additive mask."""
        torch, lib, P = self.torch, self.lib, self.ext._ptr
        d = 256
        gen = torch.Generator(device=self.dev).manual_seed(7)
        q = torch.randn(b, s, h * d, device=self.dev, generator=gen).half()
        k = torch.randn(b, s, kvh * d, device=self.dev, generator=gen).half()
        v = torch.randn(b, s, kvh * d, device=self.dev, generator=gen).half()
        ang = torch.rand(b, s, d, device=self.dev, generator=gen) * 6.28
        cos, sin = ang.cos().half(), ang.sin().half()
        s4 = (s + 3) // 4 * 4
        mask = torch.zeros(b, s, s4, dtype=torch.float16, device=self.dev)
        k_rope = torch.empty(b, kvh, s, d, dtype=torch.float16, device=self.dev)
        kvm = torch.empty(int(lib.pi05w4a4_attn_kv_mfma_elems(b, s, kvh, d)), dtype=torch.float16, device=self.dev)
        out = torch.empty(b, s, h * d, dtype=torch.float16, device=self.dev)
        prep = lambda: self._check(lib.pi05w4a4_attn_kv_prep(  # noqa: E731
            P(k), P(v), kvh * d, P(cos), P(sin), b, s, kvh, d, P(k_rope), P(kvm), self._stream()))
        attn = lambda: self._check(lib.pi05w4a4_prefix_attention(  # noqa: E731
            P(q), h * d, P(kvm), P(cos), P(sin), P(mask), s * s4, s4, s4, d**-0.5,
            b, s, h, kvh, d, P(out), h * d, None, None, self._stream()))
        prep()
        us_prep = self._time(prep)
        us_attn = self._time(attn)
        attn_offset = self.last_pair_offset_us
        flops = 4.0 * b * h * s * s * d
        s_pad = (s + 63) // 64 * 64
        # Bytes that cross each workgroup's vector-memory path: every workgroup streams all
        # of K and V (keys x 2 x 512 B) plus its 32 query rows (and cos/sin) once per wave.
        wgs = b * kvh * -(-(s * h // kvh) // 32)
        per_wg = 2.0 * s_pad * d * 2 + 4 * 32 * d * 2 * 3 + 4 * 32 * s_pad * 2 / 4
        tflops = flops / (us_attn * 1e-6) / 1e12
        return {
            "attention": {"b": b, "s": s, "h": h, "kvh": kvh, "avg_us": round(us_attn, 3), "flops": flops,
                          "tflops": round(tflops, 2), "frac_fp16_peak": round(tflops / FP16_PEAK_TFLOPS, 4),
                          "workgroups": wgs, "bytes_per_workgroup": per_wg, "pair_offset_us": attn_offset,
                          "l2_to_cu_gbs": round(wgs * per_wg / (us_attn * 1e-6) / 1e9, 1)},
            "attn_kv_prep": {"avg_us": round(us_prep, 3),
                             "bytes": 2.0 * b * s * kvh * d * 2 * 2 + 2.0 * b * s * d * 2},
        }

    def rmsnorm(self, m, k=2048):
        torch, lib, P = self.torch, self.lib, self.ext._ptr
        x = torch.randn(m, k, device=self.dev, dtype=torch.float16)
        w = torch.randn(k, device=self.dev, dtype=torch.float16)
        y = torch.empty_like(x)
        us = self._time(lambda: self._check(lib.pi05w4a4_rmsnorm(P(x), P(w), 1e-6, 1, m, k, P(y), self._stream())))
        nbytes = 4.0 * m * k + 2 * k
        return {"m": m, "k": k, "avg_us": round(us, 3), "bytes": nbytes,
                "frac_hbm": round(nbytes / (us * 1e-6) / 1e9 / HBM_PEAK_GBS, 4)}


def forward_point(torch, model, prefix_inputs, dev, tokens: int, batch: int, steps: int) -> dict:
    """ms per graph-replayed forward at another prefix length / batch (same model)."""
    x = prefix_inputs(batch, tokens, dev)
    mask = torch.zeros(batch, 1, tokens, tokens, dtype=torch.float16, device=dev)
    model(x, mask)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        model(x, mask)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        model(x, mask)
    for _ in range(3):
        graph.replay()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        graph.replay()
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t0) * 1e3 / steps
    del graph
    return {"tokens": tokens, "batch": batch, "ms_per_forward": round(ms, 4),
            "tokens_per_s": round(tokens * batch / ms * 1e3, 1)}


def _in_forward_label(fn_name: str, args: tuple, kwargs: dict) -> str:
    """Kernel class of one library call made by the forward."""
    if fn_name == "_gemm_e3m2_from_q":
        return "gate_up_gelu" if kwargs.get("gelu") else ("gate_up" if len(args[3]) == 2 else "gemm")
    if fn_name == "quantize_e3m2":
        return "rmsnorm_quant_k2048" if len(args) > 1 and args[1] is not None else "quant_k2048"
    if fn_name == "_gemm_from_q":
        k, weights = args[2], args[3]
        if kwargs.get("gelu"):
            return "gate_up_gelu"
        if kwargs.get("residual") is not None:
            return "down_residual" if k == 16384 else "o_residual"
        return {3: "qkv", 2: "gate_up"}.get(len(weights), "gemm")
    if fn_name == "quantize":
        return f"quant_k{int(args[0].size(-1))}"
    if fn_name == "rms_norm_quantize":
        return "rmsnorm_quant_k2048"
    if fn_name == "_gemm_qkv_rope":
        return "qkv_rope"
    if fn_name == "_gemm_gelu_quant_from_q":
        return "gate_up_gelu_quant"
    return "attention" if kwargs.get("kv_mfma") is not None else "attention_with_kv_prep"


def in_forward_times(torch, ext, model, x, mask, reps: int = 5) -> dict:
    """Per-kernel GPU time inside the real forward: the eager forward runs with HIP events
    recorded on the launching stream around each library call (GEMM launches, activation
    quants, the two attention kernels).  A bounded spin kernel (torch.cuda._sleep) queued
    ahead of each forward holds the GPU until the host has enqueued the whole forward, so
    the kernels run back to back with no host gaps, in the cache state the forward leaves
    them (preceding kernels, weight cache warming) and the event pairs time the kernels
    alone.  `raw_avg_us` is the mean pair interval; `calibrate_in_forward` takes off it
    the event-pair cost that the same kernel shows when launched alone (`avg_us`)."""
    names = ("_gemm_from_q", "quantize", "rms_norm_quantize", "_prefix_attention_impl", "_gemm_qkv_rope",
             "_gemm_gelu_quant_from_q", "_gemm_e3m2_from_q", "quantize_e3m2")
    orig = {n: getattr(ext, n) for n in names}
    records = []

    def wrap(name):
        fn = orig[name]

        def timed(*args, **kwargs):
            e0 = torch.cuda.Event(enable_timing=True)
            e1 = torch.cuda.Event(enable_timing=True)
            e0.record()
            out = fn(*args, **kwargs)
            e1.record()
            records.append((_in_forward_label(name, args, kwargs), e0, e1))
            return out

        return timed

    # spin length: calibrate cycles -> ms, aim at twice the host enqueue time
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    torch.cuda._sleep(1_000_000)
    e1.record()
    torch.cuda.synchronize()
    ms_per_mcycle = max(e0.elapsed_time(e1), 1e-3)
    for n in names:
        setattr(ext, n, wrap(n))
    primed = True
    try:
        t0 = time.perf_counter()
        model(x, mask)
        torch.cuda.synchronize()
        enqueue_ms = (time.perf_counter() - t0) * 1e3
        spin_ms = min(4.0 * enqueue_ms + 5.0, 200.0)
        records.clear()
        for _ in range(reps):
            torch.cuda.synchronize()
            torch.cuda._sleep(int(spin_ms / ms_per_mcycle * 1e6))
            t0 = time.perf_counter()
            model(x, mask)
            host_ms = (time.perf_counter() - t0) * 1e3
            torch.cuda.synchronize()
            primed = primed and host_ms < spin_ms
    finally:
        for n in names:
            setattr(ext, n, orig[n])
    # An event pair costs time of its own (two marker packets on the queue; an empty pair's
    # interval is reported as event_pair_us), but how much of it adds to a kernel's
    # interval depends on the kernel: calibrate_in_forward corrects each class with its
    # own isolated launches.
    torch.cuda.synchronize()
    torch.cuda._sleep(int(10.0 / ms_per_mcycle * 1e6))
    empty = []
    for _ in range(200):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        b.record()
        empty.append((a, b))
    torch.cuda.synchronize()
    pair_us = statistics.median(a.elapsed_time(b) * 1e3 for a, b in empty)
    per = {}
    for label, a, b in records:
        per.setdefault(label, []).append(a.elapsed_time(b) * 1e3)
    out = {lab: {"calls_per_forward": len(v) // reps, "raw_avg_us": round(statistics.fmean(v), 3)}
           for lab, v in per.items()}
    return {"kernels": out, "reps": reps, "queue_primed": primed, "spin_ms": round(spin_ms, 2),
            "event_pair_us": round(pair_us, 3)}


_KERNEL_CLASS_RULES = (
    # (regex on the kernel name as the profiler reports it, demangled or mangled) -> class
    (r"fwht_quant_kernel(?:<14,|ILi14E)", "quant_k16384"),
    (r"fwht_quant_kernel(?:<11, 6, 4, true[,>]|ILi11ELi6ELi4ELb1E)", "rmsnorm_quant_k2048"),
    (r"fwht_quant_kernel(?:<11,|ILi11E)", "quant_k2048"),
    (r"prefix_attention_(?:wide_)?kernel", "attention"),
    (r"kv_prep_kernel", "attn_kv_prep"),
    (r"rmsnorm_kernel", "rmsnorm"),
)


def _gemm_template_args(name: str) -> list[int] | None:
    """The template arguments of a gemm_w4a4_kernel instance, from its demangled
    (``<7, 4, 4, 1, true, ...>``) or mangled (``ILi7ELi4E...Lb1E...``) name: ints, with
    booleans as 0 / 1.  None for other kernels."""
    m = re.search(r"gemm_w4a4_kernel<([^>]*)>", name)
    if m:
        return [1 if a.strip() == "true" else 0 if a.strip() == "false" else int(a) for a in m.group(1).split(",")]
    m = re.search(r"gemm_w4a4_kernelI((?:L[ib]\d+E)+)E", name)
    if m:
        return [int(v) for v in re.findall(r"L[ib](\d+)E", m.group(1))]
    return None


def kernel_class(name: str) -> str:
    """Kernel class of a profiled kernel name.  gemm_w4a4_kernel<MI, NI, NWAVES, KW, GELU,
    RING, WPE, QKV_PREP, QFUSE, E3M2, QPRO, NKB>: the 776-token forward's GEMMs by their tile
    configuration and epilogue."""
    a = _gemm_template_args(name)
    if a is not None:
        mi, ni, nwaves, kw, gelu = a[:5]
        qkv_prep = len(a) > 7 and a[7] == 1
        qfuse = len(a) > 8 and a[8] == 1
        if gelu:
            return "gate_up_gelu_quant" if qfuse else "gate_up_gelu"
        if qkv_prep:
            return "qkv_rope"
        if kw == 8:
            return "down_residual"
        if (mi, ni, nwaves, kw) == (7, 4, 4, 1):
            return "gate_up"
        if (mi, ni, nwaves, kw) in ((2, 2, 4, 1), (4, 4, 4, 4)):
            return "o_residual"
        return "gemm"
    return next((c for rx, c in _KERNEL_CLASS_RULES if re.search(rx, name)), "other")


def profiled_in_forward(torch, replay, reps: int = 10, warm_s: float = 0.5) -> dict | None:
    """Per-kernel device time inside the graph-replayed forward, from the kernels' own
    begin/end timestamps as torch.profiler (roctracer) records them, the source rocprofv3's
    kernel trace reads too: no markers between the kernels.  After ~warm_s seconds of
    replays (clocks settle), `reps` replays are profiled; each class's mean duration and
    launches per forward are reported.  None if the profiler records no kernels."""
    import collections

    from torch.profiler import ProfilerActivity, profile

    t0 = time.perf_counter()
    while time.perf_counter() - t0 < warm_s:
        replay()
        torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        for _ in range(reps):
            replay()
        torch.cuda.synchronize()
    per = collections.defaultdict(list)
    for e in prof.events():
        if e.device_type != torch.autograd.DeviceType.CUDA:
            continue
        dur = getattr(e, "device_time_total", None)
        if dur is None:
            dur = e.cuda_time_total
        label = kernel_class(e.name)
        per[label].append(float(dur))
    if not per:
        return None
    out = {lab: {"calls_per_forward": len(v) // reps, "profiled_avg_us": round(statistics.fmean(v), 3),
                 "profiled_us_per_forward": round(sum(v) / reps, 2)} for lab, v in per.items()}
    total = sum(sum(v) for v in per.values()) / reps
    return {"kernels": out, "reps": reps, "profiled_kernel_us_per_forward": round(total, 2),
            "method": "torch.profiler kernel timestamps over graph replays, normalised to the unprofiled forward"}


def normalise_profiled(prof_fwd: dict, forward_ms: float) -> None:
    """Under the profiler every kernel of the forward runs a few % slower, about uniformly
    (measured against a rocprofv3 kernel trace of the same forward: +2 to +7% per class,
    while rocprof's own per-forward kernel sum equals the unprofiled replay time).  The
    per-class times are scaled so that the forward's kernels sum to the unprofiled
    graph-replay time (`forward_ms`, less the idle gaps the profile shows none of)."""
    scale = forward_ms * 1e3 / prof_fwd["profiled_kernel_us_per_forward"]
    prof_fwd["scale"] = round(scale, 4)
    for rec in prof_fwd["kernels"].values():
        rec["avg_us"] = round(rec["profiled_avg_us"] * scale, 3)
        rec["us_per_forward"] = round(rec["profiled_us_per_forward"] * scale, 2)


def calibrate_in_forward(in_fwd: dict, offsets: dict) -> None:
    """avg_us of each in-forward kernel class = its raw event-pair interval less the
    event-pair cost its kernel shows alone (pair interval of an eager launch minus the
    graph-timed launch, `pair_offset_us` of the kernel table; the attention class uses the
    prefix-attention kernel's).  Classes without a calibration keep the raw interval."""
    for label, rec in in_fwd["kernels"].items():
        off = offsets.get(label)
        rec["pair_offset_us"] = off
        rec["avg_us"] = round(rec["raw_avg_us"] - (off or 0.0), 3)


def kernel_table(kb: KernelBench, m: int, only: str = "") -> dict:
    h, inter = 2048, 16384
    jobs = {
        "quant_k2048": lambda: kb.quant(m, h),
        "quant_k16384": lambda: kb.quant(m, inter),
        "qkv": lambda: kb.gemm(m, h, [2048, 256, 256]),
        "o": lambda: kb.gemm(m, h, [2048]),
        # gate/up as the forward runs it: E3M2 operands (the load-time default) unless
        # PI05_W4A4_E3M2=0; the INT4 kernels beside them
        "gate_up": lambda: kb.gemm(m, h, [inter, inter], e3m2=E3M2_GATE_UP),
        "gate_up_gelu": lambda: kb.gemm(m, h, [inter, inter], gelu=True, e3m2=E3M2_GATE_UP),
        "gate_up_int4": lambda: kb.gemm(m, h, [inter, inter]),
        "gate_up_gelu_int4": lambda: kb.gemm(m, h, [inter, inter], gelu=True),
        "down": lambda: kb.gemm(m, inter, [h]),
        "o_residual": lambda: kb.gemm(m, h, [2048], residual=True),
        "down_residual": lambda: kb.gemm(m, inter, [h], residual=True),
        "rmsnorm_quant_k2048": lambda: kb.rmsnorm_quant(m),
        "rmsnorm_quant_e3m2": lambda: kb.rmsnorm_quant(m, e3m2=True),
        "qkv_rope": lambda: kb.qkv_rope(1, m),
        "gate_up_gelu_quant": lambda: kb.gelu_quant(m),
        "gate_up_gelu_then_quant": lambda: kb.gelu_quant(m, fused=False),
    }

    def copy():  # calibration for the HBM traffic counters: a plain 64 MiB copy
        src = kb.torch.empty(64 << 20, dtype=kb.torch.uint8, device=kb.dev).fill_(1)
        dst = kb.torch.empty_like(src)
        us = kb._time(lambda: dst.copy_(src))
        return {"bytes_read": float(64 << 20), "bytes_written": float(64 << 20), "avg_us": round(us, 3)}

    if only:  # one class or a comma-separated list (also "copy", "qkv_m_sweep")
        extra = {"copy": copy, "qkv_m_sweep": lambda: qkv_m_sweep(kb)}
        return {name: {**jobs, **extra}[name]() for name in only.split(",")}
    return {name: fn() for name, fn in jobs.items()}


def qkv_m_sweep(kb: KernelBench, ms=(1, 4, 64, 640, 776)) -> dict:
    """The fused QKV projection (int4_gemm3: one activation quant, N = 2048 + 256 + 256,
    K = 2048) and its RMSNorm + quant over a range of token counts, down to the
    weight-streaming regime of M = 1 and 64.  `hot`: the same weights every launch (they
    stay in the L2 / Infinity Cache); `cold`: each launch of the timed graph reads its own
    copy of the 2.6 MB of packed weights (200 copies, 0.5 GB, beyond the 256 MB Infinity
    Cache), as a forward that streams every layer's weights once does."""
    out = {}
    wbytes = 2560 * (2048 // 2 + 4)
    for m in ms:
        hot = kb.gemm(m, 2048, [2048, 256, 256])
        cold = kb.gemm(m, 2048, [2048, 256, 256], copies=200)
        nq = kb.rmsnorm_quant(m)
        out[str(m)] = {
            "gemm_hot_us": hot["avg_us"], "gemm_hot_tops": hot["tops"],
            "gemm_cold_us": cold["avg_us"], "gemm_cold_tops": cold["tops"],
            "frac_int8_peak_cold": cold["frac_int8_peak"],
            "bytes": cold["bytes"], "weight_bytes": wbytes,
            "gemm_cold_gbs": cold["gbs"], "frac_hbm_cold": round(cold["gbs"] / HBM_PEAK_GBS, 4),
            "rmsnorm_quant_us": nq["avg_us"],
            "block_cold_us": round(cold["avg_us"] + nq["avg_us"], 3),
            # the two launches back to back in one graph, without and with the norm + quant
            # launch warming the weights of its GEMM
            "block_cold_pair_us": kb.qkv_block(m, warm=False),
            "block_cold_warm_us": kb.qkv_block(m, warm=True),
        }
        if m <= 4:
            # the one-launch form the ops take at these sizes (norm + quant inside the GEMM)
            out[str(m)]["block_cold_fused_us"] = kb.qkv_block(m, warm=False, fused=True)
    return out


def read_traffic(kernel: str) -> tuple[float | None, str | None]:
    """HBM bytes per launch of a kernel class from the committed rocprofv3 summary."""
    path = TRAFFIC_FILE
    if not path.is_file():
        return None, None
    m = re.search(rf"traffic_bytes_per_launch\[{kernel}\]:\s*([0-9.eE+]+)", path.read_text())
    if not m:
        return None, None
    return float(m.group(1)), str(path.relative_to(ROOT))


# ----------------------------------------------------------------------------- CPU baseline
def _cpu_model() -> str:
    try:
        for line in Path("/proc/cpuinfo").read_text().splitlines():
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(tokens: int, batch: int, layers: int, budget_s: float) -> dict:
    """The reference's W4A4 semantics on the host CPU with PyTorch (oracle/w4a4_torch_cpu.py,
    the restatement of pack.py:113-145): per projection call, fp32 FWHT + per-token INT4
    quant, unpack of the packed weights, exact integer matmul, fp16 dequant -- one decoder
    layer's calls at M = tokens * batch (QKV with one shared quant, o, gate/up with one shared
    quant, down), each timed with both integer matmul forms (the reference's fp32
    ``a @ b.T`` and ``torch._int_mm``): 2 warm-up calls, then the median of up to 5 calls.
    The faster form of each call is summed and scaled to ``layers`` layers."""
    import torch

    from oracle import w4a4_torch_cpu as tcpu

    torch.set_num_threads(os.cpu_count() or 1)
    m = tokens * batch
    gen = torch.Generator().manual_seed(20260923 + 4)

    def act(k: int, geglu: bool = False) -> torch.Tensor:
        if geglu:
            g = torch.randn(m, k, generator=gen)
            return (torch.nn.functional.gelu(g, approximate="tanh") * torch.randn(m, k, generator=gen)).half()
        x = torch.randn(m, k, generator=gen)
        x[:, torch.randperm(k, generator=gen)[: max(1, k // 100)]] *= 20.0
        return x.half()

    def packed(n: int, k: int) -> torch.Tensor:
        # codes ~ round(N(0, 2)) in [-7, 7] (a packed N(0, 0.02) weight's statistics), scale 0.01
        codes = torch.randn(n, k, generator=gen).mul_(2.0).round_().clamp_(-7, 7).to(torch.int32) & 0xF
        words = torch.zeros(n, k // 8, dtype=torch.int32)
        c = codes.view(n, k // 8, 8)
        for j in range(8):
            words |= c[..., j] << (4 * j)
        scale = torch.full((n, 1), 0.01, dtype=torch.float32).view(torch.int32)
        return torch.cat([words, scale], dim=1)

    calls = [("qkv", act(2048), [packed(2048, 2048), packed(256, 2048), packed(256, 2048)]),
             ("o", act(2048), [packed(2048, 2048)]),
             ("gate_up", act(2048), [packed(16384, 2048), packed(16384, 2048)]),
             ("down", act(16384, geglu=True), [packed(2048, 16384)])]
    per_gemm = {}
    t_start = time.perf_counter()
    for name, x, ws in calls:
        row = {}
        for method in ("fp32", "int_mm"):
            fn = lambda: tcpu.int4_gemm_ref(x, ws, method)  # noqa: E731
            fn()
            t0 = time.perf_counter()
            fn()
            one = time.perf_counter() - t0
            reps = 5 if one * 5 < budget_s / 8 else 3
            times = []
            for _ in range(reps):
                t0 = time.perf_counter()
                fn()
                times.append(time.perf_counter() - t0)
            row[method] = round(statistics.median(times) * 1e3, 2)
        row["best"] = min(("fp32", "int_mm"), key=lambda k_: row[k_])
        per_gemm[name] = row
    per_layer_ms = sum(r[r["best"]] for r in per_gemm.values())
    return {
        "value": round(per_layer_ms * layers, 1),
        "unit": "ms",
        "cores": torch.get_num_threads(),
        "kind": "port",
        "sample": (
            f"one decoder layer's W4A4 projection calls at M={m} (QKV and gate/up with one shared "
            f"activation quant each, o, down), each: fp32 FWHT + INT4 quant, weight unpack, exact "
            f"integer matmul, fp16 dequant (pack.py:113-145 semantics in PyTorch CPU); the faster of "
            f"the fp32 and torch._int_mm matmul per call, x {layers} layers; attention and norms not "
            f"included; {round(time.perf_counter() - t_start, 1)} s of CPU timing"
        ),
        "cpu_model": _cpu_model(),
        "os_cpu_count": os.cpu_count(),
        "torch_threads": torch.get_num_threads(),
        "per_gemm_ms": per_gemm,
        "per_layer_ms": round(per_layer_ms, 2),
    }


# ----------------------------------------------------------------------------- main
def main() -> int:
    args = parse_args()
    if args.gpus != 1:
        print(
            f"bench.py runs on one GPU only (asked for --gpus {args.gpus}); the W4A4 path is "
            "measured at one GPU's share, multi-GPU sharding is design-only.",
            file=sys.stderr,
        )
        return 2

    import torch

    from pi05_fast.w4a4 import extension as ext

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    ext.preload()
    m = args.tokens * args.batch
    kb = KernelBench(torch, ext, dev, args.kernel_iters, args.kernel_warmup_s)
    if args.only_kernel:
        print(json.dumps(kernel_table(kb, m, args.only_kernel)), flush=True)
        return 0

    from pi05_fast.w4a4.prefix_lm import build_prefix_lm, prefix_inputs, prefix_ops

    os.environ["PI05_W4A4_FUSE_GELU"] = "0" if args.unfused_gelu else "1"
    model, _ = build_prefix_lm(dev, num_layers=args.layers)
    x = prefix_inputs(args.batch, args.tokens, dev)
    s = args.tokens
    # Prefix-LM mask over the prefix: every prefix token sees every other one (additive 4D).
    mask = torch.zeros(args.batch, 1, s, s, dtype=torch.float16, device=dev)

    with torch.no_grad():
        y_eager = model(x, mask)
        torch.cuda.synchronize()
        graph = None
        if not args.no_graph:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                for _ in range(2):
                    model(x, mask)
            torch.cuda.current_stream().wait_stream(side)
            graph = torch.cuda.CUDAGraph()
            try:
                with torch.cuda.graph(graph):
                    y_graph = model(x, mask)
            except Exception as exc:  # capture unsupported: time eager forwards instead
                print(f"bench: graph capture failed ({exc!r}); timing eager forwards", file=sys.stderr)
                graph = None
                torch.cuda.synchronize()
        graph_exact = None
        if graph is not None:
            # Replays interleaved with eager work must all give the same output, and that
            # output must match the eager forward.
            first = None
            for i in range(3):
                graph.replay()
                torch.cuda.synchronize()
                if first is None:
                    first = y_graph.clone()
                    graph_exact = bool(torch.equal(first, y_eager))
                    err = ((first.float() - y_eager.float()).norm() / y_eager.float().norm()).item()
                    if not err <= 1e-3:
                        raise RuntimeError(f"graph replay differs from the eager forward (rel_l2={err:.3e})")
                elif not torch.equal(y_graph, first):
                    raise RuntimeError(f"graph replay {i} differs from replay 0")
                model(x, mask)
                torch.cuda.synchronize()

        # Eager forwards, for reference (host-dispatch bound).
        torch.cuda.synchronize()
        n_eager = max(3, args.steps // 4)
        t0 = time.perf_counter()
        for _ in range(n_eager):
            model(x, mask)
        torch.cuda.synchronize()
        eager_ms = (time.perf_counter() - t0) * 1e3 / n_eager
        in_fwd = None if args.forward_only else in_forward_times(torch, ext, model, x, mask)
        prof_fwd = None
        if not args.forward_only and graph is not None:
            try:
                prof_fwd = profiled_in_forward(torch, graph.replay)
            except Exception as exc:  # profiler unavailable: the event-pair figures stand
                print(f"bench: torch.profiler failed ({exc!r})", file=sys.stderr)

        def step():
            if graph is not None:
                graph.replay()
            else:
                model(x, mask)

        for _ in range(args.warmup):
            step()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.steps):
            step()
        torch.cuda.synchronize()
        ms = (time.perf_counter() - t0) * 1e3 / args.steps
        if prof_fwd is not None:
            normalise_profiled(prof_fwd, ms)
        del graph
        if args.forward_only:
            print(json.dumps({"forward_only": True, "ms_per_forward": round(ms, 4), "steps": args.steps,
                              "graph_replay_bit_exact_vs_eager": graph_exact}), flush=True)
            return 0

        kernels = kernel_table(kb, m)
        sweep = qkv_m_sweep(kb)
        others = kb.attention(args.batch, args.tokens)
        others["rmsnorm"] = kb.rmsnorm(m)
        offsets = {name: rec.get("pair_offset_us") for name, rec in kernels.items()}
        offsets["attention"] = others["attention"]["pair_offset_us"]
        offsets["attention_with_kv_prep"] = others["attention"]["pair_offset_us"]
        calibrate_in_forward(in_fwd, offsets)
        if prof_fwd is not None:
            # The profiler's timestamps are the in-forward figures; the calibrated event
            # pairs stay beside them for comparison.
            events = in_fwd
            in_fwd = prof_fwd
            in_fwd["event_pairs"] = events

        # The other prefix lengths and the batch-8 throughput point of the same workload,
        # and the 776-token forward with transformers' fp16 eager attention instead of the
        # prefix-attention kernels (everything else unchanged).
        points = {}
        if not args.no_extra_points:
            for tok, bat in ((640, 1), (768, 1), (776, 8)):
                points[f"{tok}x{bat}"] = forward_point(torch, model, prefix_inputs, dev, tok, bat, 10)
            old = os.environ.get("PI05_W4A4_FUSE_ATTN")
            os.environ["PI05_W4A4_FUSE_ATTN"] = "0"
            try:
                p = forward_point(torch, model, prefix_inputs, dev, args.tokens, args.batch, 10)
            finally:
                if old is None:
                    del os.environ["PI05_W4A4_FUSE_ATTN"]
                else:
                    os.environ["PI05_W4A4_FUSE_ATTN"] = old
            p["attention"] = "transformers fp16 eager (PI05_W4A4_FUSE_ATTN=0)"
            points[f"{args.tokens}x{args.batch}_eager_attention"] = p

    ops = prefix_ops(args.tokens, args.batch, args.layers)
    total_ops = sum(ops.values())
    # The W4A4 kernels one decoder layer launches (fused layer: RMSNorm in the QKV and
    # gate/up quants, the o-proj quant inside the attention kernel, residual adds in the o
    # and down epilogues).
    fused_kv = os.environ.get("PI05_W4A4_FUSE_KV", "1") != "0" and args.tokens % 8 == 0
    calls = {"rmsnorm_quant_k2048": 1 if E3M2_GATE_UP else 2, "rmsnorm_quant_e3m2": 1 if E3M2_GATE_UP else 0,
             "quant_k2048": 0, "quant_k16384": 1, "qkv": 0 if fused_kv else 1,
             "qkv_rope": 1 if fused_kv else 0, "o_residual": 1, "down_residual": 1, "gate_up_gelu": 1, "gate_up": 0,
             "o": 0, "down": 0}
    if args.unfused_gelu:
        calls.update({"rmsnorm_quant_k2048": 0, "rmsnorm_quant_e3m2": 0, "quant_k2048": 3, "qkv": 1, "qkv_rope": 0,
                      "o_residual": 0,
                      "down_residual": 0, "gate_up_gelu": 0, "gate_up": 1, "o": 1, "down": 1})
    for name, c in calls.items():
        kernels[name]["calls_per_layer"] = c
    w4a4_us_per_layer = sum(kernels[n]["avg_us"] * c for n, c in calls.items())
    # The dominant kernel of the forward: the gate/up GEMM as the forward launches it (with
    # the fused GELU-tanh*up epilogue unless --unfused-gelu).
    dk_name = "gate_up" if args.unfused_gelu else "gate_up_gelu"
    dk = kernels[dk_name]
    traffic, traffic_src = read_traffic(dk_name)
    fwd_dk = in_fwd["kernels"].get(dk_name)
    in_forward_roof = None
    if fwd_dk is not None:
        tops_fwd = dk["ops"] / (fwd_dk["avg_us"] * 1e-6) / 1e12
        in_forward_roof = {"avg_launch_us": fwd_dk["avg_us"], "achieved": round(tops_fwd, 1),
                           "frac": round(tops_fwd / INT8_PEAK_TOPS, 4),
                           "calls_per_forward": fwd_dk["calls_per_forward"]}
    roofline = {
        "bound": "mfma",
        "achieved": dk["tops"],
        "peak": INT8_PEAK_TOPS,
        "unit": "TFLOP/s",
        "frac": round(dk["tops"] / INT8_PEAK_TOPS, 4),
        "traffic": traffic,
        "kernel": ("gemm_w4a4_kernel (gate/up, int4_gemm2)" if args.unfused_gelu
                   else "gemm_w4a4_kernel (gate/up + GELU-tanh*up epilogue, int4_gemm2_gelu)")
                  + (", E3M2 operands on the FP6 MFMA (v_mfma_f32_16x16x128_f8f6f4)" if E3M2_GATE_UP else ""),
        "ops_per_launch": dk["ops"],
        "avg_launch_us": dk["avg_us"],
        "ops_unit": "int8 MAC x 2 per second (dense int8 MFMA)",
        "traffic_source": traffic_src,
        # E3M2: the operand bytes of the form the kernel reads (6 bits per code)
        "algorithmic_bytes_per_launch": dk.get("operand_bytes", dk["bytes"]),
        # the same kernel timed inside the eager forward (in_forward below)
        "in_forward": in_forward_roof,
    }
    out = {
        "metric": METRIC,
        "value": round(ms, 4),
        "unit": "ms",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 4),
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "i8",
        "data": "synthetic: random packed INT4 weights (codes ~ round(N(0,2)) in [-7,7], scales ~0.01), "
                "N(0,1/sqrt(2048)) fp16 prefix embeddings",
        "config": {
            "workload": f"PaliGemma-2B-shaped W4A4 prefix LM forward, {args.layers} layers, "
                        f"{args.tokens} tokens x batch {args.batch}",
            "tokens": args.tokens,
            "batch": args.batch,
            "layers": args.layers,
            "timed": "hip-graph replay" if not args.no_graph else "eager",
            "fused_gelu_up": not args.unfused_gelu,
            # idle CUs pre-read weights from HBM into the Infinity Cache inside the timed
            # forward: the attention launch each layer's o/gate/up weights, the K=16384
            # quant launch its down weights
            "weight_cache_warm": os.environ.get("PI05_W4A4_CACHE_WARM", "1") != "0",
            "attention": "prefix-attention kernels (fp16, eager-attention semantics); "
                         "forward_points has the eager-attention forward",
            "graph_replay_bit_exact_vs_eager": graph_exact,
        },
        "eager_ms_per_forward": round(eager_ms, 3),
        "w4a4_gop_per_forward": round(total_ops / 1e9, 1),
        "w4a4_kernel_ms_per_forward": round(w4a4_us_per_layer * args.layers / 1e3, 3),
        "gemms": kernels,
        "qkv_m_sweep": sweep,
        "other_kernels": others,
        "forward_points": points,
        "roofline": roofline,
        "in_forward": in_fwd,
    }
    if not args.no_cpu_baseline:
        out["cpu_baseline"] = cpu_baseline(args.tokens, args.batch, args.layers, args.cpu_seconds)
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
