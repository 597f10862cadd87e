// Prefix attention with 128 query rows per workgroup, for launches with enough rows to fill
// the chip that way (the semantics and the K / V^T fragment layout are attention.hip's).
//
// Structure.  Four waves, two workgroups per CU.  A wave owns 32 query rows for all keys:
// its queries (RoPE'd) and its O^T accumulators stay in registers.  The keys go by in steps
// of 32, 16 KB of K and 16 KB of V^T in one of two LDS stages that direct global-to-LDS
// loads fill one step ahead; one barrier per step.
//   S^T = K Q^T   The K fragments' lanes are permuted on their way into LDS so that row m of
//                 the step's 16-key block h is key 8 (m / 4) + 4 h + m % 4.  A lane's eight
//                 results for a query row are then keys 8 (L / 16) + 0..7 of the step, which is
//                 the lane's B operand of the P V product: probabilities never leave the wave.
//   softmax       e = exp(s - m) against a running reference m per row, p = fp16(e) with an
//                 fp32 row sum, O / sum at the end.  m moves (and O and the sum are rescaled)
//                 only when a score exceeds it by more than 8 in log2 units, so that p stays
//                 below 2^8 and the check needs no exchange between lanes.
// The direct loads (direct_load.h) stay in flight over the LDS reads of a step; the full wait
// and the barrier at the top of a step order them.  The mask of the next step is loaded after
// this one's was used and handed over behind that same wait.
//
// What bounds it (776 tokens x 8, 392 workgroups, one or two per CU): a step of a workgroup
// that has its CU for itself takes ~2300 cycles, 1024 of them MFMAs, ~600 the softmax's vector
// instructions, the rest the loads' issue, the barrier and the first LDS reads; with two
// workgroups the MFMAs of one and the vector instructions of the other overlap only in part
// (~4200 cycles for both).  Besides the steps ~8 us go into reading the queries (all
// workgroups start at once) and ~4 us into the output rows.  LDS reads and exp2 are hidden:
// without them the time is the same.
// Measured (with the K/V prep, masked / not): 99.9 / 97.7 us with 32-row workgroups, which
// stream K and V through every CU's vector memory path once per 32 rows, 62.2 / 59.4 now.
// Each LDS read right before its MFMAs: 70.3 / 69.3; fp32 products for the scaling and the
// compiler's max: 71.4 / 67.6 on a box where this form took 67.0 / 64.0; all loads of a step
// issued together 67.6 / 64.4; spread over both products 68.8 / 64.2; a raised wave priority
// (s_setprio) during the MFMAs 71.5 / 64.8, during the softmax 67.7 / 64.9.
#pragma once

#include "direct_load.h"
#include "quant_row.h"

namespace w4a4 {
namespace {

typedef _Float16 half2 __attribute__((ext_vector_type(2)));

constexpr int kWideWaves = 4;
constexpr int kWideThreads = 64 * kWideWaves;
constexpr int kWideRows = 32 * kWideWaves;
constexpr int kRing = 4;  // operand fragments in flight from LDS (even)
constexpr int kWideStage = 32 * 1024;  // K (16 pieces of 1 KB), then V^T (16)
constexpr size_t kWideLds = 2 * kWideStage;
constexpr size_t kWideLdsQuant = sizeof(_Float16) * (kWideRows / 8) * kOld;  // the staged output tokens
static_assert(kWideLdsQuant >= kWideLds, "the staged tokens reuse the stages");

// Packed fp16 max as one instruction (the compiler's form quiets its operands first).
__device__ __forceinline__ uint32_t pk_max(uint32_t a, uint32_t b) {
  uint32_t r;
  asm("v_pk_max_f16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// Grid: 8 * ceil(B * KVH * row_blocks / 8) workgroups of 256 threads; workgroup i runs on
// XCD i % 8, and consecutive row blocks go to one XCD, whose L2 then holds their K and V.
template <bool MASK>
__global__ __launch_bounds__(kWideThreads, 2) void prefix_attention_wide_kernel(const AttnParams p) {
  extern __shared__ __align__(16) _Float16 lds[];
  const int total = p.row_blocks * p.kvh * p.b;
  const int per = gridDim.x / 8;
  const int item = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (item >= total) return;
  const int bg = item / p.row_blocks;
  const int row0 = (item - bg * p.row_blocks) * kWideRows;
  const int g = bg % p.kvh;
  const int64_t b = bg / p.kvh;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15;
  const int lg = lane >> 4;
  const int S = p.s;
  const int n_rep = p.h / p.kvh;
  const int rows = S * n_rep;
  const int nst = p.s_pad / 32;
  const int steps = (S + 31) / 32;
  const char* kt = reinterpret_cast<const char*>(p.kv_mfma + (b * p.kvh + g) * 2 * static_cast<int64_t>(p.s_pad) * kD);
  const char* vt = kt + static_cast<int64_t>(p.s_pad) * kD * 2;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) _Float16*)lds));

  // Wave w loads K pieces 4 w .. 4 w + 3 (piece 8 h + t: block h, dimensions 32 t ..) and V^T
  // pieces 4 w .. (piece db: dimensions 16 db ..).
  const int key0 = 8 * (lr >> 2) + (lr & 3) + 4 * (w >> 1);
  const uint32_t koff = (key0 >> 4) * 8192 + ((key0 & 15) + 16 * lg) * 16;
  const uint32_t voff = lane * 16;
  auto load_piece = [&](int u, int u1, int j) {  // j = 0..3: K, 4..7: V^T
    const uint32_t st = lds0 + (u & 1) * kWideStage + 4 * w * 1024;
    if (j < 4)
      load_lds_1k(kt + static_cast<int64_t>(u1) * 16384 + (4 * (w & 1) + j) * 1024, koff, st + j * 1024);
    else
      load_lds_1k(vt + (static_cast<int64_t>(4 * w + j - 4) * nst + u1) * 1024, voff, st + 16384 + (j - 4) * 1024);
  };

  // Mask chunks of a step: row 16 qb + L % 16, keys 8 (L / 16) + 0..7, in 8-byte halves
  // clamped into the row (keys past it are masked below).
  typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
  typedef const __attribute__((address_space(1))) u32x2* gptr2;
  const _Float16* mrow = MASK ? p.mask + b * p.mask_bs : nullptr;
  u32x2 mv[2][2];
  int32_t moff[2];  // the launcher checks that a sequence's mask fits
  half8 qop[2][8];
  auto load_mask = [&](int u) {
    if constexpr (MASK) {
      const int kc = 32 * u + 8 * lg;
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int i = 0; i < 2; ++i) mv[qb][i] = *(gptr2)(mrow + (moff[qb] + min(kc + 4 * i, p.mask_len - 4)));
    }
  };

  // The queries as MFMA operand B: lane L holds row 16 qb + L % 16, dimensions
  // 32 t + 8 (L / 16) + 0..7; the RoPE pairs (d, d + 128) are t and t + 4 of one lane.  Rows
  // past the group are clamped (computed, never stored).
#pragma unroll
  for (int j = 0; j < 8; ++j) load_piece(0, 0, j);
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const int rr = min(row0 + 32 * w + 16 * qb + lr, rows - 1);
    const int64_t tk = b * S + rr / n_rep;
    moff[qb] = MASK ? rr / n_rep * static_cast<int32_t>(p.mask_rs) : 0;
    const _Float16* qr = p.q + tk * p.ld_q + (g * n_rep + rr % n_rep) * kD + 8 * lg;
    const _Float16* cr = p.cosb + tk * kD + 8 * lg;
    const _Float16* sr = p.sinb + tk * kD + 8 * lg;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      qop[qb][t] = ld8(qr + 32 * t);
      qop[qb][t + 4] = ld8(qr + 128 + 32 * t);
      rope_pair(qop[qb][t], qop[qb][t + 4], ld8(cr + 32 * t), ld8(cr + 128 + 32 * t), ld8(sr + 32 * t), ld8(sr + 128 + 32 * t));
    }
  }
  load_mask(0);

  f4 o[16][2];
#pragma unroll
  for (int db = 0; db < 16; ++db) o[db][0] = o[db][1] = f4{0, 0, 0, 0};
  constexpr float kLog2e = 1.4426950408889634f;
  // The reference of a row, times log2 e.  It starts finite, so that -inf scores give e = 0
  // before any other score was seen; a row of -inf alone ends as 0 / 0.
  const _Float16 scale16 = static_cast<_Float16>(p.scaling);  // exact (the launcher checks it)
  float ml[2] = {-3.0e38f, -3.0e38f};
  float l[2] = {0.0f, 0.0f};

  for (int u = 0; u < steps; ++u) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if constexpr (MASK) asm volatile("" : "+v"(mv[0][0]), "+v"(mv[0][1]), "+v"(mv[1][0]), "+v"(mv[1][1]));
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int u1 = min(u + 1, steps - 1);  // the last step loads once more, unread
    const _Float16* st = lds + (u & 1) * (kWideStage / 2) + 8 * lane;

    f4 acc[2][2];  // [block h][qb]
#pragma unroll
    for (int h = 0; h < 2; ++h) acc[h][0] = acc[h][1] = f4{0, 0, 0, 0};
    // The fragments go through a ring of kRing registers; the barriers keep the scheduler
    // from moving the reads next to their use.
    half8 ring[kRing];
#pragma unroll
    for (int n = 0; n < kRing; ++n) ring[n] = ld8(st + (8 * (n & 1) + (n >> 1)) * 512);
#pragma unroll
    for (int n = 0; n < 16; ++n) {  // block n % 2, dimensions 32 (n / 2) ..
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
        acc[n & 1][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ring[n % kRing], qop[qb][n >> 1], acc[n & 1][qb], 0, 0, 0);
      if (n + kRing < 16) ring[n % kRing] = ld8(st + (8 * (n & 1) + ((n + kRing) >> 1)) * 512);
      if (n & 1) load_piece(u + 1, u1, n >> 1);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < kRing; ++n) ring[n] = ld8(st + 8192 + n * 512);

    half8 sv[2];
    float mt[2];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
#pragma clang fp contract(off)
      const half4 lo = __builtin_convertvector(acc[0][qb], half4), hi = __builtin_convertvector(acc[1][qb], half4);
      sv[qb] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7) * scale16;
      if constexpr (MASK) {
        // fp16 additions round exactly like torch's fp32-opmath fp16 add.
        const uint4 m4 = {mv[qb][0].x, mv[qb][0].y, mv[qb][1].x, mv[qb][1].y};
        sv[qb] = sv[qb] + __builtin_bit_cast(half8, m4);
      }
    }
    if (32 * u + 32 > S) {  // the last step: padding keys
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (32 * u + 8 * lg + e >= S) sv[qb][e] = static_cast<_Float16>(-__builtin_inff());
    }
    if (u + 1 < steps) load_mask(u + 1);
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      const uint4 x = __builtin_bit_cast(uint4, sv[qb]);
      const half2 m2 = __builtin_bit_cast(half2, pk_max(pk_max(x.x, x.y), pk_max(x.z, x.w)));
      mt[qb] = fmaxf(static_cast<float>(m2[0]), static_cast<float>(m2[1])) * kLog2e;
    }
    if (__builtin_amdgcn_ballot_w64(mt[0] > ml[0] + 8.0f || mt[1] > ml[1] + 8.0f) != 0) {
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        float m = fmaxf(mt[qb], __shfl_xor(mt[qb], 16));
        m = fmaxf(fmaxf(m, __shfl_xor(m, 32)), ml[qb]);
        const float alpha = __builtin_amdgcn_exp2f(ml[qb] - m);
        ml[qb] = m;
        l[qb] *= alpha;
#pragma unroll
        for (int db = 0; db < 16; ++db)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[db][qb][i] *= alpha;
      }
    }
    half8 pv[2];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = __builtin_amdgcn_exp2f(__builtin_fmaf(static_cast<float>(sv[qb][e]), kLog2e, -ml[qb]));
        l[qb] += x;
        pv[qb][e] = static_cast<_Float16>(x);
      }

#pragma unroll
    for (int db = 0; db < 16; ++db) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
        o[db][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ring[db % kRing], pv[qb], o[db][qb], 0, 0, 0);
      if (db + kRing < 16) ring[db % kRing] = ld8(st + 8192 + (db + kRing) * 512);
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  float rl[2];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    float s = l[qb] + __shfl_xor(l[qb], 16);
    s += __shfl_xor(s, 32);
    rl[qb] = 1.0f / s;
  }
  // Result lane L: O[row 16 qb + L % 16][16 db + 4 (L / 16) + i].
  auto out4 = [&](int db, int qb) {
    half4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = static_cast<_Float16>(o[db][qb][i] * rl[qb]);
    return v;
  };
  if (p.out != nullptr) {
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      const int rr = row0 + 32 * w + 16 * qb + lr;
      if (rr >= rows) continue;
      _Float16* orow = p.out + (b * S + rr / n_rep) * p.ld_out + (g * n_rep + rr % n_rep) * kD + 4 * lg;
#pragma unroll
      for (int db = 0; db < 16; ++db) *reinterpret_cast<half4*>(orow + 16 * db) = out4(db, qb);
    }
  }

  // One KV head of 8 query heads: the wave's 32 rows are 4 whole tokens of the o-proj input,
  // staged in LDS and quantized by the same wave (the K = 2048 activation quant).
  if (p.qcodes != nullptr) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave is done with the stages
    _Float16* otile = lds + 4 * w * kOld;
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int db = 0; db < 16; ++db)
        *reinterpret_cast<half4*>(otile + (2 * qb + (lr >> 3)) * kOld + (lr & 7) * kD + 16 * db + 4 * lg) = out4(db, qb);
    for (int i = 0; i < 4; ++i) {
      const int tok = (row0 >> 3) + 4 * w + i;
      if (tok >= S) break;
      float v[32];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const half8 x = ld8(otile + i * kOld + 32 * lane + 8 * c);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[8 * c + e] = static_cast<float>(x[e]);
      }
      fwht_quant_row_wave<11>(v, lane, b * S + tok, p.qcodes, p.qscales, p.qcorr, p.inv_sqrt_k);
    }
  }
}

}  // namespace
}  // namespace w4a4
