// Shared device code of the activation quantizers: the Sylvester FWHT of one row held in
// registers (passes of register butterflies with LDS transposes between them), the
// per-token INT4 quantization and the stores of the codes, the scale and the row
// correction.  Used by quant_rot.hip (one row per workgroup or per wave) and by the
// prefix attention kernel, whose workgroup quantizes the o-proj input rows it produced.
#pragma once

#include "w4a4_internal.h"

namespace w4a4 {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));

constexpr int kDppXor1 = 0xB1;       // quad_perm [1,0,3,2]
constexpr int kDppXor2 = 0x4E;       // quad_perm [2,3,0,1]
constexpr int kDppRev4 = 0x1B;       // quad_perm [3,2,1,0]: lane i^3 within the quad
constexpr int kDppHalfMirror = 0x141;  // row_half_mirror: lane i^7 within 8
constexpr int kDppRor8 = 0x128;      // row_ror:8: lane i^8 within the 16-lane row

template <int CTRL>
__device__ __forceinline__ float dpp_f(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}
template <int CTRL>
__device__ __forceinline__ int dpp_i(int x) {
  return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xF, 0xF, false);
}
// x of lane (this lane ^ (1 << K)), K = 0..3.
template <int K>
__device__ __forceinline__ float lane_xor_f(float x) {
  if constexpr (K == 0) return dpp_f<kDppXor1>(x);
  else if constexpr (K == 1) return dpp_f<kDppXor2>(x);
  else if constexpr (K == 2) return dpp_f<kDppHalfMirror>(dpp_f<kDppRev4>(x));
  else return dpp_f<kDppRor8>(x);
}
template <int K>
__device__ __forceinline__ int lane_xor_i(int x) {
  if constexpr (K == 0) return dpp_i<kDppXor1>(x);
  else if constexpr (K == 1) return dpp_i<kDppXor2>(x);
  else if constexpr (K == 2) return dpp_i<kDppHalfMirror>(dpp_i<kDppRev4>(x));
  else return dpp_i<kDppRor8>(x);
}
// Max / sum over the 64 lanes, the result in every lane.
__device__ __forceinline__ float wave_max_dpp(float v) {
  v = fmaxf(v, lane_xor_f<0>(v));
  v = fmaxf(v, lane_xor_f<1>(v));
  v = fmaxf(v, lane_xor_f<2>(v));
  v = fmaxf(v, lane_xor_f<3>(v));
  auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(r16[0]), __uint_as_float(r16[1]));
  auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r32[0]), __uint_as_float(r32[1]));
}
__device__ __forceinline__ int wave_sum_dpp(int v) {
  v += lane_xor_i<0>(v);
  v += lane_xor_i<1>(v);
  v += lane_xor_i<2>(v);
  v += lane_xor_i<3>(v);
  auto r16 = __builtin_amdgcn_permlane16_swap(static_cast<unsigned>(v), static_cast<unsigned>(v), false, false);
  v = static_cast<int>(r16[0]) + static_cast<int>(r16[1]);
  auto r32 = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(v), static_cast<unsigned>(v), false, false);
  return static_cast<int>(r32[0]) + static_cast<int>(r32[1]);
}
// The same reductions under the names the quantizers use.  Max and integer sums do not
// depend on the order.  The fp32 sum keeps the xor butterfly 32, 16, 8, 4, 2, 1 (each
// step v + partner, and fp32 addition is commutative), so it equals the LDS-permute
// loop v += shfl_xor(v, o) for o = 32 .. 1 bit for bit, without its six LDS round trips.
__device__ __forceinline__ float wave_max(float v) { return wave_max_dpp(v); }
__device__ __forceinline__ int wave_sum(int v) { return wave_sum_dpp(v); }
__device__ __forceinline__ float wave_sum_f(float v) {
  auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __fadd_rn(__uint_as_float(r32[0]), __uint_as_float(r32[1]));
  auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __fadd_rn(__uint_as_float(r16[0]), __uint_as_float(r16[1]));
  v = __fadd_rn(v, lane_xor_f<3>(v));
  v = __fadd_rn(v, lane_xor_f<2>(v));
  v = __fadd_rn(v, lane_xor_f<1>(v));
  return __fadd_rn(v, lane_xor_f<0>(v));
}

// 16 * (sum of the four codes in the high nibbles of w, the odd-k codes): a signed dot
// product of the bytes 16c with ones.
__device__ __forceinline__ int odd_code_sum16(uint32_t w) {
  return __builtin_amdgcn_sdot4(static_cast<int>(w & kHiNib), 0x01010101, 0, false);
}

// Sum over the T threads of a row (T / 64 waves); the result is valid in thread 0.
template <int T>
__device__ __forceinline__ int row_sum(int v, int* red) {
  v = wave_sum(v);
  if constexpr (T > 64) {
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
#pragma unroll
    for (int i = 1; i < T / 64; ++i) v += red[i];
  }
  return v;
}

// Eight codes c = clamp(rint(v / sdiv), -7, 7) packed as nibbles 0..7 of one word in the
// stored form: low nibble of each byte c + 8 (offset binary), high nibble c & 0xF (two's
// complement).  Each code is computed as c + 8, in [1, 15], and placed with one
// shift-or; the final xor turns the high nibbles from offset binary to two's complement
// ((c + 8) ^ 8 == c & 0xF).  A NaN quotient gives -7 (the clamp keeps the non-NaN bound).
__device__ __forceinline__ uint32_t quant_pack8(const float (&v)[8], float sdiv) {
  uint32_t word = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float r = __builtin_rintf(__fdiv_rn(v[e], sdiv));
    r = fminf(fmaxf(r, -7.0f), 7.0f) + 8.0f;
    word |= static_cast<uint32_t>(r) << (4 * e);
  }
  return word ^ kObFlipHi;
}

// Same eight codes without a division per element.  qa = fl(v * rcp(sdiv) + 8) (one
// fused rounding) differs from the exact q + 8, q = v / sdiv, by less than 1.31e-6:
// |q| <= 7 and v_rcp_f32 is documented to 1 ulp, a relative error of at most 2^-23, so
// v * rcp is within 7 * 2^-23 (8.3e-7) of q; the fma adds 8 exactly and rounds once, at an
// ulp of at most 2^-20 for results below 16 (error <= 2^-21, 4.8e-7).
// rint(q + 8) == rint(q) + 8 (8 is even, so ties still go to even), so rint(qa) - 8 ==
// rint(q) unless q lies within 1.31e-6 of a half-integer.  Any lane that sees qa within
// 3e-6 of one (more than twice that bound) raises `near_tie` for this word; the caller then
// redoes that word's codes with quant_pack8 (exact division).  Both paths therefore
// produce the reference's round-half-even codes bit for bit.  One slow row sets a
// launch's end, so the redo is kept small: a 3e-6 window (1e-5 before) and only the
// flagged words redone (before: every word of the wave), which took the K=16384 quant at
// 776 rows from 18.4 to 16.9 us.
__device__ __forceinline__ uint32_t quant_pack8_rcp(const float (&v)[8], float rcp, bool& near_tie) {
  uint32_t word = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float qa = __builtin_fmaf(v[e], rcp, 8.0f);
    float r = __builtin_rintf(qa);
    near_tie |= fabsf(qa - r) > 0.499997f;
    r = fminf(fmaxf(r, 1.0f), 15.0f);
    word |= static_cast<uint32_t>(r) << (4 * e);
  }
  return word ^ kObFlipHi;
}

// The codes of quant_pack8 / quant_pack8_rcp as floats c + 8 in [1, 15] (same arithmetic,
// so the same codes), for the E3M2 operand form.
__device__ __forceinline__ void quant_codes8(const float (&v)[8], float sdiv, float* c) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float r = __builtin_rintf(__fdiv_rn(v[e], sdiv));
    c[e] = fminf(fmaxf(r, -7.0f), 7.0f) + 8.0f;
  }
}
__device__ __forceinline__ void quant_codes8_rcp(const float (&v)[8], float rcp, bool& near_tie, float* c) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float qa = __builtin_fmaf(v[e], rcp, 8.0f);
    const float r = __builtin_rintf(qa);
    near_tie |= fabsf(qa - r) > 0.499997f;
    c[e] = fminf(fmaxf(r, 1.0f), 15.0f);
  }
}

// One lane's 32 consecutive codes of row `row` (elements 32 t .. 32 t + 31, t the lane) as
// an E3M2 fragment slot (the q6 layout of w4a4_internal.h): c holds code + 8.
// v_cvt_scalef32_2xpk16_bf6_f32 converts two 16-value vectors, interleaving them (output
// value 2i from the first, 2i + 1 from the second), so the even and the odd codes go in
// separately; integers in [-7, 7] convert exactly.
__device__ __forceinline__ void store_e3m2_slot(const float (&c)[32], int t, int64_t row, int32_t kb128,
                                                uint8_t* __restrict__ q6) {
  typedef float v16f __attribute__((ext_vector_type(16)));
  v16f ev, od;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    ev[i] = c[2 * i] - 8.0f;
    od[i] = c[2 * i + 1] - 8.0f;
  }
  const auto d = __builtin_amdgcn_cvt_scalef32_2xpk16_bf6_f32(ev, od, 1.0f);
  uint8_t* const frag = q6 + ((row >> 4) * kb128 + (t >> 2)) * static_cast<int64_t>(kE3m2FragBytes);
  const int slot = static_cast<int>(row & 15) + 16 * (t & 3);
  *reinterpret_cast<uint4*>(frag + 16 * slot) = make_uint4(d[0], d[1], d[2], d[3]);
  *reinterpret_cast<uint2*>(frag + 1024 + 8 * slot) = make_uint2(d[4], d[5]);
}

// ---- One wave per row, registers only (T = 64).  Lane t holds R = K / 64 consecutive
// elements t*R .. t*R + R - 1 in v[0..R-1] (r = log2 R register bits, then 6 lane bits).
// The butterfly stages still run in increasing order of the stride, each writing
// (a + b, a - b) exactly, so the result is bit-identical to the CPU transform:
//   element bits 0 .. r-1     registers (pairs v[j], v[j ^ 2^b]);
//   element bits r .. r+3     lane bits 0-3: the partner's value comes through DPP
//                             (xor 1, 2: quad_perm; xor 4: quad_perm + row_half_mirror;
//                             xor 8: row_ror:8) straight into the add, and the upper lane
//                             adds its own value negated: partner + (-own) = a - b;
//   element bits r+4, r+5     lane bits 4 and 5: v_permlane16_swap / v_permlane32_swap on
//                             the register pairs of bit 0 / bit 1 (already transformed)
//                             exchange that register bit with the lane bit, the stage runs
//                             in registers, and the swaps are undone afterwards.
// No LDS and no barrier; the wave max and sum use the same DPP / swap exchanges.
// Register pairs (v[j], v[j | 2^B]) exchange register bit B with lane bit 4 (SW = 16) or
// lane bit 5 (SW = 32); applying it twice restores the layout.
template <int SW, int B, int R>
__device__ __forceinline__ void swap_lane_bit(float (&v)[R]) {
#pragma unroll
  for (int j = 0; j < R; ++j) {
    if (j & (1 << B)) continue;
    auto r = (SW == 16) ? __builtin_amdgcn_permlane16_swap(__float_as_uint(v[j]), __float_as_uint(v[j | (1 << B)]), false, false)
                        : __builtin_amdgcn_permlane32_swap(__float_as_uint(v[j]), __float_as_uint(v[j | (1 << B)]), false, false);
    v[j] = __uint_as_float(r[0]);
    v[j | (1 << B)] = __uint_as_float(r[1]);
  }
}
template <int B, int R>
__device__ __forceinline__ void reg_stage(float (&v)[R]) {
#pragma unroll
  for (int j = 0; j < R; ++j) {
    if (j & (1 << B)) continue;
    const float a = v[j], c = v[j + (1 << B)];
    v[j] = __fadd_rn(a, c);
    v[j + (1 << B)] = __fsub_rn(a, c);
  }
}
template <int K, int R>
__device__ __forceinline__ void lane_stage(float (&v)[R], int lane) {
  const uint32_t neg = static_cast<uint32_t>((lane >> K) & 1) << 31;  // upper lane: a - b
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const float partner = lane_xor_f<K>(v[j]);
    v[j] = __fadd_rn(partner, __uint_as_float(__float_as_uint(v[j]) ^ neg));
  }
}

// Rotation, quantization and stores of one row of K = 16384 values held by 256 threads,
// thread t (lane l = t % 64, wave w = t / 64) with the 64 consecutive fp16 values 64 t .. of
// xv on entry.  The 14 butterfly stages run in increasing order of the stride, each writing
// (a + b, a - b), in three register passes over element bits 0-5, 6-11 and 12-13, so the
// rotated values are bit-identical to the CPU transform:
//   pass 0   registers = bits 0-5, lanes = bits 6-11, waves = bits 12-13.  Its first stage
//            reads the fp16 pairs directly (v_fma_mix: a * 1 + b, one rounding);
//   T1       inside a wave, through its own quarter of the LDS: no workgroup barrier;
//   pass 1   registers = bits 6-11, lanes = bits 0-5;
//   T2       across the waves;
//   pass 2   registers = bits 12-13 (2) and 0-3, thread = bits 4-11.
// Two forms of the transposes:
//   HALF = false  the whole row at a time (68 KB, two rows per CU): T1 writes and reads a
//                 wave's 4096 values, T2 writes them back in place, one barrier, and reads.
//   HALF = true   half a row at a time (36 KB, three rows per CU): v_permlane32_swap exchanges
//                 bits 5 and 11, then T1 is two 32 x 32 transposes per half wave; T2 takes two
//                 rounds (bit 11): every wave writes its 32 registers of the round, then the
//                 two waves that own those elements read them.  Three rows overlap their loads,
//                 vector work and LDS phases better, but one row takes longer.
// What bounds it is the chain of one row's phases (load, three register passes of 2 x 64
// vector instructions per thread and stage pair, two transposes, one wide reduction) and how
// many rows per CU hide each other's: at 6208 rows 305 MB move in 70 us (4.4 TB/s of the 4.9 a
// copy reaches; 83 us before with three workgroup-wide transposes and rows written in
// order); at 776 rows, three rows per CU, 14.8 us (17.0).  With four half rows per CU the
// compiler has 128 registers and spills: 75.7 us at 6208 rows.
// L: kRow16kLds<HALF> floats of LDS, padded by 4 floats per 64 (per 32 in T1's half form)
// against bank conflicts; red / ired: 4 floats / ints.  E3M2: the codes go out as E3M2
// fragment slots (q points at the q6 buffer; no row corrections).
template <bool HALF>
constexpr int kRow16kLds = HALF ? 4 * 2 * 32 * 36 : 256 * 68;
typedef uint32_t row16k_in __attribute__((ext_vector_type(4)));

template <bool HALF, bool E3M2 = false>
__device__ __forceinline__ void fwht_quant_row16k(const row16k_in (&xv)[8], float* L, float* red, int* ired, int t,
                                                  int64_t row, int32_t* __restrict__ q, float* __restrict__ sa,
                                                  int32_t* __restrict__ qcorr, float inv_sqrt_k) {
  const int lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  float v[64];
#pragma unroll
  for (int i = 0; i < 32; ++i) {  // stage 0: the halves of a dword
    const uint32_t x = xv[i / 4][i % 4];
    asm("v_fma_mix_f32 %0, %1, 1.0, %1 op_sel:[0,0,1] op_sel_hi:[1,0,1]" : "=v"(v[2 * i]) : "v"(x));
    asm("v_fma_mix_f32 %0, %1, 1.0, -%1 op_sel:[0,0,1] op_sel_hi:[1,0,1]" : "=v"(v[2 * i + 1]) : "v"(x));
  }
  reg_stage<1>(v);
  reg_stage<2>(v);
  reg_stage<3>(v);
  reg_stage<4>(v);
  reg_stage<5>(v);
  if constexpr (HALF) {
    // After the swap register bit 5 holds element bit 11 and lane bit 5 element bit 5.
    swap_lane_bit<32, 5>(v);
    float* const Lw = L + w * (2 * 32 * 36) + (lane >> 5) * (32 * 36);
    const int l = lane & 31;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int j = 0; j < 32; j += 4)
        *reinterpret_cast<float4*>(Lw + l * 36 + j) =
            make_float4(v[32 * c + j], v[32 * c + j + 1], v[32 * c + j + 2], v[32 * c + j + 3]);
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < 32; ++j) v[32 * c + j] = Lw[j * 36 + l];
      __builtin_amdgcn_wave_barrier();
    }
  } else {
#pragma unroll
    for (int j = 0; j < 64; j += 4)
      *reinterpret_cast<float4*>(L + t * 68 + j) = make_float4(v[j], v[j + 1], v[j + 2], v[j + 3]);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < 64; ++j) v[j] = L[w * 4352 + lane + 68 * j];
    __builtin_amdgcn_wave_barrier();
  }
  reg_stage<0>(v);
  reg_stage<1>(v);
  reg_stage<2>(v);
  reg_stage<3>(v);
  reg_stage<4>(v);
  reg_stage<5>(v);
  if constexpr (HALF) {
    // Element e without bit 11 (bits 0-10, then 12-13) of a round at e' + 4 (e' / 64).
    float u[64];
    float* const wb = L + w * (2048 + 128) + lane;
    const float* const rb = L + (t & 127) * 16 + 4 * ((t & 127) >> 2);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int j = 0; j < 32; ++j) wb[j * 68] = v[32 * c + j];
      __syncthreads();
      if ((w >> 1) == c) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g) u[g + 4 * i] = rb[g * (2048 + 128) + i];
      }
      if (c == 0) __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < 64; ++j) v[j] = u[j];
  } else {
    // Element e at e + 4 (e / 64).
#pragma unroll
    for (int j = 0; j < 64; ++j) L[w * 4352 + lane + 68 * j] = v[j];
    __syncthreads();
    const float* const rb = L + t * 16 + 4 * (t >> 2);
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) v[g + 4 * i] = rb[g * 4352 + i];
  }
  reg_stage<0>(v);
  reg_stage<1>(v);

  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < 64; ++j) amax = fmaxf(amax, fabsf(v[j]));
  amax = wave_max(amax);
  if ((t & 63) == 0) red[t >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float sdiv = __fadd_rn(__fdiv_rn(amax, 7.0f), 1e-12f);
  if (t == 0) sa[row] = __fmul_rn(sdiv, inv_sqrt_k);

  // For each g the registers g + 4 i, i = 0 .. 15, hold the run of 16 consecutive elements from
  // 16 t + 4096 g on: packed 8 at a time, two words (16 codes, 8 bytes: consecutive words of
  // the row's slot in its fragment) to a store.
  constexpr int NW = 8;  // code words per thread
  auto gather8 = [&](int g, int u, float (&c8)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) c8[e] = v[g + 4 * (8 * u + e)];
  };
  bool tie[NW];
  bool near_tie = false;
  const float rcp = __builtin_amdgcn_rcpf(sdiv);
  if constexpr (E3M2) {
    typedef float v16f __attribute__((ext_vector_type(16)));
    uint32_t d[2][6];  // runs 2 h and 2 h + 1, three dwords each
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float c[4][8];  // codes + 8
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float c8[8];
        gather8(2 * h + i / 2, i % 2, c8);
        tie[i] = false;
        quant_codes8_rcp(c8, rcp, tie[i], c[i]);
      }
      near_tie = tie[0] | tie[1] | tie[2] | tie[3];
      if (__builtin_amdgcn_ballot_w64(near_tie) != 0) {  // rare: redo the flagged groups exactly
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (__builtin_amdgcn_ballot_w64(tie[i]) != 0) {
            float c8[8], x8[8];
            gather8(2 * h + i / 2, i % 2, c8);
            quant_codes8(c8, sdiv, x8);
#pragma unroll
            for (int e = 0; e < 8; ++e) c[i][e] = tie[i] ? x8[e] : c[i][e];
          }
        }
      }
      v16f ev, od;  // even and odd codes of run 2 h, then of run 2 h + 1
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        ev[i] = c[i / 4][2 * (i & 3)] - 8.0f;
        od[i] = c[i / 4][2 * (i & 3) + 1] - 8.0f;
      }
      const auto x = __builtin_amdgcn_cvt_scalef32_2xpk16_bf6_f32(ev, od, 1.0f);
#pragma unroll
      for (int i = 0; i < 6; ++i) d[h][i] = x[i];
    }
    // Threads 2u and 2u + 1 hold the two halves of four slots: the even one takes the other's
    // halves of slots 0 and 1, the odd one of slots 2 and 3, so that a slot is stored whole.
    const bool odd = (t & 1) != 0;
    uint32_t mine[6], got[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      got[i] = static_cast<uint32_t>(dpp_i<kDppXor1>(static_cast<int>(odd ? d[0][i] : d[1][i])));
      mine[i] = odd ? d[1][i] : d[0][i];
    }
    uint8_t* const q6 = reinterpret_cast<uint8_t*>(q);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint32_t w[6];  // the slot's six dwords, the even thread's half first
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        w[i] = odd ? got[3 * h + i] : mine[3 * h + i];
        w[3 + i] = odd ? mine[3 * h + i] : got[3 * h + i];
      }
      const int e0 = 16 * (t & ~1) + 4096 * ((odd ? 2 : 0) + h);  // the slot's first element
      uint8_t* const frag = q6 + ((row >> 4) * kblocks128(16384) + (e0 >> 7)) * static_cast<int64_t>(kE3m2FragBytes);
      const int slot = static_cast<int>(row & 15) + 16 * ((e0 >> 5) & 3);
      *reinterpret_cast<uint4*>(frag + 16 * slot) = make_uint4(w[0], w[1], w[2], w[3]);
      *reinterpret_cast<uint2*>(frag + 1024 + 8 * slot) = make_uint2(w[4], w[5]);
    }
    return;
  }
  uint32_t words[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    float c8[8];
    gather8(i / 2, i % 2, c8);
    tie[i] = false;
    words[i] = quant_pack8_rcp(c8, rcp, tie[i]);
    near_tie |= tie[i];
  }
  if (__builtin_amdgcn_ballot_w64(near_tie) != 0) {  // rare: redo the flagged words exactly
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      if (__builtin_amdgcn_ballot_w64(tie[i]) != 0) {
        float c8[8];
        gather8(i / 2, i % 2, c8);
        const uint32_t exact = quant_pack8(c8, sdiv);
        words[i] = tie[i] ? exact : words[i];
      }
    }
  }
  int s16 = 0;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const uint2 wd = make_uint2(words[2 * g], words[2 * g + 1]);
    *reinterpret_cast<uint2*>(&q[frag_word_index(row, 2 * t + 512 * g, kblocks128(16384))]) = wd;
    s16 += odd_code_sum16(wd.x) + odd_code_sum16(wd.y);
  }
  s16 = row_sum<256>(s16, ired);
  if (t == 0) qcorr[row] = -8 * s16;
}


// RMSNorm of one row held by one wave (transformers' GemmaRMSNorm, modeling_gemma.py:64-78,
// weight wv with the (1 + w) offset when unit_offset), in place:
//   h = fp16((x * r) * g),  r = 1 / sqrt(ss / K + eps) (correctly rounded sqrt and
//   division),  g = unit_offset + w,
// with ss summed per lane over its R consecutive elements in order, then over the 64 lanes
// by the xor butterfly 32, 16, .., 1; v then holds the fp16 h as fp32 values.
// r of the row (the sum of squares in the order above).
template <int K, int R>
__device__ __forceinline__ float rms_norm_rr_wave(const float (&v)[R], float eps) {
#pragma clang fp contract(off)
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < R; ++j) ss = ss + v[j] * v[j];
  ss = wave_sum_f(ss);
  return 1.0f / __builtin_sqrtf(ss * (1.0f / K) + eps);
}
// h = fp16((x * r) * g) of the N values in v, elementwise (any layout of the row).
template <int N>
__device__ __forceinline__ void rms_norm_apply(float (&v)[N], const half8 (&wv)[N / 8], float rr, int unit_offset) {
#pragma clang fp contract(off)
#pragma unroll
  for (int c = 0; c < N / 8; ++c) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float g = unit_offset ? 1.0f + static_cast<float>(wv[c][e]) : static_cast<float>(wv[c][e]);
      float y = (v[8 * c + e] * rr) * g;
      asm volatile("" : "+v"(y));  // keep the fp32 product (no v_fma_mix into fp16)
      v[8 * c + e] = static_cast<float>(static_cast<_Float16>(y));
    }
  }
}
template <int K, int R>
__device__ __forceinline__ void rms_norm_row_wave(float (&v)[R], const half8 (&wv)[R / 8], float eps,
                                                  int unit_offset) {
  rms_norm_apply<R>(v, wv, rms_norm_rr_wave<K>(v, eps), unit_offset);
}

// E3M2: the codes go out as E3M2 fragment slots (q then points at the q6 buffer; no row
// corrections), else as INT4 words and qcorr.
template <int LOGK, bool E3M2 = false>
__device__ __forceinline__ void fwht_quant_row_wave(float (&v)[1 << (LOGK - 6)], int t, int64_t row,
                                                    int32_t* __restrict__ q, float* __restrict__ sa,
                                                    int32_t* __restrict__ qcorr, float inv_sqrt_k) {
  constexpr int K = 1 << LOGK;
  constexpr int r = LOGK - 6;
  constexpr int R = 1 << r;
  static_assert(r >= 4, "runs of >= 16 consecutive elements per lane");
#pragma unroll
  for (int b = 0; b < r; ++b) {
    if (b == 0) reg_stage<0>(v);
    else if (b == 1) reg_stage<1>(v);
    else if (b == 2) reg_stage<2>(v);
    else if (b == 3) reg_stage<3>(v);
    else if (b == 4) reg_stage<4>(v);
    else if (b == 5) reg_stage<5>(v);
    else if (b == 6) reg_stage<6>(v);
    else if (b == 7) reg_stage<7>(v);
  }
  lane_stage<0>(v, t);
  lane_stage<1>(v, t);
  lane_stage<2>(v, t);
  lane_stage<3>(v, t);
  swap_lane_bit<16, 0>(v);
  reg_stage<0>(v);  // element bit r + 4
  swap_lane_bit<32, 1>(v);
  reg_stage<1>(v);  // element bit r + 5
  swap_lane_bit<32, 1>(v);
  swap_lane_bit<16, 0>(v);

  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < R; ++j) amax = fmaxf(amax, fabsf(v[j]));
  amax = wave_max_dpp(amax);
  const float sdiv = __fadd_rn(__fdiv_rn(amax, 7.0f), 1e-12f);
  if (t == 0) sa[row] = __fmul_rn(sdiv, inv_sqrt_k);
  if constexpr (E3M2) {
    static_assert(R == 32, "one E3M2 fragment slot (32 codes) per lane");
    float c[R];
    bool tie[R / 8];
    bool near_tie = false;
    const float rcp = __builtin_amdgcn_rcpf(sdiv);
#pragma unroll
    for (int u = 0; u < R / 8; ++u) {
      float c8[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) c8[e] = v[8 * u + e];
      tie[u] = false;
      quant_codes8_rcp(c8, rcp, tie[u], c + 8 * u);
      near_tie |= tie[u];
    }
    if (__builtin_amdgcn_ballot_w64(near_tie) != 0) {  // rare: redo the flagged groups exactly
#pragma unroll
      for (int u = 0; u < R / 8; ++u) {
        if (__builtin_amdgcn_ballot_w64(tie[u]) != 0) {
          float c8[8], x8[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) c8[e] = v[8 * u + e];
          quant_codes8(c8, sdiv, x8);
#pragma unroll
          for (int e = 0; e < 8; ++e) c[8 * u + e] = tie[u] ? x8[e] : c[8 * u + e];
        }
      }
    }
    store_e3m2_slot(c, t, row, kblocks128(K), reinterpret_cast<uint8_t*>(q));
    return;
  }
  // Codes of the lane's R consecutive elements: R / 8 words, word u = codes 8u .. 8u + 7.
  uint32_t words[R / 8];
  bool tie[R / 8];
  bool near_tie = false;
  const float rcp = __builtin_amdgcn_rcpf(sdiv);
#pragma unroll
  for (int u = 0; u < R / 8; ++u) {
    float c8[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) c8[e] = v[8 * u + e];
    tie[u] = false;
    words[u] = quant_pack8_rcp(c8, rcp, tie[u]);
    near_tie |= tie[u];
  }
  if (__builtin_amdgcn_ballot_w64(near_tie) != 0) {  // rare: redo the flagged words exactly
#pragma unroll
    for (int u = 0; u < R / 8; ++u) {
      if (__builtin_amdgcn_ballot_w64(tie[u]) != 0) {
        float c8[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) c8[e] = v[8 * u + e];
        const uint32_t exact = quant_pack8(c8, sdiv);
        words[u] = tie[u] ? exact : words[u];
      }
    }
  }
#pragma unroll
  for (int u = 0; u < R / 8; u += 2) {
    const uint2 wd = make_uint2(words[u], words[u + 1]);
    *reinterpret_cast<uint2*>(&q[frag_word_index(row, (t * R) / 8 + u, kblocks128(K))]) = wd;
  }
  int s16 = 0;
#pragma unroll
  for (int u = 0; u < R / 8; ++u) s16 += odd_code_sum16(words[u]);
  s16 = wave_sum_dpp(s16);
  if (t == 0) qcorr[row] = -8 * s16;
}

// ---- Two waves per row (T = 128): thread t = 64 h + lane (h = the wave of the pair) holds
// R = K / 128 consecutive elements t*R .. t*R + R - 1.  Element bits 0 .. r+5 are the
// one-wave form's (registers, then lane bits 0-5); the last stage, over the wave bit h,
// exchanges the halves through LDS: lane L of the lower wave keeps a + b, of the upper
// wave a - b, with a the lower wave's value.  The row max and the odd-code sum combine the
// two waves' through LDS too.  xch: 2 * 64 * R floats of LDS for this row; redf / redi: 2
// words each.  Every wave of the workgroup calls it together (three workgroup barriers);
// with `store` false the pair computes but writes nothing (a row past the matrix).
template <int LOGK>
__device__ __forceinline__ void fwht_quant_row_2wave(float (&v)[1 << (LOGK - 7)], int t, float* xch, float* redf,
                                                     int* redi, bool store, int64_t row, int32_t* __restrict__ q,
                                                     float* __restrict__ sa, int32_t* __restrict__ qcorr,
                                                     float inv_sqrt_k) {
  constexpr int K = 1 << LOGK;
  constexpr int r = LOGK - 7;
  constexpr int R = 1 << r;
  static_assert(r >= 4 && R % 4 == 0, "runs of >= 16 consecutive elements per lane");
  const int lane = t & 63;
  const int h = t >> 6;
#pragma unroll
  for (int b = 0; b < r; ++b) {
    if (b == 0) reg_stage<0>(v);
    else if (b == 1) reg_stage<1>(v);
    else if (b == 2) reg_stage<2>(v);
    else if (b == 3) reg_stage<3>(v);
    else if (b == 4) reg_stage<4>(v);
    else if (b == 5) reg_stage<5>(v);
    else if (b == 6) reg_stage<6>(v);
  }
  lane_stage<0>(v, lane);
  lane_stage<1>(v, lane);
  lane_stage<2>(v, lane);
  lane_stage<3>(v, lane);
  swap_lane_bit<16, 0>(v);
  reg_stage<0>(v);  // element bit r + 4
  swap_lane_bit<32, 1>(v);
  reg_stage<1>(v);  // element bit r + 5
  swap_lane_bit<32, 1>(v);
  swap_lane_bit<16, 0>(v);
  // element bit r + 6: the other wave's value of the same register and lane
#pragma unroll
  for (int j = 0; j < R; j += 4)
    *reinterpret_cast<float4*>(xch + (h * 64 + lane) * R + j) = make_float4(v[j], v[j + 1], v[j + 2], v[j + 3]);
  __syncthreads();
  const float* px = xch + ((h ^ 1) * 64 + lane) * R;
#pragma unroll
  for (int j = 0; j < R; j += 4) {
    const float4 o4 = *reinterpret_cast<const float4*>(px + j);
    const float o[4] = {o4.x, o4.y, o4.z, o4.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) v[j + e] = h == 0 ? __fadd_rn(v[j + e], o[e]) : __fsub_rn(o[e], v[j + e]);
  }

  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < R; ++j) amax = fmaxf(amax, fabsf(v[j]));
  amax = wave_max_dpp(amax);
  if (lane == 0) redf[h] = amax;
  __syncthreads();
  amax = fmaxf(redf[0], redf[1]);
  const float sdiv = __fadd_rn(__fdiv_rn(amax, 7.0f), 1e-12f);
  if (store && t == 0) sa[row] = __fmul_rn(sdiv, inv_sqrt_k);
  uint32_t words[R / 8];
  bool tie[R / 8];
  bool near_tie = false;
  const float rcp = __builtin_amdgcn_rcpf(sdiv);
#pragma unroll
  for (int u = 0; u < R / 8; ++u) {
    float c8[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) c8[e] = v[8 * u + e];
    tie[u] = false;
    words[u] = quant_pack8_rcp(c8, rcp, tie[u]);
    near_tie |= tie[u];
  }
  if (__builtin_amdgcn_ballot_w64(near_tie) != 0) {  // rare: redo the flagged words exactly
#pragma unroll
    for (int u = 0; u < R / 8; ++u) {
      if (__builtin_amdgcn_ballot_w64(tie[u]) != 0) {
        float c8[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) c8[e] = v[8 * u + e];
        const uint32_t exact = quant_pack8(c8, sdiv);
        words[u] = tie[u] ? exact : words[u];
      }
    }
  }
  if (store) {
#pragma unroll
    for (int u = 0; u < R / 8; u += 2) {
      const uint2 wd = make_uint2(words[u], words[u + 1]);
      *reinterpret_cast<uint2*>(&q[frag_word_index(row, (t * R) / 8 + u, kblocks128(K))]) = wd;
    }
  }
  int s16 = 0;
#pragma unroll
  for (int u = 0; u < R / 8; ++u) s16 += odd_code_sum16(words[u]);
  s16 = wave_sum_dpp(s16);
  if (lane == 0) redi[h] = s16;
  __syncthreads();
  if (store && t == 0) qcorr[row] = -8 * (redi[0] + redi[1]);
}
}  // namespace
}  // namespace w4a4
