// The E3M2 GEMM's main tile: 16 MI rows x 256 outputs per workgroup (GELU pairs: 128 gate
// and the same 128 up columns) on v_mfma_f32_16x16x128_f8f6f4.
//
// Structure: four waves along N, two workgroups per CU.  The row fragments of a k block are
// shared by the waves through a three-stage LDS ring filled by direct global-to-LDS loads
// (two steps ahead); each wave's column pairs stream from global memory into a two-block
// register ring.  The column pairs of a block are multiplied one after the other, so that a
// pair's registers are free half a step before the block ends and take the pair of the block
// after the next: the lead of a three-block ring in the registers of two (a three-block ring
// spills).  Two workgroups per CU leave a wave 256 registers, of which the 112-row plain tile
// takes all (accumulators 112, column pairs 48, row fragments 42): per-lane offsets of the next
// tile's rows and of the epilogue are made where they are used (opaque_copy), and the residual's
// are 32-bit ones from a uniform base.  Kept over the k loop they spilled 180 bytes, and each
// reload waited for every load under way: down projection with residual at 6208 rows 219.9 us with
// its quantizer, 206.4 now.  The workgroups walk the tiles, and the loads run on into the next tile's first
// blocks, so that the loads' latency is paid once per workgroup and not once per tile.
// The vmcnt waits and the barrier of a step order the direct loads (direct_load.h), whose lead over
// the LDS reads is the ring's.
//
// What bounds it (gate/up + GELU at 6208 rows, times with parts of the kernel taken out of a
// scratch copy): MFMAs, LDS reads and barriers alone 143 us (register operands alone 120: the
// chip holds 7.0 PFLOP/s with INT4 codes as FP6 operands, its clock falling to 1.67 GHz of
// matrix work); the epilogue adds 52-56, since a SIMD runs one wave's vector instructions and
// the other's MFMAs in turn (2.3 cycles each, 8 for exp2 and rcp); the operand loads add as
// much (a CU's vector memory path moves 56-64 B per clock: 69 KB per k block of two tiles are
// 1080 clocks beside 896 of MFMAs).  Plain at K = 16384 (down projection, 6208 rows): 127 us, 1860
// clocks per k block of two tiles, so the two overlap little there; 4.6 TB/s are read past the L2s.
// Measured (gate/up + GELU, us, the form with a full wait for all loads at every step / this
// one, one box): 200 rows 19.5 / 15.4, 776 rows 44.4 / 38.5, 6208 rows 288 / 250.  Without the
// walk over the tiles 15.0 / 38.5 / 263; both operands through LDS for 224 x 256 tiles of eight
// waves, two groups of them reading and multiplying in turn, 20.6 / 43.4 / 266 (LDS-bound: its
// reads and the loads' writes fill 960 of 896 MFMA cycles); loads spread singly among the
// MFMAs instead of in threes 15.7 / 38.6 / 256.
//
// Results: integer products with exact fp32 sums, so acc is the int32 dot product in any
// order; the epilogue's arithmetic is gemm_w4a4_kernel's.
#pragma once

#include "direct_load.h"
#include "gelu_tanh.h"
#include "w4a4_internal.h"

namespace w4a4 {
namespace {

template <int MI, bool GELU>
struct E3m2Tile {
  static constexpr int NI = 4;                         // column fragments of a wave
  static constexpr int kWaves = 4;
  static constexpr int kChunks = MI + (MI + 1) / 2;    // 1 KB pieces of an A stage
  static constexpr int kStage = kChunks * 1024;
  static constexpr int kPerWave = (kChunks + kWaves - 1) / kWaves;  // pieces a wave loads per stage
  static constexpr int kSlots = 3;
  static constexpr int OCW = GELU ? 32 : 64;           // output columns of a wave
  static constexpr int LSR = OCW + 8;                  // staged row stride in halves (pad)
  // The stages, the GELU correction table, the output staging.
  static constexpr int kFix = kSlots * kStage;
  static constexpr int kOut = kFix + (GELU ? kGeluFixEntries : 0);
  static constexpr int kLds = kOut + kWaves * 16 * LSR * 2;
};

template <int MI, bool GELU>
__device__ __forceinline__ void e3m2_tile(const GemmParams& p, char* lds, const int8_t* fix_table) {
  using T = E3m2Tile<MI, GELU>;
  constexpr int NI = T::NI;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds));

  const int nkb = kblocks128(p.k);
  const int64_t M = p.m;

  // ---- tiles of this workgroup.  XCD x = b % 8 owns a contiguous run of the tiles in an
  // order that walks the m-tiles of one m-group under each n-tile, n-tiles outside, m-groups
  // outermost: a group's activation rows (p.mgroup m-tiles) stay in the XCD's 4 MB L2 while
  // the weights stream through once.  The XCD's workgroups take its tiles in turn.
  const int xcd = blockIdx.x & 7;
  int t_next, t_end, t_stride;
  {
    const int total = p.ntiles * p.mtiles, grid = gridDim.x;
    const int q = total >> 3, r = total & 7;
    const int begin = xcd * q + min(xcd, r);
    t_next = begin + (static_cast<int>(blockIdx.x) >> 3);
    t_end = begin + q + (xcd < r ? 1 : 0);
    t_stride = (grid >> 3) + (xcd < (grid & 7) ? 1 : 0);
  }
  struct Tile {
    const int32_t* w;
    const int32_t* w2;  // GELU: the up weight
    _Float16* y;
    int n, mt, wcol;
  };
  auto tile_at = [&](int t) {
    Tile c;
    const int full = p.mgroup * p.ntiles;
    const int mg = t / full;
    const int rem = t - mg * full;
    const int size = min(p.mgroup, p.mtiles - mg * p.mgroup);
    const int nt = rem / size;
    c.mt = mg * p.mgroup + (rem - nt * size);
    c.w = p.g[0].w;
    c.w2 = p.g[1].w;
    c.y = static_cast<_Float16*>(p.g[0].y);
    c.n = p.g[0].n;
    int tile_begin = 0;
#pragma unroll
    for (int i = 1; i < kMaxGroups; ++i) {
      if (!GELU && i < p.ngroups && nt >= p.g[i].tile_begin) {
        c.w = p.g[i].w;
        c.y = static_cast<_Float16*>(p.g[i].y);
        c.n = p.g[i].n;
        tile_begin = p.g[i].tile_begin;
      }
    }
    c.wcol = GELU ? nt * 128 + wave * 32 : (nt - tile_begin) * 256 + wave * 64;
    return c;
  };

  // ---- A: the 1 KB pieces of a stage, dealt over the waves (piece c to wave c % 4):
  //   c < MI     dwords 0-3 of row fragment c,
  //   c >= MI    dwords 4-5 of row fragments 2 (c - MI) and the next one (odd MI: the last
  //              piece's upper half re-reads a fragment into unread LDS).
  // Row fragments past the matrix are clamped to its last one.
  const uint32_t frag_stride = static_cast<uint32_t>(nkb) * kE3m2FragBytes;  // one row block's k blocks
  auto a_start = [&](const Tile& c, const char*& base, uint32_t (&off)[T::kPerWave]) {
    const int mb0 = c.mt * MI;
    const int l = opaque_copy(lane);  // made at the tile's start, not kept
    base = reinterpret_cast<const char*>(p.q) + static_cast<int64_t>(mb0) * frag_stride;
#pragma unroll
    for (int j = 0; j < T::kPerWave; ++j) {
      const int pc = min(wave + T::kWaves * j, T::kChunks - 1);
      const bool lo = pc < MI;
      const int f = lo ? pc : min(2 * (pc - MI) + (l >> 5), MI - 1);
      const int rel = min(mb0 + f, p.mblocks - 1) - mb0;
      off[j] = static_cast<uint32_t>(rel) * frag_stride + (lo ? l * 16 : 1024 + (l & 31) * 16);
    }
  };
  const char* abase;
  uint32_t voff[T::kPerWave];
  auto issue_a = [&](int j, uint32_t slot) {
    if (T::kChunks % T::kWaves != 0 && j == T::kPerWave - 1 && wave + T::kWaves * j >= T::kChunks) return;  // wave-uniform
    load_lds_1k(abase, voff[j], lds0 + slot + (wave + T::kWaves * j) * 1024);
  };
  // ---- B: the wave's two column pairs (GELU: its gate pair and its up pair), pairs past N
  // clamped to the last one.  A pair's three loads land in one 12-dword value, so that both
  // fragments are consecutive register runs of it.
  auto b_start = [&](const Tile& c, int qd) {
    const int pair = min((GELU ? c.wcol : c.wcol + 32 * qd) >> 5, (c.n >> 5) - 1);
    return reinterpret_cast<const char*>((GELU && qd == 1) ? c.w2 : c.w) + static_cast<int64_t>(pair) * nkb * kE3m2PairBytes;
  };
  const char* bp[2];
  const char* bp_next[2];
  const uint32_t boff = static_cast<uint32_t>(lane) * 16u;
  const int bstep = nkb > 1 ? kE3m2PairBytes : 0;
  // A ring of two blocks.  Past a tile's last block the loads go on with the next tile's first
  // ones (bp_next).  They are unconditional, so that the compiler's vmcnt waits on them stay
  // exact: the last tile's read its own first blocks again.
  v12i b0[2], b1[2];
  auto issue_b = [&](int kb, int qd, v12i (&b)[2]) {
    const v4i c0 = load_16(bp[qd] + boff);
    const v4i c1 = load_16(bp[qd] + boff + 1024);
    const v4i c2 = load_16(bp[qd] + boff + 2048);
    const v8i c01 = __builtin_shufflevector(c0, c1, 0, 1, 2, 3, 4, 5, 6, 7);
    const v8i c2x = __builtin_shufflevector(c2, c2, 0, 1, 2, 3, 4, 5, 6, 7);
    b[qd] = __builtin_shufflevector(c01, c2x, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11);
    bp[qd] = kb + 1 == nkb ? bp_next[qd] : bp[qd] + bstep;
  };
  auto bfrag = [&](const v12i (&b)[2], int ni) {  // fragment ni: dwords 6 (ni % 2) .. + 5 of its pair's record
    const v12i r = b[ni >> 1];
    return (ni & 1) ? __builtin_shufflevector(r, r, 6, 7, 8, 9, 10, 11, 6, 7) : __builtin_shufflevector(r, r, 0, 1, 2, 3, 4, 5, 0, 1);
  };

  v4f acc[MI][NI];

  v8i aop[MI];
  auto read_a = [&](int mi, uint32_t slot) {
    const char* st = lds + slot;
    const v4i lo = *reinterpret_cast<const v4i*>(st + mi * 1024 + lane * 16);
    const int2 hi = *reinterpret_cast<const int2*>(st + MI * 1024 + mi * 512 + lane * 8);
    aop[mi] = e3m2_op(lo, hi.x, hi.y);
  };
  auto next_slot = [&](uint32_t s) { return s == (T::kSlots - 1) * T::kStage ? 0u : s + T::kStage; };
  uint32_t rd = T::kStage;  // slot of stage kb + 1 (read during step kb)
  uint32_t wr = 0;          // slot of stage kb + 3 (requested during step kb): stage kb's

  // Step kb, the MFMAs of block kb (b; its row fragments are in registers): first those of
  // column pair 0, whose registers then take pair 0 of block kb + 2; then, once every wave's
  // loads of A stage kb + 1 have landed and every wave has read stage kb, those of pair 1,
  // after which row fragment mi's registers take the fragment of block kb + 1 from LDS and
  // the pair's registers pair 1 of block kb + 2; the wave's loads of A stage kb + 3 are spread
  // among them.  Blocks and stages past the tile's last are the next tile's.
  bool more = false;  // there is a next tile
  Tile nxt = tile_at(t_next);
  auto step = [&](int kb, v12i (&b)[2]) {
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int ni = 0; ni < 2; ++ni)
        acc[mi][ni] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bfrag(b, ni), aop[mi], acc[mi][ni], 3, 3, 0, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    issue_b(kb + 2, 0, b);
    // Younger loads than A stage kb + 1's (issued in step kb - 2 or the prologue): pair 1 of block
    // kb, both pairs of block kb + 1, pair 0 of block kb + 2, three loads each, and A stage kb + 2.
    if (more || kb + 2 < nkb) {
      if (T::kChunks % T::kWaves == 0 || wave < T::kChunks % T::kWaves) wait_vm<12 + T::kPerWave>();
      else wait_vm<12 + T::kPerWave - 1>();
    } else {
      wait_vm<12>();
    }
    lds_done_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
#pragma unroll
      for (int ni = 2; ni < 4; ++ni)
        acc[mi][ni] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bfrag(b, ni), aop[mi], acc[mi][ni], 3, 3, 0, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      read_a(mi, rd);
      if (mi == 1 && (more || kb + 3 < nkb)) {
#pragma unroll
        for (int j = 0; j < T::kPerWave; ++j) issue_a(j, wr);
        abase += kE3m2FragBytes;
        if (kb + 4 == nkb && more) a_start(nxt, abase, voff);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    issue_b(kb + 2, 1, b);
    rd = next_slot(rd);
    wr = next_slot(wr);
  };

  // ---- prologue: A stages 0-2 and B blocks 0 and 1 of the first tile in the order in which the
  // steps issue them (step kb: pair 0 of block kb + 2, A stage kb + 3, pair 1 of block kb + 2), so
  // that the steps' counts hold from the first one on: A 0, B 0.0, A 1, B 0.1, B 1.0, A 2, B 1.1;
  // then the correction table, which no count relies on.
  Tile cur = tile_at(t_next);
  a_start(cur, abase, voff);
#pragma unroll
  for (int qd = 0; qd < 2; ++qd) bp[qd] = bp_next[qd] = b_start(cur, qd);
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    if (s < nkb) {
#pragma unroll
      for (int j = 0; j < T::kPerWave; ++j) issue_a(j, s * T::kStage);
      abase += kE3m2FragBytes;
    }
    if (s == 0) issue_b(0, 0, b0);
    if (s == 1) {
      issue_b(0, 1, b0);
      issue_b(1, 0, b1);
    }
    if (s == 2) issue_b(1, 1, b1);
  }
  if constexpr (GELU) {  // its two halves by direct loads, zeros between
    constexpr int kFixPieces = kGeluFixPosPieces + (kGeluFixEntries / 1024 - kGeluFixNegPiece0);
    for (int c = wave; c < kFixPieces; c += T::kWaves) {
      const int piece = c < kGeluFixPosPieces ? c : kGeluFixNegPiece0 + (c - kGeluFixPosPieces);
      load_lds_1k(reinterpret_cast<const char*>(fix_table) + piece * 1024, static_cast<uint32_t>(lane) * 16u,
                  lds0 + T::kFix + piece * 1024);
    }
    for (int i = kGeluFixPosPieces * 1024 + tid * 16; i < kGeluFixNegPiece0 * 1024; i += 64 * T::kWaves * 16)
      *reinterpret_cast<int4*>(lds + T::kFix + i) = int4{0, 0, 0, 0};
  }
  // A stage 0: younger are the 12 B loads and (with three stages) A stages 1 and 2, at least
  // kPerWave - 1 pieces each.
  if (nkb >= 3) wait_vm<12 + 2 * (T::kPerWave - 1)>();
  else wait_vm<12>();
  lds_done_barrier();
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) read_a(mi, 0);

  for (;;) {
    t_next += t_stride;
    more = t_next < t_end;
    nxt = tile_at(more ? t_next : t_next - t_stride);
#pragma unroll
    for (int qd = 0; qd < 2; ++qd) bp_next[qd] = b_start(nxt, qd);
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int ni = 0; ni < NI; ++ni) acc[mi][ni] = v4f{0, 0, 0, 0};
    int kb = 0;
    for (; kb + 2 <= nkb; kb += 2) {
      step(kb, b0);
      step(kb + 1, b1);
    }
    if (kb < nkb) step(kb, b0);  // odd: the launch gives every workgroup one tile
    if (GELU && nkb < 8) {  // the table's loads may still be under way
      wait_vm<0>();
      lds_done_barrier();
    }
    const int64_t m0 = static_cast<int64_t>(cur.mt) * (16 * MI);
    const int wcol = cur.wcol, N = cur.n;
    // The epilogue's per-lane offsets are made from a copy, so that they are not kept over the k loop.
    const int elane = opaque_copy(lane);
    const int lrow = elane & 15;
    const int lcol = (elane >> 4) * 4;
    // Epilogue scales: the lane's row of every row fragment and its four columns of every
    // column fragment (clamped: rows and columns past the matrix are never stored).
    float sv[MI];
    float4 sw[NI];
    const int64_t scale_off = static_cast<int64_t>(N) * nkb * 24;
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) sv[mi] = p.sa[min(m0 + mi * 16 + lrow, M - 1)];
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      const int col = (GELU ? wcol + (ni & 1) * 16 : wcol + ni * 16) + lcol;
      const float* s = reinterpret_cast<const float*>(((GELU && ni >= 2) ? cur.w2 : cur.w) + scale_off);
      sw[ni] = *reinterpret_cast<const float4*>(s + min(col, N - 4));
    }

  // ---- epilogue: lane L holds rows 16 mi + L % 16 and columns 16 ni + 4 (L / 16) + 0..3 of
  // its wave tile.  Each 16-row block is staged in the wave's own LDS rows and stored as
  // whole rows.
  constexpr int LSR = T::LSR;
  constexpr int LPR = T::OCW / 8;
  constexpr int RPI = 64 / LPR;
  _Float16* const stage = reinterpret_cast<_Float16*>(lds + T::kOut) + wave * (16 * LSR);
  const int8_t* const fix = reinterpret_cast<const int8_t*>(lds + T::kFix);
  char* const yw = reinterpret_cast<char*>(cur.y + m0 * N + wcol);
  const uint32_t loff = static_cast<uint32_t>((elane / LPR) * N + (elane % LPR) * 8) * 2u;
  // Residual: the 16-byte pieces that this wave's store loop adds, two row blocks ahead
  // (addresses clamped into the matrix; pieces outside it are never stored).
  const bool has_res = !GELU && p.res != nullptr;
  uint4 resv[GELU ? 1 : 3][16 / RPI];
  const int rmax = static_cast<int>(min(M - 1 - m0, static_cast<int64_t>(16 * MI - 1)));  // last row of the tile
  const uint32_t rcol = static_cast<uint32_t>(min(wcol + (elane % LPR) * 8, N - 8)) * 2u;
  auto load_res = [&](int mi) {
    if constexpr (!GELU) {
      if (mi < MI && has_res) {
        const char* const rb = reinterpret_cast<const char*>(p.res + m0 * N);
#pragma unroll
        for (int j = 0; j < 16 / RPI; ++j) {
          const uint32_t r = static_cast<uint32_t>(min(mi * 16 + j * RPI + elane / LPR, rmax));
          resv[mi % 3][j] = *reinterpret_cast<const uint4*>(rb + (r * static_cast<uint32_t>(2 * N) + rcol));
        }
      }
    }
  };
  load_res(0);
  load_res(1);
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    load_res(mi + 2);
#pragma unroll
    for (int ni = 0; ni < (GELU ? 2 : NI); ++ni) {
      const float swv[4] = {sw[ni].x, sw[ni].y, sw[ni].z, sw[ni].w};
      half4 o;
      if constexpr (GELU) {
        const float swu[4] = {sw[ni + 2].x, sw[ni + 2].y, sw[ni + 2].z, sw[ni + 2].w};
        _Float16 g16[4];
        half4 u16;
        int d[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          g16[r] = dequant(acc[mi][ni][r], sv[mi], swv[r]);
          u16[r] = dequant(acc[mi][ni + 2][r], sv[mi], swu[r]);
          d[r] = fix[gelu_fix_index(__builtin_bit_cast(uint16_t, g16[r]))];
        }
        half4 gl;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          gl[r] = __builtin_bit_cast(_Float16, static_cast<uint16_t>(gelu_tanh_fast_bits(g16[r]) + d[r]));
        o = gl * u16;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = dequant(acc[mi][ni][r], sv[mi], swv[r]);
      }
      *reinterpret_cast<half4*>(stage + lrow * LSR + ni * 16 + lcol) = o;
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < 16 / RPI; ++j) {
      const int rr = j * RPI + elane / LPR;
      const int tcol = (elane % LPR) * 8;
      const int trow = mi * 16 + rr;
      uint4 v = *reinterpret_cast<const uint4*>(stage + rr * LSR + tcol);
      char* const yrow = yw + static_cast<int64_t>(mi * 16 + j * RPI) * N * 2;  // uniform; + loff per lane
      if (m0 + trow < M && wcol + tcol < N) {
        if constexpr (!GELU) {
          if (has_res) v = __builtin_bit_cast(uint4, __builtin_bit_cast(half8, v) + __builtin_bit_cast(half8, resv[mi % 3][j]));
        }
        __builtin_nontemporal_store(v4i{static_cast<int>(v.x), static_cast<int>(v.y), static_cast<int>(v.z), static_cast<int>(v.w)},
                                    reinterpret_cast<v4i*>(yrow + loff));
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
    if (!more) break;
    cur = nxt;
    // The last step read the new tile's first row fragments too, but its registers are not
    // kept over the epilogue.
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) read_a(mi, wr);
  }
  wait_vm<0>();  // no load outlives the workgroup's LDS
}

}  // namespace
}  // namespace w4a4
