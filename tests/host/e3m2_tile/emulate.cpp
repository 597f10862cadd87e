// Runs the E3M2 GEMM's main tile (csrc/gemm_e3m2_tile.h, as it stands) on the CPU to check how
// its loads, waits and barriers order the operands.  Two lanes of each of a workgroup's four
// waves (0 and 32, which between them load what lane 0 multiplies) run as fibers that switch at
// the barriers.  Operands are tagged with their fragment and k block; every MFMA of a lane 0
// checks that its row operand is the fragment of its step.  `lazy`: a direct load lands when an
// explicit wait of its wave forces it, so only the kernel's own counts are relied on (a wave's
// ordinary loads and the waits for them would cover more).  `eager`: it lands at once, and each
// fiber runs as far ahead as the barriers let it, which shows a stage overwritten too early.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <ucontext.h>
#include <vector>

#include <hip/hip_runtime.h>

#undef __device__
#define __device__
#undef __forceinline__
#define __forceinline__ inline

typedef int load_16_t __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v12i __attribute__((ext_vector_type(12)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));

struct Dim {
  unsigned x;
};
static Dim threadIdx_, blockIdx_, gridDim_;
#define threadIdx threadIdx_
#define blockIdx blockIdx_
#define gridDim gridDim_

template <typename A, typename B>
static auto min(A a, B b) -> decltype(a + b) {
  return a < b ? a : b;
}

static v4f emu_mfma(v8i b, v8i a, v4f acc);
#define __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(B, A, C, ...) emu_mfma(B, A, C)
#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_sched_barrier(x) ((void)0)
#define __builtin_amdgcn_wave_barrier() ((void)0)

#include "direct_load.h"

namespace w4a4 {
namespace {
inline _Float16 dequant(float, float, float) { return 0; }
inline v8i e3m2_op(v4i lo, int d4, int d5) { return v8i{lo.x, lo.y, lo.z, lo.w, d4, d5, 0, 0}; }
}  // namespace
}  // namespace w4a4

#include "gemm_e3m2_tile.h"

namespace w4a4 {
namespace {

constexpr int kLanes[2] = {0, 32};
struct Fiber {
  ucontext_t ctx;
  std::unique_ptr<char[]> stack;
  int wave, lane;
  bool done = false;
  std::vector<Pending> q;
  long mfmas = 0;
  int mb0 = 0;
};
std::vector<std::unique_ptr<Fiber>> fibers;
Fiber* current;
ucontext_t main_ctx;
char* lds_base;
bool eager, count_table;
int nkb_now, mi_now, fix_at, fix_end, mblocks_now;
long errors;
GemmParams params;
std::function<void()> body;

std::vector<Pending>& queue() { return current->q; }
char* lds_at(uint32_t addr) { return lds_base + (addr - static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds_base))); }
bool table_piece(const char* p) { return p >= lds_base + fix_at && p < lds_base + fix_end; }
void barrier() { swapcontext(&current->ctx, &main_ctx); threadIdx_.x = 64 * current->wave + current->lane; }

inline void load_lds_1k(const char* base, uint32_t voff, uint32_t dst) {
  const Pending e{base + voff, lds_at(dst) + 16 * current->lane};
  if (eager) land(e);
  else if (!count_table && table_piece(e.dst)) return;  // must not be needed by any count
  else queue().push_back(e);
}

uint32_t gelu_fix_index(uint32_t) {  // the table is read: every wave's pieces must have landed
  if (count_table)
    for (const auto& f : fibers)
      for (const Pending& e : f->q) errors += e.src != nullptr && table_piece(e.dst);
  return 0;
}

// Every dword of a fragment is tagged row block (or column pair) << 8 | k block.
void check(bool ok) { errors += !ok; }

}  // namespace
}  // namespace w4a4

static v4f emu_mfma(v8i b, v8i a, v4f acc) {
  using namespace w4a4;
  Fiber* f = current;
  if (f->lane != 0) return acc;
  const long n = f->mfmas++;
  const int kb = static_cast<int>((n / (4 * mi_now)) % nkb_now), mi = static_cast<int>(n / 2 % mi_now);
  for (int i = 1; i < 6; ++i) check(a[i] == a[0] && b[i] == b[0]);
  check((a[0] & 255) == kb && (b[0] & 255) == kb);
  const int mb = a[0] >> 8;
  if (mi == 0) f->mb0 = mb;
  check(mb == (f->mb0 + mi < mblocks_now ? f->mb0 + mi : mblocks_now - 1) && f->mb0 % mi_now == 0);
  return acc;
}

namespace w4a4 {
namespace {

void entry() {
  body();
  current->done = true;
  swapcontext(&current->ctx, &main_ctx);
}

template <int MI, bool GELU>
long run(int nkb, int mtiles, int ntiles, unsigned grid, bool eager_, bool count_table_, bool reverse) {
  using T = E3m2Tile<MI, GELU>;
  errors = 0;
  eager = eager_;
  count_table = count_table_;
  mi_now = MI;
  nkb_now = nkb;
  fix_at = T::kFix;
  fix_end = T::kFix + (GELU ? kGeluFixEntries : 0);
  const int64_t m = mtiles * 16 * MI - 17;  // the last block is ragged, the one before it whole
  mblocks_now = static_cast<int>((m + 15) / 16);
  const int n = ntiles * (GELU ? 128 : 256);
  std::vector<int32_t> q(static_cast<size_t>(mblocks_now) * nkb * kE3m2FragBytes / 4 + 64);
  for (size_t i = 0; i < q.size(); ++i) {
    const int frag = static_cast<int>(i / (kE3m2FragBytes / 4));
    q[i] = frag / nkb << 8 | frag % nkb;
  }
  std::vector<int32_t> w(static_cast<size_t>(n) * nkb * 24 + n + 64);
  for (size_t i = 0; i < w.size(); ++i) {
    const int pair = static_cast<int>(i / (kE3m2PairBytes / 4));
    w[i] = pair / nkb << 8 | pair % nkb;
  }
  std::vector<float> sa(m);
  std::vector<_Float16> y(static_cast<size_t>(m) * n), res(y.size());
  std::vector<int8_t> table(kGeluFixEntries);
  GemmParams p{};
  p.q = q.data();
  p.sa = sa.data();
  p.m = m;
  p.mblocks = mblocks_now;
  p.k = 128 * nkb;
  p.ngroups = GELU ? 2 : 1;
  p.g[0] = p.g[1] = GemmGroup{w.data(), y.data(), n, 0};
  p.ntiles = ntiles;
  p.mtiles = mtiles;
  p.mi = MI;
  p.mgroup = 2;
  p.res = GELU ? nullptr : res.data();
  params = p;
  std::vector<char> lds(T::kLds + 64);
  lds_base = lds.data() + (64 - reinterpret_cast<uintptr_t>(lds.data()) % 64) % 64;
  gridDim_.x = grid;
  body = [&] { e3m2_tile<MI, GELU>(params, lds_base, table.data()); };
  for (unsigned b = 0; b < grid; ++b) {
    blockIdx_.x = b;
    memset(lds_base, 0xff, T::kLds);
    fibers.clear();
    for (int i = 0; i < 8; ++i) {
      auto f = std::make_unique<Fiber>();
      f->wave = i / 2;
      f->lane = kLanes[i % 2];
      f->stack.reset(new char[1 << 18]);
      getcontext(&f->ctx);
      f->ctx.uc_stack.ss_sp = f->stack.get();
      f->ctx.uc_stack.ss_size = 1 << 18;
      f->ctx.uc_link = &main_ctx;
      makecontext(&f->ctx, entry, 0);
      fibers.push_back(std::move(f));
    }
    for (bool any = true; any;) {
      any = false;
      int ended = 0;
      for (int i = 0; i < 8; ++i) {
        current = fibers[reverse ? 7 - i : i].get();
        if (current->done) {
          ++ended;
          continue;
        }
        any = true;
        threadIdx_.x = 64 * current->wave + current->lane;
        swapcontext(&main_ctx, &current->ctx);
      }
      check(!any || ended == 0);  // every wave passes the same barriers
    }
    for (const auto& f : fibers) {
      for (const Pending& e : f->q) check(e.src == nullptr);  // no direct load outlives the workgroup
      if (f->lane == 0) check(f->mfmas > 0 && f->mfmas % (4L * MI * nkb) == 0);
    }
  }
  return errors;
}

template <int MI, bool GELU>
int all() {
  int bad = 0;
  struct Shape {
    int nkb, mtiles, ntiles;
    unsigned grid;
  };
  // one tile per workgroup at every short k range, then walks over several tiles
  std::vector<Shape> shapes;
  for (int nkb = 1; nkb <= 9; ++nkb) shapes.push_back({nkb, 2, 1, 2});
  shapes.push_back({16, 1, 2, 2});
  for (int nkb : {4, 6, 8, 16}) shapes.push_back({nkb, 3, 9, 8});
  for (const Shape& s : shapes)
    for (int mode = 0; mode < 6; ++mode) {
      const bool eager_ = mode >= 4;
      const long e = run<MI, GELU>(s.nkb, s.mtiles, s.ntiles, s.grid, eager_, !eager_ && (mode & 2), mode & 1);
      if (e != 0) {
        printf("MI %d %s, %d k blocks, %d x %d tiles on %u workgroups, %s%s: %ld wrong operands\n", MI,
               GELU ? "GELU" : "plain", s.nkb, s.mtiles, s.ntiles, s.grid, eager_ ? "eager" : "lazy",
               !eager_ && (mode & 2) ? ", table loads counted" : "", e);
        ++bad;
      }
    }
  return bad;
}

}  // namespace
}  // namespace w4a4

int main() {
  using namespace w4a4;
  const int bad = all<4, false>() + all<5, false>() + all<6, false>() + all<7, false>() + all<4, true>() +
                  all<5, true>() + all<6, true>() + all<7, true>();
  printf("%d failing runs\n", bad);
  return bad != 0;
}
