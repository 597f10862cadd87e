// Stands in for csrc/direct_load.h: direct loads are queued and land in LDS when an explicit
// wait forces them (or at once, `eager`), ordinary loads only count, a barrier switches fibers.
#pragma once

#include "w4a4_internal.h"

namespace w4a4 {
namespace {

struct Pending {
  const char* src;  // null: an ordinary load
  char* dst;
};
std::vector<Pending>& queue();
char* lds_at(uint32_t addr);
bool table_piece(const char* lds);
void barrier();

inline void land(const Pending& e) {
  if (e.src != nullptr) memcpy(e.dst, e.src, 16);
}
inline void load_lds_1k(const char* base, uint32_t voff, uint32_t dst);
inline load_16_t load_16(const char* p) {
  queue().push_back({nullptr, nullptr});
  return *reinterpret_cast<const load_16_t*>(p);
}
// EMULATE_LOOSE: loads that every wait leaves too many (the test's own check that this is noticed).
#ifndef EMULATE_LOOSE
#define EMULATE_LOOSE 0
#endif
template <int N>
void wait_vm() {
  auto& q = queue();
  while (q.size() > static_cast<size_t>(N + EMULATE_LOOSE)) {
    land(q.front());
    q.erase(q.begin());
  }
}
inline void lds_done_barrier() { barrier(); }
inline int opaque_copy(int v) { return v; }

}  // namespace
}  // namespace w4a4
