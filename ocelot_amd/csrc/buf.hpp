// Device workspaces: a buffer that keeps its largest size, and the growth of one
// that a call can do without.  No HIP here, so that the rule runs anywhere.
#pragma once
#include <cstddef>

namespace ocsc {

struct Buf {
  void* p = nullptr;
  size_t cap = 0;
  size_t refused_at = 0;  // free memory when a growth was refused (grow_optional), 0: none was
};

// Grows a buffer whose call has another way to go.  The new memory is taken
// before the old is given up, so a refusal leaves the buffer (and the launch
// sequences captured with its address) as they were, and it is not tried again
// until there is more memory free than when it was refused.
// Mem: size_t available(); bool take(void**, size_t); void give(void*) (after
// everything that still uses the memory).
template <class Mem>
bool grow_optional(Buf& b, size_t bytes, Mem&& mem) {
  if (b.cap >= bytes) return true;
  const size_t have = mem.available();
  if (have < bytes || (b.refused_at && have <= b.refused_at)) return false;
  void* p = nullptr;
  if (!mem.take(&p, bytes)) {
    b.refused_at = have;
    return false;
  }
  if (b.p) mem.give(b.p);
  b.p = p;
  b.cap = bytes;
  b.refused_at = 0;
  return true;
}

}  // namespace ocsc
