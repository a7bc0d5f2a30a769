"""Growth of the workspaces that a kick can do without (field lines, bricks) when
memory is short: the rule of csrc/buf.hpp, run on the host with a counted
stand-in for device memory."""
import os
import subprocess

from ocelot_amd import build

MAIN = r"""
#include <cassert>
#include <cstdlib>
#include "buf.hpp"
using namespace ocsc;

struct Mem {
  size_t total, used = 0, hole = 0;  // hole: largest piece that can be had (0: all that is free)
  int taken = 0, given = 0, refused = 0;
  size_t size[8] = {};
  void* at[8] = {};
  size_t available() { return total - used; }
  bool take(void** p, size_t n) {
    if (n > total - used || (hole && n > hole)) return ++refused, false;
    *p = at[taken] = malloc(1);
    size[taken++] = n;
    used += n;
    return true;
  }
  void give(void* p) {
    for (int k = 0; k < taken; ++k)
      if (at[k] == p) used -= size[k];
    ++given;
    free(p);
  }
};

int main() {
  Mem m{100};
  Buf b;
  assert(grow_optional(b, 40, m) && b.cap == 40 && m.taken == 1 && m.given == 0);
  assert(grow_optional(b, 30, m) && b.cap == 40 && m.taken == 1);
  void* const p = b.p;
  // too large: the buffer stays, call after call, and nothing is taken or given
  for (int k = 0; k < 3; ++k) assert(!grow_optional(b, 70, m) && b.p == p && b.cap == 40);
  assert(m.taken == 1 && m.given == 0 && m.refused == 0 && m.used == 40);
  assert(grow_optional(b, 40, m) && b.p == p);  // what it has is still good
  // free, but not in one piece: asked for once
  m.hole = 10;
  for (int k = 0; k < 3; ++k) assert(!grow_optional(b, 50, m) && b.p == p && b.cap == 40);
  assert(m.refused == 1 && m.given == 0);
  // and again when there is more of it
  m.total = 120;
  assert(!grow_optional(b, 50, m) && m.refused == 2);
  m.hole = 0, m.total = 130;
  assert(grow_optional(b, 50, m) && b.cap == 50 && b.p != p && m.given == 1 && m.used == 50);
  return 0;
}
"""


def test_a_refused_growth_leaves_the_buffer_and_is_not_repeated(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(build.HERE, "csrc"), "-o", str(exe),
                    str(src)], check=True)
    subprocess.run([str(exe)], check=True)
