"""A buffer that cannot grow stays usable (bl_grow.h), with an allocator that
has no memory: compiled for the host."""
import os
import subprocess

from tests.conftest import ROOT

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include <set>
#include "bl_grow.h"
static std::set<float*> live;
static bool full = false;
static float* take(int n) {
  if (full) return nullptr;
  float* p = static_cast<float*>(std::malloc(sizeof(float) * n));
  live.insert(p);
  return p;
}
static void give(float* p) {
  if (!live.erase(p)) std::exit(9);
  std::free(p);
}
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
int main() {
  float* b = nullptr;
  int cap = 0;
  full = true;
  CHECK(!bl::grow(&b, &cap, 4, take, give) && !b && cap == 0);
  full = false;
  CHECK(bl::grow(&b, &cap, 4, take, give) && live.count(b) && cap == 4);
  float* const first = b;
  CHECK(bl::grow(&b, &cap, 3, take, give) && b == first && cap == 4);
  full = true;
  CHECK(!bl::grow(&b, &cap, 5, take, give) && b == first && live.count(b) && cap == 4);
  CHECK(bl::grow(&b, &cap, 4, take, give) && b == first);
  full = false;
  CHECK(bl::grow(&b, &cap, 5, take, give) && live.count(b) && !live.count(first) && cap == 5);
  CHECK(live.size() == 1);
  return 0;
}
"""


def test_a_buffer_that_cannot_grow_stays(tmp_path):
    src, exe = tmp_path / "growth.cpp", tmp_path / "growth"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "bookleaf_f90_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_training_grows_its_losses_this_way():
    """bl_mlp_gradient writes through the loss buffer bl_mlp_train grows: the
    buffer is freed nowhere but with the network."""
    with open(os.path.join(ROOT, "bookleaf_f90_amd", "csrc", "bl_mlp.hip")) as f:
        text = f.read()
    assert "grow(&m->loss" in text
    assert "hipFree(m->loss)" not in text


def test_the_tiles_grow_the_partials_this_way():
    """The drivers' dt reductions write to the partials a tiling may grow."""
    with open(os.path.join(ROOT, "bookleaf_f90_amd", "csrc", "bl_tiles.hip")) as f:
        text = f.read()
    assert "grow(&h->d_part," in text and "grow(&h->d_parti," in text
    assert "hipFree(h->d_part" not in text
