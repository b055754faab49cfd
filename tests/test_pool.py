"""The pool of equal blocks (axisem_amd/csrc/axh_pool.h): built by the host
compiler with blocks of ordinary memory."""
import os
import subprocess

from conftest import REPO

PROGRAM = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <thread>
#include "axh_pool.h"
static std::atomic<int> made{0}, dropped{0};
static bool fails = false;
static void *make() {
  if (fails) throw std::bad_alloc();
  made++;
  return std::malloc(64);
}
static void drop(void *p) { dropped++; std::free(p); }
#define CHECK(x) if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; }
int main() {
  axh::BlockPool pool(make, drop, 2);
  void *a = pool.take();
  // one in use: a block given back is the next one taken
  for (int k = 0; k < 5; k++) {
    void *b = pool.take();
    CHECK(b && b != a);
    pool.give(b);
  }
  CHECK(made == 2 && dropped == 0);
  // at most two are kept
  void *p[4];
  for (auto &q : p) q = pool.take();
  CHECK(made == 5);
  for (auto q : p) pool.give(q);
  CHECK(dropped == 2);
  // none with the last one in use
  pool.give(a);
  CHECK(dropped == 5);
  a = pool.take();
  CHECK(made == 6);
  // a block that cannot be made is not in use
  fails = true;
  bool threw = false;
  try { pool.take(); } catch (const std::bad_alloc &) { threw = true; }
  CHECK(threw);
  fails = false;
  pool.give(a);
  CHECK(dropped == made);
  std::thread t[8];
  std::atomic<int> bad{0};
  for (auto &q : t)
    q = std::thread([&] {
      for (int k = 0; k < 2000; k++) {
        int *b = (int *)pool.take();
        *b = k;
        std::this_thread::yield();
        if (*b != k) bad++;
        pool.give(b);
      }
    });
  for (auto &q : t) q.join();
  CHECK(bad == 0 && dropped == made);
  return 0;
}
"""


def test_block_pool(tmp_path):
    src, exe = tmp_path / "pool.cpp", tmp_path / "pool"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I",
                    os.path.join(REPO, "axisem_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
