"""The pool that keeps the memory of destroyed grids (csrc/grid_pool.h), compiled for the CPU with a stub for the device:
bounds, devices, size classes, and giving memory up when an allocation fails."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include "grid_pool.h"

#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

struct Stub {  // device memory of `room` bytes in all
  static constexpr int OUT_OF_MEMORY = 2;
  static std::map<void *, size_t> live;
  static size_t used, room, host_live;
  static int device(void **p, size_t bytes) {
    if (used + bytes > room) return OUT_OF_MEMORY;
    *p = malloc(1);
    live[*p] = bytes;
    used += bytes;
    return 0;
  }
  static void free_device(void *p) {
    if (!live.count(p)) { printf("freed twice\n"); exit(1); }
    used -= live[p];
    live.erase(p);
    free(p);
  }
  static int host(void **p, size_t bytes) { *p = malloc(bytes); host_live++; return 0; }
  static void free_host(void *p) { host_live--; free(p); }
};
std::map<void *, size_t> Stub::live;
size_t Stub::used = 0, Stub::room = 1 << 20, Stub::host_live = 0;
typedef insc::GridPool<Stub> Pool;

int main() {
  for (size_t b = 1; b < (1u << 22); b = b * 5 / 4 + 1) {
    const size_t c = Pool::size_class(b);
    CHECK(c >= b && c <= b + b / 8 + 256 && Pool::size_class(c) == c);
  }
  Pool pool(64 << 10, 2);
  void *a = nullptr, *b = nullptr, *c = nullptr;
  // a block serves the next one of its class on its device, and no other
  CHECK(pool.alloc(0, 10000, &a) == 0);
  pool.give(0, 10000, a);
  CHECK(pool.held() == Pool::size_class(10000));
  CHECK(pool.alloc(1, 10000, &b) == 0 && b != a);
  CHECK(pool.alloc(0, 20000, &c) == 0 && c != a);
  Stub::free_device(c);
  CHECK(pool.alloc(0, 10001, &c) == 0 && c == a && pool.held() == 0);
  pool.give(0, 10000, a);
  pool.give(1, 10000, b);
  // at most 64 KB, oldest out first; a block of more than half of that is not kept
  for (int i = 0; i < 20; i++) {
    CHECK(pool.alloc(0, 6000 + i * 1000, &c) == 0);
    pool.give(0, 6000 + i * 1000, c);
    CHECK(pool.held() <= (64u << 10) && pool.held() == Stub::used);
  }
  CHECK(pool.alloc(0, 40000, &c) == 0);
  size_t before = pool.held();
  pool.give(0, 40000, c);
  CHECK(pool.held() == before && Stub::used == before);
  // trimming one device leaves the other's
  CHECK(pool.alloc(1, 5000, &c) == 0);
  pool.give(1, 5000, c);
  CHECK(pool.trim(0) && !pool.trim(0) && pool.held() == Pool::size_class(5000));
  CHECK(pool.trim(1) && pool.held() == 0 && Stub::used == 0);
  // an allocation that fails, here or outside the pool, gets the pool's memory of that device
  for (int way = 0; way < 2; way++) {
    CHECK(pool.alloc(0, 30000, &c) == 0);
    pool.give(0, 30000, c);
    Stub::room = 35000;
    CHECK((way ? pool.outside(0, 20000, &c) : pool.alloc(0, 20000, &c)) == 0);
    CHECK(pool.held() == 0);
    Stub::free_device(c);
    CHECK(pool.alloc(1, 30000, &c) == 0);
    pool.give(1, 30000, c);
    CHECK((way ? pool.outside(0, 20000, &a) : pool.alloc(0, 20000, &a)) == Stub::OUT_OF_MEMORY);
    CHECK(pool.trim(1));
    Stub::room = 1 << 20;
  }
  // pinned words stay on the device they were allocated for, two at most
  void *h[4];
  for (int i = 0; i < 4; i++) CHECK(pool.alloc_host(i & 1, 64, &h[i]) == 0);
  for (int i = 0; i < 4; i++) pool.give_host(i & 1, 64, h[i]);
  CHECK(Stub::host_live == 2);
  CHECK(pool.alloc_host(1, 64, &c) == 0 && c == h[1]);
  CHECK(pool.alloc_host(1, 64, &a) == 0 && a != h[0]);
  CHECK(pool.alloc_host(0, 64, &b) == 0 && b == h[0]);
  printf("ok\n");
  return 0;
}
"""


def test_pool(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "ins-conv_amd", "csrc"), str(src), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
