"""Plan creation when an allocation or an upload fails: the error is returned and
everything allocated before is freed again.

On the CPU: a small program takes the place of the runtime's memory calls
(its own definitions come before the shared library's) and fails the n-th of
them, for every n until a plan is made."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "openpfc_amd", "libopenpfc_hip.so")

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <dlfcn.h>
#include <set>

static int calls = 0, fail_at = -1;
static std::set<void *> live;
static bool failing() { return calls++ == fail_at; }

extern "C" {
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipSetDevice(int) { return 0; }
int hipGetLastError() { return 0; }
int hipFuncSetAttribute(const void *, int, int) { return 0; }
int hipMalloc(void **p, size_t n) {
  if (failing()) return 2;
  *p = std::malloc(n);
  live.insert(*p);
  return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int) {
  if (failing()) return 999;
  std::memcpy(d, s, n);
  return 0;
}
int hipFree(void *p) {
  if (p && !live.erase(p)) std::exit(3);
  std::free(p);
  return 0;
}
}

int main(int argc, char **argv) {
  void *h = dlopen(argv[1], RTLD_NOW);
  if (!h) { std::puts(dlerror()); return 4; }
  auto create = (int (*)(int, int, int, int, int, void **))dlsym(h, "pfc_hip_plan_create");
  auto destroy = (int (*)(void *))dlsym(h, "pfc_hip_plan_destroy");
  int n[5];
  for (int i = 0; i < 5; ++i) n[i] = std::atoi(argv[2 + i]);
  for (fail_at = 0;; ++fail_at) {
    calls = 0;
    void *plan = nullptr;
    const int rc = create(n[0], n[1], n[2], n[3], n[4], &plan);
    if (rc == 0) {
      if (fail_at < calls) { std::printf("call %d: failure not reported\n", fail_at); return 5; }
      destroy(plan);
      if (!live.empty()) { std::printf("destroy: %zu left\n", live.size()); return 6; }
      std::printf("%d calls\n", calls);
      return 0;
    }
    if (plan) { std::printf("call %d: error and a plan\n", fail_at); return 7; }
    if (!live.empty()) { std::printf("call %d: %zu left\n", fail_at, live.size()); return 6; }
  }
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("planfail")
    (d / "t.cpp").write_text(SOURCE)
    exe = d / "t"
    subprocess.run(["g++", "-std=c++17", "-O1", "-rdynamic", "-o", str(exe), str(d / "t.cpp"),
                    "-ldl"], check=True, timeout=120)
    return str(exe)


# plane kernels' tables (FP64, FP32 with its table in double), none, double butterflies
@pytest.mark.parametrize("args", [(32, 32, 32, 0, 0), (192, 96, 48, 1, 0), (1024, 512, 12, 0, 0),
                                  (256, 128, 128, 1, 1)])
def test_failed_plans_leave_nothing_allocated(program, args):
    if not os.path.exists(LIB):
        pytest.fail(f"{LIB} missing: run __graft_entry__.build()")
    r = subprocess.run([program, LIB, *map(str, args)], capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[0]) > 0
